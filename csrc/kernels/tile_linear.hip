// Linear layers of a few hundred to a few thousand rows, y = x w^T, bf16: a tile of 64 or 128 rows x 128 outputs a workgroup, one round
// of the CUs.
//
// What bounds such a product is neither the matrix cores nor memory but the wait for a stage of K: a round that is not full has one
// workgroup a CU, and nothing else runs there meanwhile.  So the stages of 64 stand in a ring that takes all of the CU's LDS (six of
// 64 + 128 rows or five of 128 + 128) and are asked for by direct loads as soon as their place is free, four ahead at 128 rows;
// a wave reads its fragments half a stage ahead of their products, and a stage has one barrier.  Four waves, 2 x 2.
// LDS rows are 128 B with the 16-byte chunk c stored at another place of the row, by the load's source, so fragment reads do not
// conflict; a wave's weight rows are read in an order in which a lane's 16 outputs of a row lie side by side: it stores 32 bytes.
// K is split where tiles would leave half of the CUs idle: of a tile's workgroups the last to arrive adds the parts in their order (nobody
// waits; the counter is set back to zero).
// A stage takes 0.25 us at 64 rows and 0.34 at 128, most of it LDS traffic, start and end 3 to 4.5.  Library -> so, us: 1000 rows of 2048 x
// 2048 15.9 -> 14.0, 700 of 2048 x 8192 in two slices 44.4 -> 38.9, 331 of 4864 x 14336 in two 88 -> 71.3; the rule's lines stand in
// ops.tile_plan.  (The bound of two workgroups a CU keeps the sums in the registers that products write: with all 512 the compiler moved
// them in the loop, 1000 rows of 2048 x 2048 18.1.)
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "direct_lds.h"
#include "hybrid_launchers.h"

namespace {

constexpr int BN = 128, CU_LDS = 160 * 1024, GROUP = 8;
constexpr int stage_bytes(int BM) { return (BM + BN) * 128; }
constexpr int ring(int BM) { return CU_LDS / stage_bytes(BM); }

struct TileArgs {
  const void *x, *w;
  void* y;
  int M, N, K, vec, per;      // vec: 16-byte stores; per: stages of a slice of K
  long long ldx, ldy;
  float* slab;
  int* counters;
};

// (a wide store still reads its data while the next instruction issues, and what stands in assembly the compiler does not keep apart)
SYM_DEV void store_through(float* p, f32x4 v) {
  asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1\n\ts_nop 1" ::"v"(p), "v"(v) : "memory");
}

template <int FM>      // a wave: 16 FM rows x 64 outputs
__global__ __launch_bounds__(256, 2) void tile_linear_kernel(TileArgs a) {
  constexpr int BM = 32 * FM, D = ring(BM), STAGE = stage_bytes(BM), LA = BM / 32, LB = BN / 32, LOADS = LA + LB, READS = FM + 4;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wr = wave >> 1, wc = wave & 1;
  const int mt = (a.M + BM - 1) / BM, nt = (a.N + BN - 1) / BN, tiles = mt * nt;

  // ---- this workgroup's tile: an XCD takes a run of them, all row tiles of GROUP column tiles before the next GROUP
  const int per = (tiles + 7) / 8, t = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per || t >= tiles) return;
  const int g = t / (GROUP * mt), in = t - g * GROUP * mt, cols = min(GROUP, nt - GROUP * g), m = in / cols;
  const int m0 = BM * m, n0 = BN * (GROUP * g + in - m * cols);

  // ---- direct loads of 8 rows each: instruction i covers rows 32 i + 8 wave + lane / 8 of an operand; rows past the end re-read
  // the last one (never stored)
  const int lrow = 8 * wave + (lane >> 3), K2 = a.K * 2;
  const int split = blockIdx.y, S = gridDim.y, k0 = 128 * split * a.per;      // (bytes of a row in front of the slice)
  const u32x4 xbuf = buffer_words(a.x, ((long long)(a.M - 1) * a.ldx + a.K) * 2), wbuf = buffer_words(a.w, (long long)a.N * K2);
  int xoff[LA], woff[LB];
#pragma unroll
  for (int i = 0; i < LA; ++i)
    xoff[i] = min(m0 + 32 * i + lrow, a.M - 1) * (int)a.ldx * 2 + 16 * ((lane & 7) ^ ((lrow >> 1) & 7));
#pragma unroll
  for (int i = 0; i < LB; ++i) {
    const int r = 32 * i + lrow;
    woff[i] = min(n0 + r, a.N - 1) * K2 + 16 * ((lane & 7) ^ (2 * ((r >> 4) & 3) + ((r >> 1) & 1)));
  }
  const unsigned int lds0 = lds_address(smem) + 1024 * wave;
  auto load = [&](int i, int kx, unsigned int at) {
    kx += k0;
    if (i < LA) direct_buffer_load16(xbuf, xoff[i], kx, lds0 + at + 4096 * i);
    else direct_buffer_load16(wbuf, woff[i - LA], kx, lds0 + at + 128 * BM + 4096 * (i - LA));
  };

  f32x4 acc[4][FM];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int q = 0; q < FM; ++q) acc[i][q] = f32x4{0.f, 0.f, 0.f, 0.f};
  Pack8 f0[READS], f1[READS];      // the fragments of a stage's halves: 4 of weight rows, FM of rows
  const int j = lane & 15, hq = lane >> 4, ch = 16 * (hq ^ ((j >> 1) & 7));
  // of weight rows: 16 (j / 4) + 4 i + j % 4 of the wave's 64 stands in row j of fragment i
  const int a0 = 128 * (16 * FM * wr + j) + ch, b0 = 128 * (BM + 64 * wc + 16 * (j >> 2) + (j & 3)) + ch;
  auto fragment = [&](Pack8 (&f)[READS], int half, unsigned int at, int i) {
    if (i < 4) f[i].u = *reinterpret_cast<const uint4*>(smem + at + (b0 ^ half) + 512 * i);
    else f[i].u = *reinterpret_cast<const uint4*>(smem + at + (a0 ^ half) + 2048 * (i - 4));
  };
  constexpr int RI = (READS + 2) / 3;      // fragments read beside a row of products: all of them in front of the last one
  const int nk = min(a.per, a.K / 64 - split * a.per);
  unsigned int at = 0;
  auto first_half = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int u = 0; u < RI; ++u)
        if (RI * i + u < READS) fragment(f1, 64, at, RI * i + u);
#pragma unroll
      for (int q = 0; q < FM; ++q) acc[i][q] = mfma16(f0[i].v, f0[4 + q].v, acc[i][q]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // every wave: the next stage has landed (behind it: those of `behind` stages), this one's fragments are in registers
  auto meet = [&](auto behind) __attribute__((always_inline)) {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(decltype(behind)::value * LOADS) : "memory");
    __builtin_amdgcn_s_waitcnt(0xc07f);      // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  auto second_half = [&](auto next, int kx) __attribute__((always_inline)) {      // 0: nothing follows, 1: a stage, 2: and one to load
    constexpr int NX = decltype(next)::value, LI = (LOADS + 3) / 4;
    const unsigned int from = at + STAGE == D * STAGE ? 0u : at + STAGE;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int u = 0; u < LI; ++u)
        if (NX == 2 && LI * i + u < LOADS) load(LI * i + u, kx, at);
#pragma unroll
      for (int u = 0; u < RI; ++u)
        if (NX && RI * i + u < READS) fragment(f0, 0, from, RI * i + u);
#pragma unroll
      for (int q = 0; q < FM; ++q) acc[i][q] = mfma16(f1[i].v, f1[4 + q].v, acc[i][q]);
      __builtin_amdgcn_sched_barrier(0);
    }
    at = from;
  };
  using Zero = std::integral_constant<int, 0>;
  using One = std::integral_constant<int, 1>;
  using Two = std::integral_constant<int, 2>;

  // (nk >= D)
#pragma unroll
  for (int s = 0; s < D; ++s)
#pragma unroll
    for (int i = 0; i < LOADS; ++i) load(i, 128 * s, s * STAGE);
  meet(std::integral_constant<int, D - 1>{});
#pragma unroll
  for (int i = 0; i < READS; ++i) fragment(f0, 0, 0, i);
  int s = 0;
  for (; s + D < nk; ++s) {
    first_half();
    meet(std::integral_constant<int, D - 2>{});
    second_half(Two{}, 128 * (s + D));
  }
  for (; s + 1 < nk; ++s) {      // the last D stages: nothing left to load
    first_half();
    if (D > 5 && nk - 2 - s >= 4) meet(std::integral_constant<int, D - 2 < 4 ? D - 2 : 4>{});
    else if (D > 4 && nk - 2 - s >= 3) meet(std::integral_constant<int, D - 2 < 3 ? D - 2 : 3>{});
    else if (D > 3 && nk - 2 - s >= 2) meet(std::integral_constant<int, D - 2 < 2 ? D - 2 : 2>{});
    else if (nk - 2 - s >= 1) meet(One{});
    else meet(Zero{});
    second_half(One{}, 0);
  }
  first_half();
  second_half(Zero{}, 0);
  settle(acc[3][FM - 1]);      // (the last of them)

  if (S > 1) {
    // parts as they lie in the registers, written through; the last arriver reads them past its L2
    constexpr int PART = BM * BN, SB = 8 / FM;
    float* const mine = a.slab + ((long long)t * S + split) * PART + wave * (FM * 1024) + lane * 4;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int q = 0; q < FM; ++q) store_through(mine + (i * FM + q) * 256, acc[i][q]);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    int* last = reinterpret_cast<int*>(smem);      // (every wave is past its reads)
    if (threadIdx.x == 0) {
      const int got = __hip_atomic_fetch_add(a.counters + t, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (got == S - 1) __hip_atomic_store(a.counters + t, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      *last = got == S - 1;
    }
    __syncthreads();
    if (!*last) return;
    const __amdgpu_buffer_rsrc_t parts = __builtin_amdgcn_make_buffer_rsrc(a.slab, (short)0, (int)(4 * MID_SLAB), 0x00020000);
    const int from = (t * S * PART + wave * (FM * 1024) + lane * 4) * 4;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int q = 0; q < FM; ++q) acc[i][q] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < S; s0 += SB) {
      u32x4 v[SB][4 * FM];
#pragma unroll
      for (int e = 0; e < SB; ++e)
#pragma unroll
        for (int u = 0; u < 4 * FM; ++u)
          v[e][u] = __builtin_amdgcn_raw_buffer_load_b128(parts, from, (min(s0 + e, S - 1) * PART + u * 256) * 4, 17);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int e = 0; e < SB; ++e) {
        if (s0 + e >= S) break;
#pragma unroll
        for (int u = 0; u < 4 * FM; ++u) acc[u / FM][u % FM] += __builtin_bit_cast(f32x4, v[e][u]);
      }
    }
  }

  // lane (j, hq): row 16 q + j of the wave's, outputs 16 hq .. 16 hq + 15 of its 64
  const int n = n0 + 64 * wc + 16 * hq;
#pragma unroll
  for (int q = 0; q < FM; ++q) {
    const int row = m0 + 16 * FM * wr + 16 * q + j;
    if (row < a.M) {
      bf16* o = reinterpret_cast<bf16*>(a.y) + row * a.ldy + n;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        Pack8 p;
#pragma unroll
        for (int u = 0; u < 8; ++u) p.v[u] = (bf16)acc[2 * h + (u >> 2)][q][u & 3];
        if (a.vec) {
          if (n + 8 * h < a.N) *reinterpret_cast<uint4*>(o + 8 * h) = p.u;
        } else {
#pragma unroll
          for (int u = 0; u < 8; ++u)
            if (n + 8 * h + u < a.N) o[8 * h + u] = p.h[u];
        }
      }
    }
  }
}

template <int FM>
void launch(const TileArgs& a, int tiles, int splits, hipStream_t s) {
  constexpr int LDS = ring(32 * FM) * stage_bytes(32 * FM);
  static const hipError_t once =
      hipFuncSetAttribute(reinterpret_cast<const void*>(&tile_linear_kernel<FM>), hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
  (void)once;
  tile_linear_kernel<FM><<<dim3((tiles + 7) / 8 * 8, splits), 256, LDS, s>>>(a);
}

}  // namespace

bool launch_tile_linear(const void* x, long long ldx, const void* w, void* y, long long ldy, int M, int N, int K, int rows, int splits,
                        float* slab, int* counters, hipStream_t s) {
  const bool vec = N % 8 == 0 && ldy % 8 == 0 && reinterpret_cast<uintptr_t>(y) % 16 == 0;
  const long long tiles = (long long)((M + rows - 1) / rows) * ((N + BN - 1) / BN);
  if ((rows != 64 && rows != 128) || splits < 1 || tiles > (1 << 20) || (splits > 1 && (!slab || tiles * splits > 256))) return false;
  TileArgs a{x, w, y, M, N, K, vec, (K / 64 + splits - 1) / splits, ldx, ldy, slab, counters};
  if (K / 64 - (splits - 1) * a.per < ring(rows)) return false;      // (the last slice's stages)
  rows == 64 ? launch<2>(a, (int)tiles, splits, s) : launch<4>(a, (int)tiles, splits, s);
  return true;
}
