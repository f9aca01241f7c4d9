// Linear layers of 17 to 256 rows (wide decode batches, short prompts): y = x . W^T with x [M][K], W [N][K] bf16 row-major, fp32
// accumulation on v_mfma_f32_16x16x32_bf16; or silu(gate) * up of a projection whose rows are [gate | up] (GLU).
//
// Still a weight stream (17440 x 2048 is 71 MB, 200 rows of x 0.8): a workgroup owns 16 WV weight rows (GLU: 16 WV pairs), all
// rows of x and a slice of K.  Both operands go through an LDS ring of 64-deep chunks by direct loads, a row's 128 bytes in
// 16-byte pieces that are swizzled by (row >> 1) & 7 at the source, so that fragment reads touch every bank alike.  A wave's
// fragments of a step are read while the step before is multiplied (one wave a SIMD: nothing else covers the reads), and the
// barrier stands in a chunk's middle, behind which its slot is free.  K is split where whole columns would leave CUs idle; of
// a column group's workgroups the last to arrive adds the others' parts, in their order, to the sum (nobody waits; the counter is
// set back to zero).  The last one's loads go out for eight parts at once: a round trip past the L2 is what they cost.
//
// The weights pass by the caches, which keep x, and workgroups start at different chunks (first_chunk).  With column groups of 32 and
// 48 outputs beside 64 and 80 and row tiles of 48, us: 17440 x 2048 at 24 rows 17.5 -> 13.7, 64 19.2 -> 16.6; pairs of 8192 x 2048
// at 24 16.3 -> 12.7, 64 18.7 -> 14.9; 2048 x 8192 at 40 13.3 -> 10.9; 8192 x 8192 at 24 34.7 -> 24.5; 2048 x 2048 at 40 9.4 -> 6.9.
#include "common.h"
#include "hybrid_launchers.h"

#include <algorithm>

namespace {

constexpr int RING = 160 * 1024;
typedef __attribute__((address_space(3))) void lds_t;

SYM_DEV __amdgpu_buffer_rsrc_t rows_buffer(const void* base, long long bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes, 0x00020000);
}

SYM_DEV void store_through(float* p, f32x4 v) {
  asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1" ::"v"(p), "v"(v) : "memory");
}

struct Args {
  const bf16* x;
  const bf16* W;
  bf16* out;
  float* slab;
  int* counters;
  int ldx, ldo, M, N, K;      // GLU: N outputs, W has 2 N rows
  int per;                    // chunks of a slice
};

template <int MT, int WV, bool GLU>
struct Cfg {
  static constexpr int RW = GLU ? 2 : 1;
  static constexpr int XB = MT * 2048, WB = WV * RW * 2048, SLOT = XB + WB;      // bytes of a chunk
  static constexpr int SLOTS = RING / SLOT > 8 ? 8 : RING / SLOT;
  static constexpr int NX = (2 * MT + WV - 1) / WV, ND = NX + 2 * RW;            // direct loads of a wave and chunk
  static constexpr int KEEP = (SLOTS - 2) * ND, KEEP0 = KEEP + ND < 63 ? KEEP + ND : 63;
  static_assert(SLOTS >= 3 && KEEP <= 63, "ring");
};

template <int MT, int WV, bool GLU, bool F32 = false>
__global__ __launch_bounds__(64 * WV, 1) void mid_linear_kernel(Args a) {
  using C = Cfg<MT, WV, GLU>;
  constexpr int RW = C::RW;
  __shared__ __attribute__((aligned(1024))) char smem[C::SLOTS * C::SLOT];
  asm volatile("" ::: "a0");      // accumulators may live in AGPRs
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int M = a.M, N = a.N, K = a.K, split = blockIdx.y, S = gridDim.y;
  const int c0 = split * a.per, nch = min(a.per, K / 64 - c0);
  const int n0 = (blockIdx.x * WV + wid) * 16;

  // rows of x past M read zeros (the buffer's range); weight rows past N repeat the last one, their products are not stored
  const __amdgpu_buffer_rsrc_t rx = rows_buffer(a.x, ((long long)(M - 1) * a.ldx + K) * 2);
  const __amdgpu_buffer_rsrc_t rw = rows_buffer(a.W, (long long)(GLU ? 2 : 1) * N * K * 2);
  int vx[C::NX], vw[RW][2];
#pragma unroll
  for (int i = 0; i < C::NX; ++i) {
    const int row = min(C::NX * wid + i, 2 * MT - 1) * 8 + (lane >> 3);
    vx[i] = row * a.ldx * 2 + 16 * ((lane & 7) ^ ((row >> 1) & 7)) + c0 * 128;
  }
#pragma unroll
  for (int rt = 0; rt < RW; ++rt)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int row = 8 * i + (lane >> 3);
      vw[rt][i] = (min(n0 + row, N - 1) + rt * N) * K * 2 + 16 * ((lane & 7) ^ ((row >> 1) & 7)) + c0 * 128;
    }
  auto load = [](__amdgpu_buffer_rsrc_t r, int off, int soff, char* lds) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_t*)lds, 16, off, soff, 0, 0);
  };
  auto load_once = [](__amdgpu_buffer_rsrc_t r, int off, int soff, char* lds) {      // (past the caches, which keep x)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_t*)lds, 16, off, soff, 0, 2);
  };
  const int turn = first_chunk(blockIdx.x + gridDim.x * split, nch, (long long)M * K * 2);
  auto issue = [&](int c, int slot) {
    c = c + turn < nch ? c + turn : c + turn - nch;
    char* const s = smem + slot * C::SLOT;
#pragma unroll
    for (int i = 0; i < C::NX; ++i) load(rx, vx[i], c * 128, s + min(C::NX * wid + i, 2 * MT - 1) * 1024);
#pragma unroll
    for (int rt = 0; rt < RW; ++rt)
#pragma unroll
      for (int i = 0; i < 2; ++i) load_once(rw, vw[rt][i], c * 128, s + C::XB + ((wid * RW + rt) * 2 + i) * 1024);
  };

  const int j = lane & 15, h = lane >> 4;
  const int fo = j * 128 + 16 * (h ^ ((j >> 1) & 7));      // a fragment's piece of the first step; of the second: 64 bytes across
  // F32: the sums are the result, of all of K: in parts of 256, as long chains lose bits
  f32x4 acc[RW][MT], total[F32 ? RW : 1][F32 ? MT : 1];
#pragma unroll
  for (int rt = 0; rt < RW; ++rt)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      acc[rt][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
      if constexpr (F32) total[rt][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
  struct Frag {
    bf16x8 w[RW], x[MT];
  };
  Frag f0, f1;
  auto step = [&](Frag& next, int slot, int s, const Frag& now, bool reads, bool multiplies) __attribute__((always_inline)) {
    const char* const sb = smem + slot * C::SLOT;
    const int o = s ? fo ^ 64 : fo;
    constexpr int READS = RW + MT, PER = (READS + MT - 1) / MT;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
      for (int u = 0; u < PER; ++u) {
        const int i = PER * mt + u;
        if (!reads || i >= READS) continue;
        if (i < RW) next.w[i] = *(const bf16x8*)(sb + C::XB + (wid * RW + i) * 2048 + o);
        else next.x[i - RW] = *(const bf16x8*)(sb + (i - RW) * 2048 + o);
      }
      if (multiplies) {
#pragma unroll
        for (int rt = 0; rt < RW; ++rt) acc[rt][mt] = mfma16(now.w[rt], now.x[mt], acc[rt][mt]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
#pragma unroll
  for (int c = 0; c < C::SLOTS; ++c)
    if (c < nch) issue(c, c);
  if (C::SLOTS <= nch) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(C::KEEP0) : "memory");
  else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  step(f0, 0, 0, f1, true, false);
  int slot = 0;
  for (int c = 0; c + 1 < nch; ++c) {
    const int after = slot == C::SLOTS - 1 ? 0 : slot + 1;
    step(f1, slot, 1, f0, true, true);
    // chunk c + 1 has landed (those up to c + SLOTS - 1 stay in flight), chunk c is in registers
    if (c + C::SLOTS - 1 < nch) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(C::KEEP) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xc07f);      // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (c + C::SLOTS < nch) issue(c + C::SLOTS, slot);
    step(f0, after, 0, f1, true, true);
    if (F32 && c % 4 == 3) {
#pragma unroll
      for (int rt = 0; rt < (F32 ? RW : 0); ++rt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          total[rt][mt] += acc[rt][mt];
          acc[rt][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
    slot = after;
  }
  step(f1, slot, 1, f0, true, true);
  step(f0, slot, 0, f1, false, true);

  if (S > 1) {
    // parts as they lie in the registers, written through; the last arriver reads them past its L2, many at a time: what it costs
    // is the round trips
    float* const mine = a.slab + ((long long)blockIdx.x * S * WV + wid) * (RW * MT * 256) + lane * 4;
    constexpr long long PART = (long long)WV * RW * MT * 256;
#pragma unroll
    for (int rt = 0; rt < RW; ++rt)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
        if (16 * mt < M) store_through(mine + split * PART + (rt * MT + mt) * 256, acc[rt][mt]);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    int* last = reinterpret_cast<int*>(smem);      // (every wave is past its reads)
    if (threadIdx.x == 0) {
      const int got = __hip_atomic_fetch_add(a.counters + blockIdx.x, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (got == S - 1) __hip_atomic_store(a.counters + blockIdx.x, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      *last = got == S - 1;
    }
    __syncthreads();
    if (!*last) return;
    constexpr int MB = RW * MT < 8 ? RW * MT : 8, SB = MB <= 4 ? 8 : 4;
    const __amdgpu_buffer_rsrc_t rp = rows_buffer(a.slab, 4LL * MID_SLAB);
    const int from = (int)((blockIdx.x * S * WV + wid) * (RW * MT * 256) + lane * 4) * 4;
#pragma unroll
    for (int t0 = 0; t0 < RW * MT; t0 += MB) {
#pragma unroll
      for (int u = 0; u < MB; ++u)
        if (t0 + u < RW * MT) acc[(t0 + u) / MT][(t0 + u) % MT] = f32x4{0.f, 0.f, 0.f, 0.f};
      for (int s0 = 0; s0 < S; s0 += SB) {
        u32x4 v[SB][MB];
#pragma unroll
        for (int e = 0; e < SB; ++e)
#pragma unroll
          for (int u = 0; u < MB; ++u)
            if (t0 + u < RW * MT)
              v[e][u] = __builtin_amdgcn_raw_buffer_load_b128(rp, from, (int)(min(s0 + e, S - 1) * PART + (t0 + u) * 256) * 4, 17);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < SB; ++e) {
          if (s0 + e >= S) break;
#pragma unroll
          for (int u = 0; u < MB; ++u)
            if (t0 + u < RW * MT) acc[(t0 + u) / MT][(t0 + u) % MT] += __builtin_bit_cast(f32x4, v[e][u]);
        }
      }
    }
  }
  // lane (j, h): outputs n0 + 4 h .. + 3 of row 16 mt + j; N is a multiple of 4
  const int n = n0 + 4 * h;
  if (n >= N) return;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int m = 16 * mt + j;
    if (m >= M) continue;
    if constexpr (F32) {
      *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(a.out) + (long long)m * a.ldo + n) = acc[0][mt] + total[0][mt];
      continue;
    }
    bf16x4 y;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float v = acc[0][mt][r];
      // (the two projections are rounded to bf16 first, as separate launches leave them)
      if constexpr (GLU) v = silu((float)(bf16)v) * (float)(bf16)acc[RW - 1][mt][r];
      y[r] = (bf16)v;
    }
    *reinterpret_cast<bf16x4*>(a.out + (long long)m * a.ldo + n) = y;
  }
}

constexpr int CUS = 256;

template <int MT, int WV, bool GLU>
void run(const Args& a, int S, hipStream_t s) {
  mid_linear_kernel<MT, WV, GLU><<<dim3((a.N + 16 * WV - 1) / (16 * WV), S), 64 * WV, 0, s>>>(a);
}

template <int WV, bool GLU>
void run_rows(const Args& a, int S, hipStream_t s) {
  if (a.M <= 32) run<2, WV, GLU>(a, S, s);
  else if (a.M <= 48) run<3, WV, GLU>(a, S, s);
  else if (a.M <= 64) run<4, WV, GLU>(a, S, s);
  else if (a.M <= 96) run<6, WV, GLU>(a, S, s);
  else if (a.M <= 128) run<8, WV, GLU>(a, S, s);
  else if (a.M <= 160) run<10, WV, GLU>(a, S, s);
  else if (a.M <= 192) run<12, WV, GLU>(a, S, s);
  else run<16, WV, GLU>(a, S, s);
}

// A plan's time beside what all have, us: a workgroup takes in its weight rows at 31 KB / us, all together at 7.3 MB / us, x from its
// L2 at 110 KB / us; to hand parts over costs 3.3, and 87 KB / us of the others' parts.  (Fitted to all plans of 1463 sizes, 17 to 250
// rows, 2048 to 17440 outputs, K of 2048 to 14336; the plan that it picks takes 1.007 of the best one's time, at worst 1.15.)
float plan_time(const Args& a, int groups, int rows, int S) {
  const int per = (a.K / 64 + S - 1) / S;
  const float weights = std::max(per * 128e-3f * rows / 31.f, 2e-3f * groups * rows * a.K / 7300.f);
  return weights + per * 128e-3f * a.M / 110.f + (S > 1 ? 3.3f : 0.f) + (S - 1) * 4e-3f * rows * a.M / 87.f;
}

}  // namespace

// slab: MID_SLAB floats; counters: 256, zero before and after.  false: not one of the widths or sizes
bool launch_mid_linear(const void* x, long long ldx, const void* W, void* out, long long ldo, int M, int N, int K, int glu, float* slab,
                       int* counters, hipStream_t s) {
  Args a{(const bf16*)x, (const bf16*)W, (bf16*)out, slab, counters, (int)ldx, (int)ldo, M, N, K, K / 64};
  constexpr long long top = 0x7fffffffLL;      // (a buffer's range, and a lane's offset in it)
  if (M < 1 || M > 256 || K % 64 || N % 4 || 256 * ldx * 2 + K * 2LL > top || (glu ? 2LL : 1LL) * N * K * 2 > top) return false;
  const int rw = glu ? 2 : 1;
  int best = 0, splits = 1;
  float least = 1e30f;
  for (int wv : {4, 5, 3, 2}) {
    if (glu && wv == 5) continue;
    const int groups = (N + 16 * wv - 1) / (16 * wv);
    for (int S = 1; S <= 16 && groups * S <= CUS && S <= K / 64; ++S) {
      const float t = plan_time(a, groups, 16 * wv * rw, S);
      if (t < least) least = t, best = wv, splits = S;
    }
  }
  if (!best) return false;
  a.per = (K / 64 + splits - 1) / splits;
  splits = (K / 64 + a.per - 1) / a.per;
  if (best == 2) glu ? run_rows<2, true>(a, splits, s) : run_rows<2, false>(a, splits, s);
  else if (best == 3) glu ? run_rows<3, true>(a, splits, s) : run_rows<3, false>(a, splits, s);
  else if (best == 4) glu ? run_rows<4, true>(a, splits, s) : run_rows<4, false>(a, splits, s);
  else run_rows<5, false>(a, splits, s);
  return true;
}

// ... of 17 to 64 rows into fp32, over all of K, in rounds of workgroups of 64 outputs: an lm_head, 32768 x 2048 at 24 rows 26.8 us
// (5 TB/s; the library 36.4), 65536 x 4096 at 32 94 (125)
bool launch_mid_linear_f32(const void* x, long long ldx, const void* W, float* out, long long ldo, int M, int N, int K, hipStream_t s) {
  const Args a{(const bf16*)x, (const bf16*)W, (bf16*)out, nullptr, nullptr, (int)ldx, (int)ldo, M, N, K, K / 64};
  constexpr long long top = 0x7fffffffLL;
  if (M < 1 || M > 64 || K % 64 || N % 4 || 64 * ldx * 2 + K * 2LL > top || 2LL * N * K > top) return false;
  const int groups = (N + 63) / 64;
  if (M <= 32) mid_linear_kernel<2, 4, false, true><<<groups, 256, 0, s>>>(a);
  else if (M <= 48) mid_linear_kernel<3, 4, false, true><<<groups, 256, 0, s>>>(a);
  else mid_linear_kernel<4, 4, false, true><<<groups, 256, 0, s>>>(a);
  return true;
}
