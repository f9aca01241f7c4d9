// Medium-M projection GEMM (17..256 rows: prefill chunks, wide decode batches): fp32 split-K slabs
//   y[s][m][n] = sum_{k in slice s} x[m][k] * W[n][k],   x [M][K], W [N][K] bf16, M <= 256.
//
// Why a separate kernel: at these M a projection is still weight-streaming (Llama-3-8B: 128 tokens x
// 436 MB of weights per layer), but the library GEMM picks tiles that leave most CUs idle or stream the
// weights at 1.3-2.7 TB/s (profiles/prefill_gemm_hipblaslt_r1.jsonl), and the decode kernels re-read
// x once per 16-row weight tile (built for M <= 64).  Here every CU streams its own weight rows once,
// while the activation slice it needs is shared by its 4 waves through LDS:
//
//   * orientation Y^T = W . x^T on v_mfma_f32_16x16x32_bf16: the weight tile is the A operand and comes
//     from the MFMA-preshuffled weight copy (models/layout.py::preshuffle, the decode layout), so every
//     weight DMA instruction reads 1 KB contiguous; x fragments are the B operand;
//   * workgroup = CT 16-row weight tiles (4 waves x RW of them, or 3, 6, 7 or 14 where those fill more CUs) x all M tokens x
//     one k slice; the k split S is chosen on the host so the grid fills the 256 CUs; partial sums go to fp32 slabs
//     that the consumer (rope_cache / add_rms_norm / swiglu, LinOut) sums in its prologue, as the skinny
//     decode GEMM's do;
//   * x AND the weight blocks stream through an LDS ring of 64-deep chunks by LDS-DMA (buffer loads: x
//     rows past M read as zeros), up to 7 chunks ahead (as many as 160 KB of LDS holds), so one counted
//     vmcnt per chunk covers both operands (an ordinary weight load beside LDS-DMA makes hipcc drain
//     vmcnt to 0 at its first use); a preshuffled weight block is
//     1 KB in fragment order, so its DMA and its ds_read_b128 are both lane-linear; the 16-B chunk index
//     of each 128-B x row is XOR-swizzled with (row >> 1) & 7 on the DMA source and on the read, which
//     makes the x fragment reads bank-conflict free;
//   * a step's fragments are read from LDS while the step before is multiplied: with one wave a SIMD nothing else covers the
//     reads (a ring of its own for the weights, two chunks deeper, was slower, also with waves of its own that fill it);
//   * what bounds it is the bytes in flight: 137 rows of 28672 x 4096 take 50 us with no product at all, and as many with them.
//     So x tiles come in steps of 16 rows up to 192 and of 32 above (a slot less of padding is a slot more of the ring), the chunk's DMAs are dealt to the
//     waves one by one, and the weights are loaded past the caches (read once; x stays in the L2).  Against row tiles in steps of
//     32 and cached weights, us: 28672 x 4096 at 20 rows 41.9 -> 38.7, 64 43.1 -> 40.5, 137 57.8 -> 50.9, 192 65.0 -> 62.9;
//     4096 x 14336 at 64 24.3 -> 22.8, 137 31.6 -> 28.6, 240 46.1 -> 40.4; 4096 x 4096 at 137 14.5 -> 13.4.
//     Workgroups start at different chunks (first_chunk), in step -> so, us: 28672 x 4096 at 24 rows 38.8 -> 37.9, 64 40.7 -> 39.7;
//     16384 x 2048 at 24 14.7 -> 13.1, 137 21.6 -> 20.9; 4096 x 4096 at 24 10.1 -> 8.0, 64 10.8 -> 9.2; 2048 x 8192 at 24 8.9 -> 7.9;
//     8192 x 8192 at 24 25.3 -> 21.9, 225 in four slices 42.3 -> 40.7 (51.5 if an XCD's start at one place); 22016 x 4096 at 137 48.9 -> 47.5;
//     but 2560 x 2560 at 97, slices of 8 chunks, 7.9 -> 8.2: those stay in step.  A K range for every
//     wave, x in registers, was slower (64 to 70 at 137 rows): its waves wait for the weights each by itself;
//   * the 16x16 accumulator of (weight tile, token tile) holds 4 consecutive features of one token per
//     lane: one float4 store per accumulator into the slab.
#include "common.h"
#include "decode_epi.h"
#include "launchers.h"

namespace {

constexpr int MG_LDS = 160 * 1024;

typedef __attribute__((address_space(3))) void lds_t;

SYM_DEV __amdgpu_buffer_rsrc_t mg_rsrc(const void* base, long long bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0,
                                           (int)(bytes < 0x7fffffffLL ? bytes : 0x7fffffffLL), 0x00020000);
}

SYM_DEV void mg_dma(__amdgpu_buffer_rsrc_t r, int voff, int soff, char* lds) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_t*)lds, 16, voff, soff, 0, 0);
}

// non-temporal (aux = 2) LDS-DMA for the once-read weight stream
SYM_DEV void mg_dma_nt(__amdgpu_buffer_rsrc_t r, int voff, int soff, char* lds) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_t*)lds, 16, voff, soff, 0, 2);
}

// CT weight tiles, WV waves of RW of them.  A chunk's 2 MT x DMAs and 2 CT weight DMAs, 1 KB each, go round the waves; x's last ones
// twice where they do not divide
template <int MT, int CT, int WV>
struct MgCfg {
  static constexpr int RW = CT / WV;
  static constexpr int XB = 16 * MT * 128;                   // x bytes of one 64-deep chunk
  static constexpr int WB = CT * 2 * 1024;                   // weight bytes of one chunk (2 blocks per tile)
  static constexpr int SLOT = XB + WB;
  static constexpr int SLOTS = MG_LDS / SLOT > 8 ? 8 : MG_LDS / SLOT;
  static constexpr int D = SLOTS - 1;                        // chunks in flight ahead of the computed one
  static constexpr int NX = (2 * MT + WV - 1) / WV;          // x, weight DMA instructions per wave per chunk
  static constexpr int NB = 2 * RW;
  static constexpr int NDMA = NX + NB;
  static constexpr int VM_KEEP = (D - 1) * NDMA;             // younger DMAs left in flight at the wait
  static_assert(CT == RW * WV && D >= 1 && VM_KEEP <= 63, "mgemm config");
};

// MT: 16-token tiles (M <= 16 MT); CT: 16-row weight tiles.  Weights MFMA-preshuffled
// (models/layout.py::preshuffle): block (t, kb) = 16 rows x 32 k, 1 KB in fragment order.
// EPI < 0: the k split's fp32 slab is the output (the consumer kernel sums the slabs).  EPI >= 0: a fused
// consumer (decode_epi.h): with one split the accumulators go straight to epilogue<EPI>; with S splits every
// workgroup stores its slab, and the LAST of the S workgroups of a column group (agent-scope release /
// acquire around a per-group counter) sums the S
// slabs of its columns in the accumulator layout, applies the deferred-RMSNorm row scale (e.ss_in) and runs
// the epilogue -- the separate rope_cache / add+RMSNorm / SwiGLU launches of the slab path disappear.
// `counters` [N / (16 CT)] start at zero and are re-armed by the last arriver (graph-replay safe).
template <int MT, int CT, int EPI, int WV>
__global__ __launch_bounds__(64 * WV, 1) void mgemm_kernel(const bf16* __restrict__ x, const bf16* __restrict__ W,
                                                           float* __restrict__ y, int M, int N, int K, int kslice,
                                                           DecodeEpi e, int* __restrict__ counters) {
  using C = MgCfg<MT, CT, WV>;
  constexpr int RW = C::RW;
  __shared__ __attribute__((aligned(1024))) char smem[C::SLOTS * C::SLOT];
  asm volatile("" ::: "a0");  // accumulators may live in AGPRs

  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int split = blockIdx.y;
  const int k0 = split * kslice;
  const int nch = kslice / 64;
  const int tile0 = blockIdx.x * CT + wid * RW;  // first 16-row weight tile of this wave

  // ---- x DMA: wave w fills rows (NX w + i) * 8 .. + 8 of each chunk; lane -> (row lane >> 3, 16-B chunk
  // lane & 7), source chunk swizzled by (row >> 1) & 7.  Rows >= M read as zeros (buffer range).
  const __amdgpu_buffer_rsrc_t rx = mg_rsrc(x, (long long)M * K * 2);
  int vx[C::NX];
#pragma unroll
  for (int i = 0; i < C::NX; ++i) {
    const int row = min(C::NX * wid + i, 2 * MT - 1) * 8 + (lane >> 3);
    vx[i] = row * K * 2 + 16 * ((lane & 7) ^ ((row >> 1) & 7)) + k0 * 2;
  }
  // ---- weight DMA: block (tile, 2c + s) -> its 1 KB LDS block, lane-linear; wave w fills blocks NB w + i of the chunk's 2 CT.
  // Tiles past N (EPI_ARGMAX) read zeros (buffer range)
  const __amdgpu_buffer_rsrc_t rw = mg_rsrc(W + (long long)blockIdx.x * CT * 16 * K, (long long)min(16 * CT, N - (int)blockIdx.x * CT * 16) * K * 2);
  int vw[C::NB];
#pragma unroll
  for (int i = 0; i < C::NB; ++i) {
    const int b = C::NB * wid + i;
    vw[i] = ((b >> 1) * (K / 32) + k0 / 32 + (b & 1)) * 1024 + lane * 16;
  }

  // (of a few chunks, in step.  Spread also where x is past an L2, whose slices of K are not)
  const int turn = nch < 16 ? 0 : first_chunk(blockIdx.x + gridDim.x * split, nch, 0);
  auto issue = [&](int c, int slot) {
    c = c + turn < nch ? c + turn : c + turn - nch;
    const int xo = c * 128, wo = c * 2048;
#pragma unroll
    for (int i = 0; i < C::NX; ++i) mg_dma(rx, vx[i], xo, smem + slot * C::SLOT + min(C::NX * wid + i, 2 * MT - 1) * 1024);
    char* const dw = smem + slot * C::SLOT + C::XB;
#pragma unroll
    for (int i = 0; i < C::NB; ++i) mg_dma_nt(rw, vw[i], wo, dw + (C::NB * wid + i) * 1024);
  };

  // ---- fragment reads: x lane holds token (16 mt + (lane & 15)), k 8 (lane >> 4) .. + 8 of step s
  // (swizzled chunk 4 s + (lane >> 4)); weight block reads are lane-linear (fragment order)
  const int fr = lane & 15;
  const int xo0 = fr * 128 + 16 * ((lane >> 4) ^ ((fr >> 1) & 7));
  const int xo1 = fr * 128 + 16 * ((4 + (lane >> 4)) ^ ((fr >> 1) & 7));
  const int wo_l = C::XB + lane * 16;

  // EPI_ARGMAX sums all of K here, in parts of 256, of a short K 128: longer chains lose bits (K = 2048, 32768 outputs: one chain
  // 1.9e-7 of the result off, parts of 512 1.3e-7, 256 1.0e-7)
  constexpr bool PARTS = EPI == DECODE_EPI_ARGMAX;
  f32x4 acc[RW][MT], total[PARTS ? RW : 1][PARTS ? MT : 1];
#pragma unroll
  for (int rt = 0; rt < RW; ++rt)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      acc[rt][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
      if constexpr (PARTS) total[rt][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
    }

  struct Frag {
    bf16x8 w[RW], x[MT];
  };
  Frag f0, f1;      // a chunk's two 32-deep steps
  // reads step s of a chunk's slot into `next`, between the products of `now`: with one wave a SIMD nothing else hides a read
  auto step = [&](Frag& next, int slot, int s, const Frag& now, bool reads, bool multiplies) __attribute__((always_inline)) {
    const char* const sb = smem + slot * C::SLOT;
    constexpr int READS = RW + MT, PER = (READS + MT - 1) / MT;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
      for (int u = 0; u < PER; ++u) {
        const int i = PER * mt + u;
        if (!reads || i >= READS) continue;
        if (i < RW) next.w[i] = *(const bf16x8*)(sb + wo_l + (2 * (wid * RW + i) + s) * 1024);
        else next.x[i - RW] = *(const bf16x8*)(sb + (s ? xo1 : xo0) + (i - RW) * 2048);
      }
      if (multiplies) {
#pragma unroll
        for (int rt = 0; rt < RW; ++rt) acc[rt][mt] = mfma16(now.w[rt], now.x[mt], acc[rt][mt]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };

  // deferred-RMSNorm row scales (EPI >= 0 with e.ss_in): tpr threads per row sum the producer's partials.
  // Loads issued before the DMA prologue, summed after it (the DMAs stay in flight); the scale lives in one
  // register until the epilogue.  (Computed in the epilogue with one wave-serial loop per row, it cost
  // ~13 us per launch at 64 rows: 16 dependent load round trips per wave.)
  float rn_reg = 1.f;
  int rn_row = -1;
  float rn_part = 0.f;
  int tpr = 1;
  if constexpr (EPI >= 0) {
    if (e.ss_in) {
      while (tpr < 64 && tpr * 2 * M <= 64 * WV) tpr *= 2;
      const int row = threadIdx.x / tpr, sub = threadIdx.x % tpr;
      if (row < M) {
        rn_row = row;
        const float* sp = e.ss_in + (long long)row * e.ss_tiles;
        if (e.ss_tiles % (4 * tpr) == 0) {
          const float4* s4 = reinterpret_cast<const float4*>(sp);
#pragma unroll 8
          for (int i = sub; i < e.ss_tiles / 4; i += tpr) {
            const float4 q = s4[i];
            rn_part += (q.x + q.y) + (q.z + q.w);
          }
        } else {
#pragma unroll 8
          for (int i = sub; i < e.ss_tiles; i += tpr) rn_part += sp[i];
        }
      }
    }
  }

  // prologue: every slot of the ring in flight
#pragma unroll
  for (int c = 0; c < C::SLOTS; ++c)
    if (c < nch) issue(c, c);

  if constexpr (EPI >= 0) {
    if (e.ss_in) {  // tpr consecutive lanes of one wave (tpr divides 64)
      for (int o = 1; o < tpr; o *= 2) rn_part += __shfl_xor(rn_part, o, 64);
      rn_reg = rsqrtf(rn_part * e.inv_d + e.eps);
    }
  }

  // chunk c lives in ring slot c % SLOTS.  Its second step is read while the first is multiplied, then this wave waits until
  // its DMAs of chunk c + 1 have landed (the younger ones stay in flight) and its reads of chunk c are in registers; behind the
  // barrier every wave's x rows of chunk c + 1 are visible and slot c is free: it is refilled with c + SLOTS.
  auto landed = [&](int c) {      // chunk c is; those up to c + D - 1 stay in flight
    if (c + C::D - 1 < nch) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(C::VM_KEEP) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  };
  if (C::SLOTS <= nch) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(C::VM_KEEP + C::NDMA < 63 ? C::VM_KEEP + C::NDMA : 63) : "memory");
  else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  step(f0, 0, 0, f1, true, false);
  const int part = K < 2048 ? 1 : 3;
  int slot = 0;
  for (int c = 0; c + 1 < nch; ++c) {
    const int after = slot == C::SLOTS - 1 ? 0 : slot + 1;
    step(f1, slot, 1, f0, true, true);
    landed(c + 1);
    __builtin_amdgcn_s_waitcnt(0xc07f);      // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (c + C::SLOTS < nch) issue(c + C::SLOTS, slot);
    step(f0, after, 0, f1, true, true);
    if (PARTS && (c & part) == part) {
#pragma unroll
      for (int rt = 0; rt < (PARTS ? RW : 0); ++rt)
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

  // ---- epilogue: lane holds features 16 t + 4 (lane >> 4) .. + 3 of token 16 mt + (lane & 15)
  const int S = gridDim.y;
  float* ys = y + (long long)split * M * N;
  if (EPI < 0 || S > 1) {
#pragma unroll
    for (int rt = 0; rt < RW; ++rt) {
      const int n = 16 * (tile0 + rt) + 4 * (lane >> 4);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const int m = 16 * mt + (lane & 15);
        if (m >= M) continue;
        const float4 f4 = make_float4(acc[rt][mt][0], acc[rt][mt][1], acc[rt][mt][2], acc[rt][mt][3]);
        if constexpr (EPI >= 0) {  // read back in this launch by the last split: write-through (see below)
          unsigned long long* q = reinterpret_cast<unsigned long long*>(ys + (long long)m * N + n);
          const unsigned long long* w64 = reinterpret_cast<const unsigned long long*>(&f4);
          __hip_atomic_store(q, w64[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          __hip_atomic_store(q + 1, w64[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        } else {
          *reinterpret_cast<float4*>(ys + (long long)m * N + n) = f4;
        }
      }
    }
  }
  if constexpr (EPI >= 0) {
    // LDS ring is free once every wave is past its last compute: row scales + the "last arriver" word
    __syncthreads();
    float* rn = reinterpret_cast<float*>(smem);
    int* last = reinterpret_cast<int*>(smem + 1024 * 4);
    if (S > 1) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's slab stores are out
      __syncthreads();
      // hand-off without L2 maintenance: write-through slab stores drained above,
      // relaxed agent add, the last split reads the slabs with agent-scope (L2-bypassing) loads.  Agent
      // fences here wrote back / invalidated the XCD's whole L2 once per workgroup: the fused general path
      // ran 6.22 vs 4.43 ms per 64-client step (profiles/r3/mg_fused_ab.jsonl).
      if (threadIdx.x == 0) {
        const int got = __hip_atomic_fetch_add(counters + blockIdx.x, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const int is_last = got == S - 1;
        if (is_last) __hip_atomic_store(counters + blockIdx.x, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        *last = is_last;
      }
      __syncthreads();
      if (!*last) return;
    }
    // deferred-RMSNorm row scales of the input rows (summed before the main loop)
    if (e.ss_in) {
      if (rn_row >= 0 && threadIdx.x % tpr == 0) rn[rn_row] = rn_reg;
      __syncthreads();
    }
#pragma unroll
    for (int rt = 0; rt < RW; ++rt) {
      if (EPI == DECODE_EPI_ARGMAX && 16 * (tile0 + rt) >= N) continue;
      const int n = 16 * (tile0 + rt) + 4 * (lane >> 4);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const int m = 16 * mt + (lane & 15);
        const bool mok = m < M;
        f32x4 v = acc[rt][mt];
        if constexpr (PARTS) v += total[rt][mt];
        if (S > 1) {
          v = f32x4{0.f, 0.f, 0.f, 0.f};
          if (mok)
            for (int sp = 0; sp < S; ++sp) {  // fixed split order: bitwise reproducible
              const unsigned long long* q =
                  reinterpret_cast<const unsigned long long*>(y + ((long long)sp * M + m) * N + n);
              unsigned long long r[2];
              r[0] = __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
              r[1] = __hip_atomic_load(q + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
              const float* p = reinterpret_cast<const float*>(r);
              v[0] += p[0];
              v[1] += p[1];
              v[2] += p[2];
              v[3] += p[3];
            }
        }
        const float sc = (e.ss_in && mok) ? rn[m] : 1.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] *= sc;
        epilogue<EPI>(e, v, tile0 + rt, m, mok, lane >> 4, N);
      }
    }
  }
}

template <int MT, int CT, int EPI, int WV = 4>
void launch_ct(const bf16* x, const bf16* W, float* y, int M, int N, int K, int S, const DecodeEpi& e, int* counters,
               hipStream_t s) {
  mgemm_kernel<MT, CT, EPI, WV><<<dim3(N / (16 * CT), S), 64 * WV, 0, s>>>(x, W, y, M, N, K, K / S, e, counters);
}

template <int MT, int EPI>
void launch_mt(const bf16* x, const bf16* W, float* y, int M, int N, int K, int S, int rw, const DecodeEpi& e,
               int* counters, hipStream_t s) {
  if constexpr (EPI == DECODE_EPI_SWIGLU && MT <= 12) {
    // Seven waves where their columns fill the CUs better than four waves' do (widths of 7 x 2^n, as 2 x 14336): a CU's intake
    // is what bounds the stream.  28672 x 4096, 224 workgroups of four waves / 256 of seven, us: 20 rows 42.6 / 38.7, 64
    // 41.3 / 40.5, 112 48.0 / 45.0, 137 53.0 / 50.9, 192 65.4 / 62.9; 57344 x 8192 at 96 rows 177 / 175
    if (S == 1 && N % 112 == 0 && N / 112 <= 256 && N / 112 > N / (64 * rw)) return launch_ct<MT, 7, EPI, 7>(x, W, y, M, N, K, S, e, counters, s);
    if (S == 1 && N % 224 == 0 && N / 224 <= 256 && N / 224 > N / (64 * rw)) return launch_ct<MT, 14, EPI, 7>(x, W, y, M, N, K, S, e, counters, s);
  }
  if constexpr (EPI < 0) {
    // ... and three or six waves of a tile each for widths of 3 x 2^n, by the same rule (4 / 3 tiles, us: 6144 x 4096 at 40 rows
    // 13.1 / 10.9, 64 13.9 / 12.5; 3072 x 2048 at 40 5.8 / 5.4, 240 11.5 / 10.9; 8 / 6 tiles: 6144 x 4096 at 100 rows 15.2 / 14.6,
    // 137 17.7 / 16.2, 240 24.4 / 21.5)
    if (rw == 1 && N % 48 == 0 && N / 48 * S <= 256) return launch_ct<MT, 3, EPI, 3>(x, W, y, M, N, K, S, e, counters, s);
    if (rw == 2 && N % 96 == 0 && N / 96 * S <= 256) return launch_ct<MT, 6, EPI, 6>(x, W, y, M, N, K, S, e, counters, s);
  }
  if constexpr (MT <= 8) {  // 144 to 256 rows: at most 2 weight tiles per wave (accumulators + LDS ring)
    if (rw == 3) return launch_ct<MT, 12, EPI>(x, W, y, M, N, K, S, e, counters, s);
    if (rw == 4) return launch_ct<MT, 16, EPI>(x, W, y, M, N, K, S, e, counters, s);
  }
  if (rw == 1) launch_ct<MT, 4, EPI>(x, W, y, M, N, K, S, e, counters, s);
  else launch_ct<MT, 8, EPI>(x, W, y, M, N, K, S, e, counters, s);
}

// Row tiles by EPI: steps of 16 rows up to 192 and of 32 above where the form is used by default (the others, coarser)
template <int EPI>
void launch_epi_m(const bf16* x, const bf16* W, float* y, int M, int N, int K, int S, int rw, const DecodeEpi& e,
                  int* counters, hipStream_t s) {
  const int tiles = (M + 15) / 16;
#define MG_TILES(t) \
  if (tiles <= t) return launch_mt<t, EPI>(x, W, y, M, N, K, S, rw, e, counters, s)
  MG_TILES(2);
  if constexpr (EPI < 0 || EPI == DECODE_EPI_SWIGLU) {
    MG_TILES(3); MG_TILES(4); MG_TILES(5); MG_TILES(6); MG_TILES(7); MG_TILES(8); MG_TILES(9); MG_TILES(10); MG_TILES(11);
    MG_TILES(12); MG_TILES(14);
  } else {
    MG_TILES(4); MG_TILES(8);
  }
#undef MG_TILES
  launch_mt<16, EPI>(x, W, y, M, N, K, S, rw, e, counters, s);
}

template <int CT>
void launch_argmax(const bf16* x, const bf16* W, int M, int N, int K, const DecodeEpi& e, hipStream_t s) {
  const int groups = (N + 16 * CT - 1) / (16 * CT);
#define MG_ARGMAX(t) \
  mgemm_kernel<t, CT, DECODE_EPI_ARGMAX, 4><<<groups, 256, 0, s>>>(x, W, nullptr, M, N, K, K, e, nullptr)
  if (M <= 32) MG_ARGMAX(2);
  else if (M <= 48) MG_ARGMAX(3);
  else MG_ARGMAX(4);
#undef MG_ARGMAX
}

}  // namespace

// Many outputs of 17 to 64 rows (an lm_head) in whole columns, rounds of workgroups of 64 outputs, or of 128.  The decode GEMM reads
// x once for 16 outputs: with its launch that reduces the keys, us, it on either layout's better one / 64 / 128 outputs: 32768 x
// 2048 at 24 rows 34.3 / 31.7 / 36.0, 64 43.2 / 36.5 / 38.8; 32768 x 4096 at 17 57.8 / 55.3 / 56.2, 64 67.3 / 63.4 / 57.0; 32000 x
// 8192 at 48 119 / 97 / 92; 128256 x 2048 at 64 150 / 123 / 126; 128256 x 4096 at 32 195 / 193 / 188, 64 233 / 235 / 203; 64000 x
// 1024 at 17 34.1 / 35.6 / 36.0, 64 49 / 44 / 43.  So 128 past 32 rows of a long K, and where 64 make a second round of few (20480 x
// 2048 at 24 rows 29.5 / 26.5 / 25.1, 24576 x 4096 at 48 54.5 / 50.4 / 42.1), but 64 in one round (16384 x 4096 at 64 51.1 / 34.1 /
// 40.7).  Fewer outputs leave CUs idle (10240 x 8192 at 17 rows 51.4 / 33.8, but 8192 x 4096 20.5 / 23.1) and stay with the decode GEMM, on this layout too (transformer.py::_lm_head).
bool launch_mgemm_argmax(const bf16* x, const bf16* W, int M, int N, int K, const DecodeEpi& e, hipStream_t s) {
  if (!e.wshuf || M <= 16 || M > 64 || K % 64 || K < 1024 || K > 1 << 20 || N % 16 || N < 10240) return false;
  if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(W)) % 16) return false;
  const int groups = (N + 63) / 64;
  if (groups > 256 && (groups < 448 || (M > 32 && K > 2048))) launch_argmax<8>(x, W, M, N, K, e, s);
  else launch_argmax<4>(x, W, M, N, K, e, s);
  return true;
}

void launch_mgemm(const bf16* x, const bf16* Wshuf, float* y, int M, int N, int K, int S, int rw, hipStream_t s) {
  launch_epi_m<-1>(x, Wshuf, y, M, N, K, S, rw, DecodeEpi{}, nullptr, s);
}

void launch_mgemm_epi(int epi, const bf16* x, const bf16* Wshuf, float* y, int M, int N, int K, int S, int rw,
                      const DecodeEpi& e, int* counters, hipStream_t s) {
  switch (epi) {
    case DECODE_EPI_QKV: launch_epi_m<DECODE_EPI_QKV>(x, Wshuf, y, M, N, K, S, rw, e, counters, s); break;
    case DECODE_EPI_RESID: launch_epi_m<DECODE_EPI_RESID>(x, Wshuf, y, M, N, K, S, rw, e, counters, s); break;
    case DECODE_EPI_SWIGLU: launch_epi_m<DECODE_EPI_SWIGLU>(x, Wshuf, y, M, N, K, S, rw, e, counters, s); break;
    default: launch_epi_m<DECODE_EPI_F32>(x, Wshuf, y, M, N, K, S, rw, e, counters, s); break;
  }
}
