// Routed feed-forward with squared-ReLU (or plain) experts: router, expert segments, expert products.
//
//   route_topk      logits x . Wr[e] + bias in fp32, the k largest, weights = softmax over the chosen ones, and the places of
//                   the routed rows in expert order (segment bounds, token of every place, place of every choice)
//   expert_linear   y[place] = act(W[e] x[src[place]]) over the expert segments; rows are gathered where they are read, so no
//                   permuted copy of the activations exists, and the squared ReLU is the epilogue of the up product
//
// Router in bf16: 16 tokens x 16 experts per MFMA, the waves of a workgroup split the width and meet in LDS (the products of
// bf16 values and their sums are exact to fp32 accumulation).  A step of at most 16 tokens is one workgroup, which then also
// lays out the segments; larger steps take one more launch.
// Expert products in bf16: weight-streaming kernels for few rows per expert (a wave per 16 weight rows and width slice, the
// rows of the segment as the other MFMA operand; persistent where there are many weights), and for prompt steps a 128 x 128 tile kernel and a persistent one of 256 x 256,
// staged through LDS by direct loads.  Other shapes and fp32: the all-shapes segment product of glu_moe.hip.
#include "common.h"
#include "direct_lds.h"
#include "hybrid_launchers.h"
#include "latent_launchers.h"
#include "wave_dot.h"

#include <algorithm>
#include <array>
#include <type_traits>

namespace {

constexpr int NT = 256;
constexpr int MAX_E = 1024;      // experts the segment layout handles
constexpr int PLAN_NT = 1024;

// ---- router --------------------------------------------------------------------------------------------------------------
// One wave: the k largest of z[0 .. E) (LDS), ties to the lowest index; ids / softmax weights of the chosen to global
SYM_DEV void choose(float* z, int E, int k, int lane, int* ids, float* w) {
  float zmax = 0.f, sum = 0.f;
  for (int j = 0; j < k; ++j) {
    float best = -INFINITY;
    int bi = 0x7fffffff;
    for (int e = lane; e < E; e += 64) {
      const float v = z[e];
      if (v > best) { best = v; bi = e; }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const float ob = __shfl_xor(best, o, 64);
      const int oi = __shfl_xor(bi, o, 64);
      if (ob > best || (ob == best && oi < bi)) { best = ob; bi = oi; }
    }
    if (bi >= E) bi = j;       // only with non-finite logits: keep the id a valid segment index for the kernels downstream
    if (j == 0) zmax = best;
    const float p = j == 0 || zmax == -INFINITY ? 1.f : expf(best - zmax);     // (no finite logit: equal weights)
    sum += p;
    if (lane == 0) {
      ids[j] = bi;
      w[j] = p;
    }
    if ((bi & 63) == lane) z[bi] = -INFINITY;      // (the lane that scans this entry)
  }
  const float inv = 1.f / sum;
  if (lane == 0)
    for (int j = 0; j < k; ++j) w[j] *= inv;
}

// Segment layout by one workgroup of BT threads.  Items lo .. hi - 1 of the R choices get their places; the counts run over
// all of them (tot) and over those before lo (before), so workgroups that share the items out agree on every segment.
// LDS: 3 E ints.
template <int BT>
SYM_DEV void layout_segments(const int* __restrict__ ids, int R, int E, int k, int lo, int hi, int* lds,
                             int* __restrict__ offsets, int* __restrict__ dst, int* __restrict__ src) {
  int *tot = lds, *before = lds + E, *cur = lds + 2 * E;
  for (int e = threadIdx.x; e < E; e += BT) tot[e] = 0, before[e] = 0;
  __syncthreads();
  for (int a = threadIdx.x; a < R; a += BT) {
    const int e = ids[a];
    atomicAdd(&tot[e], 1);
    if (a < lo) atomicAdd(&before[e], 1);
  }
  __syncthreads();
  if (threadIdx.x < 64) {        // exclusive sums, 64 experts at a time
    const int lane = threadIdx.x;
    int carry = 0;
    for (int e0 = 0; e0 < E; e0 += 64) {
      const int e = e0 + lane;
      const int n = e < E ? tot[e] : 0;
      int s = n;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int t = __shfl_up(s, o, 64);
        if (lane >= o) s += t;
      }
      if (e < E) {
        cur[e] = carry + s - n + before[e];
        if (lo == 0) offsets[e] = carry + s - n;
      }
      carry += __shfl(s, 63, 64);
    }
    if (lo == 0 && lane == 0) offsets[E] = carry;
  }
  __syncthreads();
  for (int a = lo + threadIdx.x; a < hi; a += BT) {
    const int pos = atomicAdd(&cur[ids[a]], 1);
    dst[a] = pos;
    src[pos] = a / k;
  }
}

__global__ __launch_bounds__(PLAN_NT) void expert_layout_kernel(const int* __restrict__ ids, int R, int E, int k,
                                                                int* __restrict__ offsets, int* __restrict__ dst,
                                                                int* __restrict__ src) {
  extern __shared__ int plds[];
  const int lo = blockIdx.x * 4 * PLAN_NT;
  layout_segments<PLAN_NT>(ids, R, E, k, lo, min(R, lo + 4 * PLAN_NT), plds, offsets, dst, src);
}

// grid ceil(T / 16), NW waves; NE expert tiles of 16 (E <= 16 NE), d % 32 == 0.  Dynamic LDS: NW NE 256 floats (partial
// logits) or, reused, 16 E floats + the layout's counters; PLAN: the single workgroup lays out the segments as well.
// a.runs: every wave takes one run of the width (d % (32 NW) == 0), and the hardware exponential: the sums and weights of
// moe_router_kernel and moe_route_kernel, to the bit.
// NORM (PLAN; d % 512 == 0, d <= 2048): x = RMSNorm(resid) is made here, a wave a row, and written to x for the experts; it meets
// the router in LDS, behind the partial logits (rows 16 B longer, so a fragment's 16 rows lie in different banks).
// Latency is all of it: 8 rows of 2048, 16 experts 8.6 -> 6.8 us with the norm's launch.  A token's choices are counted places of
// its logits: the k reductions over the wave that stood here were a chain of 12 lane exchanges each (4 of 16, alone 8.7 -> 6.5).
template <int NW, int NE, bool PLAN, bool NORM = false>
__global__ __launch_bounds__(64 * NW) void route_mfma_kernel(RouteArgs a) {
  extern __shared__ __attribute__((aligned(16))) float part[];
  __shared__ int chosen[PLAN ? 1024 : 1];      // PLAN: the workgroup's choices (at most 16 tokens x 64)
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, j = lane & 15, hq = lane >> 4;
  const int t0 = 16 * blockIdx.x, d = a.d, E = a.E;
  const bf16* x = reinterpret_cast<const bf16*>(a.x) + (long long)min(t0 + j, a.T - 1) * d + 8 * hq;
  const bf16* w[NE];
  f32x4 acc[NE];
#pragma unroll
  for (int n = 0; n < NE; ++n) {
    w[n] = reinterpret_cast<const bf16*>(a.Wr) + (long long)min(16 * n + j, E - 1) * d + 8 * hq;
    acc[n] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const int first = a.runs ? wave * (d / NW) : 32 * wave, last = a.runs ? first + d / NW : d, step = a.runs ? 32 : 32 * NW;
  constexpr int AHEAD = NORM && NW == 16 ? 4 : 0;      // (all of a wave's steps)
  Pack8 ahead[NE][AHEAD + 1];
  if constexpr (NORM) {
    bf16* rows = reinterpret_cast<bf16*>(part + NW * NE * 256);
    const int pitch = d + 8;
#pragma unroll
    for (int i = 0; i < AHEAD; ++i)
#pragma unroll
      for (int n = 0; n < NE; ++n)
        ahead[n][i].u = *reinterpret_cast<const uint4*>(w[n] + min(first + i * step, last - 32));
    for (int t = wave; t < a.T; t += NW) {
      const float* from = a.resid + (long long)t * d + 8 * lane;
      float v[4][8], ss = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (512 * i < d) load8f(from + 512 * i, v[i]);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (512 * i < d)
#pragma unroll
          for (int u = 0; u < 8; ++u) ss += v[i][u] * v[i][u];
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) ss += __shfl_xor(ss, o, 64);
      const float inv = rsqrtf(ss / (float)d + a.eps);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (512 * i < d) {
          float g[8];
          load8(reinterpret_cast<const bf16*>(a.norm) + 512 * i + 8 * lane, g);
          Pack8 o;
#pragma unroll
          for (int u = 0; u < 8; ++u) o.v[u] = (bf16)(g[u] * (v[i][u] * inv));
          *reinterpret_cast<uint4*>(rows + t * pitch + 512 * i + 8 * lane) = o.u;
          *reinterpret_cast<uint4*>(const_cast<bf16*>(reinterpret_cast<const bf16*>(a.x)) + (long long)t * d + 512 * i + 8 * lane) = o.u;
        }
    }
    __syncthreads();
    x = rows + min(j, a.T - 1) * pitch + 8 * hq;
  }
  if constexpr (AHEAD > 0) {
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) {
      const int c = first + i * step;
      if (c >= last) break;
      Pack8 xf;
      xf.u = *reinterpret_cast<const uint4*>(x + c);
#pragma unroll
      for (int n = 0; n < NE; ++n) acc[n] = mfma16(ahead[n][i].v, xf.v, acc[n]);
    }
  } else
#pragma unroll 4
  for (int c = first; c < last; c += step) {
    Pack8 xf;
    xf.u = *reinterpret_cast<const uint4*>(x + c);
#pragma unroll
    for (int n = 0; n < NE; ++n) {
      Pack8 wf;
      wf.u = *reinterpret_cast<const uint4*>(w[n] + c);
      acc[n] = mfma16(wf.v, xf.v, acc[n]);      // lane: token j, experts 16 n + 4 hq + 0..3
    }
  }
#pragma unroll
  for (int n = 0; n < NE; ++n)
    *reinterpret_cast<f32x4*>(part + (((wave * NE + n) * 16 + j) * 16 + 4 * hq)) = acc[n];
  __syncthreads();
  // the waves' partial logits of (token, expert) meet in the first slab: [NE][16 tokens][16 experts]
  for (int i = threadIdx.x; i < NE * 256; i += 64 * NW) {
    float s = part[i];
    for (int v = 1; v < NW; ++v) s += part[v * NE * 256 + i];
    const int e = 16 * (i >> 8) + (i & 15);
    part[i] = e < E ? s + (a.bias ? a.bias[e] : 0.f) : -INFINITY;
  }
  __syncthreads();
  for (int t = wave; t < 16; t += NW) {
    if (t0 + t >= a.T) break;
    float z = lane < 16 * NE ? part[((lane >> 4) * 16 + t) * 16 + (lane & 15)] : -INFINITY;   // (E <= 64: one per lane)
    if (z != z) z = -INFINITY;      // a NaN logit never wins
    // a logit's place: how many stand before it (larger, or equal and of a lower index)
    int place = 0;
#pragma unroll
    for (int e = 0; e < 16 * NE; ++e) {
      const float v = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(z), e));
      place += v > z || (v == z && e < lane);
    }
    const int to = 4 * (lane < 16 * NE ? place : lane);
    const float best = __uint_as_float(__builtin_amdgcn_ds_permute(to, __float_as_uint(z)));      // lane: the choice of this place
    int my = __builtin_amdgcn_ds_permute(to, lane);
    if (lane >= __popcll(__ballot(z > -INFINITY))) my = lane;   // only with non-finite logits: a valid segment index
    const float zmax = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(best)));
    const float mine = lane == 0 || zmax == -INFINITY ? 1.f : a.runs ? __expf(best - zmax) : expf(best - zmax);
    float sum = 0.f;
    for (int q = 0; q < a.k; ++q) sum += __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(mine), q));
    if (lane < a.k) {
      const long long o = (long long)(t0 + t) * a.k + lane;
      a.ids[o] = my;
      a.w[o] = mine / sum;
      if constexpr (PLAN) chosen[t * a.k + lane] = my;
    }
  }
  if constexpr (PLAN) {
    __syncthreads();      // (the partial logits are done with)
    layout_segments<64 * NW>(chosen, a.T * a.k, E, a.k, 0, a.T * a.k, reinterpret_cast<int*>(part), a.offsets, a.dst, a.src);
  }
}

// any width, both dtypes, E <= MAX_E: a workgroup per token, a wave per expert in turn
template <typename T>
__global__ __launch_bounds__(NT) void route_rows_kernel(RouteArgs a) {
  extern __shared__ float z[];
  const int t = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const T* x = reinterpret_cast<const T*>(a.x) + (long long)t * a.d;
  for (int e = wave; e < a.E; e += NT / 64) {
    const float s = wave_dot<T>(x, reinterpret_cast<const T*>(a.Wr) + (long long)e * a.d, a.d, lane);
    if (lane == 0) z[e] = s + (a.bias ? a.bias[e] : 0.f);
  }
  __syncthreads();
  if (wave == 0) choose(z, a.E, a.k, lane, a.ids + (long long)t * a.k, a.w + (long long)t * a.k);
}

// ---- expert products -----------------------------------------------------------------------------------------------------
SYM_DEV float relu2f(float v) {
  v = fmaxf(v, 0.f);
  return v * v;
}

enum { EPI_BF16 = 0, EPI_RELU2 = 1, EPI_GLU = 2, EPI_F32 = 3 };   // EPI_GLU: W's rows are [gate | up], y = silu(gate) * up

// Few rows per expert: grid (ceil(N / 16), E), NW waves.  A workgroup owns 16 outputs of one expert (EPI_GLU: their gate and up
// rows, so the pair meets in LDS); its waves take the width's 64-element steps in turn (weights streamed once, straight into
// registers), multiply them with up to 16 MT rows of the segment per pass, and their sums meet in LDS.  K % 32 == 0.
template <int MT, int NW, int U, int EPI>
__global__ __launch_bounds__(64 * NW) void expert_stream_kernel(ExpertArgs a) {
  constexpr int G = EPI == EPI_GLU ? 2 : 1;       // weight rows of an output
  __shared__ float part[NW][G * MT * 256];
  const int e = blockIdx.y, n0 = 16 * blockIdx.x;
  const int s0 = a.offsets[e], s1 = min(a.offsets[e + 1], a.R);
  if (s0 >= s1) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), j = lane & 15, hq = lane >> 4;
  const int K = a.K, N = a.N;
  const bf16* w[G];
#pragma unroll
  for (int g = 0; g < G; ++g)
    w[g] = reinterpret_cast<const bf16*>(a.W) + ((long long)(G * e + g) * N + min(n0 + j, N - 1)) * K + 8 * hq;
  for (int r0 = s0; r0 < s1; r0 += 16 * MT) {
    // 64 elements of every weight row per step: whole 128-byte lines.  U steps are in flight, the first ones before the rows
    // are looked up.
    Pack8 wf[U][2][G];
    auto load = [&](int c) {
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int v = 0; v < 2; ++v)
#pragma unroll
          for (int g = 0; g < G; ++g) wf[u][v][g].w = ld_nt16(w[g] + c + 64 * NW * u + 32 * v);
      __builtin_amdgcn_sched_barrier(0);
    };
    int c = 64 * wave;
    bool more = c + 64 * NW * (U - 1) + 64 <= K;
    if (more) load(c);
    const bf16* x[MT];
    f32x4 acc[G][MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const int r = min(r0 + 16 * m + j, s1 - 1);
      x[m] = reinterpret_cast<const bf16*>(a.x) + (long long)(a.src ? a.src[r] : r) * K + 8 * hq;
#pragma unroll
      for (int g = 0; g < G; ++g) acc[g][m] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    while (more) {
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        Pack8 xf[U][2];
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int v = 0; v < 2; ++v) xf[u][v].u = *reinterpret_cast<const uint4*>(x[m] + c + 64 * NW * u + 32 * v);
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int v = 0; v < 2; ++v)
#pragma unroll
            for (int g = 0; g < G; ++g)
              acc[g][m] = mfma16(wf[u][v][g].v, xf[u][v].v, acc[g][m]);     // lane: row j, outputs n0 + 4 hq + 0..3
      }
      c += 64 * NW * U;
      more = c + 64 * NW * (U - 1) + 64 <= K;
      if (more) load(c);
    }
    for (; c < K; c += 64 * NW)
#pragma unroll
      for (int v = 0; v < 2; ++v) {
        if (c + 32 * v >= K) break;
        Pack8 wt[G];
#pragma unroll
        for (int g = 0; g < G; ++g) wt[g].w = ld_nt16(w[g] + c + 32 * v);
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          Pack8 xf;
          xf.u = *reinterpret_cast<const uint4*>(x[m] + c + 32 * v);
#pragma unroll
          for (int g = 0; g < G; ++g) acc[g][m] = mfma16(wt[g].v, xf.v, acc[g][m]);
        }
      }
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int m = 0; m < MT; ++m) *reinterpret_cast<f32x4*>(&part[wave][(g * MT + m) * 256 + j * 16 + 4 * hq]) = acc[g][m];
    __syncthreads();
    for (int i = threadIdx.x; i < MT * 256; i += 64 * NW) {
      float s = part[0][i], t = G == 2 ? part[0][MT * 256 + i] : 0.f;
#pragma unroll
      for (int v = 1; v < NW; ++v) {
        s += part[v][i];
        if constexpr (G == 2) t += part[v][MT * 256 + i];
      }
      const int r = r0 + (i >> 4), n = n0 + (i & 15);
      if (r < s1 && n < N) {
        const long long at = (long long)r * N + n;
        if constexpr (EPI == EPI_F32) reinterpret_cast<float*>(a.y)[at] = s;
        else reinterpret_cast<bf16*>(a.y)[at] = (bf16)(EPI == EPI_GLU ? silu(s) * t : EPI == EPI_RELU2 ? relu2f(s) : s);
      }
    }
    __syncthreads();
  }
}

template <int MT, int NW, int U>
void launch_stream(const ExpertArgs& a, hipStream_t s) {
  dim3 grid((a.N + 15) / 16, a.E);
  if (a.glu) expert_stream_kernel<MT, NW, U, EPI_GLU><<<grid, 64 * NW, 0, s>>>(a);
  else if (a.relu2) expert_stream_kernel<MT, NW, U, EPI_RELU2><<<grid, 64 * NW, 0, s>>>(a);
  else if (a.f32_out) expert_stream_kernel<MT, NW, U, EPI_F32><<<grid, 64 * NW, 0, s>>>(a);
  else expert_stream_kernel<MT, NW, U, EPI_BF16><<<grid, 64 * NW, 0, s>>>(a);
}

// Prompt steps: tiles of BM rows x BN weight rows, waves in WR rows x WC columns, K in steps of 64 through two LDS stages filled by
// direct global -> LDS loads.  LDS rows are 128 B with the 16-byte chunk c stored at c ^ ((row >> 1) & 7) (swizzled on the
// load's source), so fragment reads do not conflict.  K % 64 == 0.
// EPI_GLU: half of a wave's weight rows are gate rows and half the up rows of the same outputs, so a pair meets in registers.
// The tile list is counted on the device; a workgroup without a tile exits before any barrier.  Tiles are dealt to the 8 XCDs
// in contiguous runs (workgroup i runs on XCD i % 8) and walk GN column tiles of every row tile of an expert before the next
// GN, so an expert's weights and a tile row's activations are shared in one L2 (16384 rows, 8 experts of 2 x 14336 x 4096:
// 0.78 -> 1.13 PFLOP/s).
constexpr int GN = 8;

// outputs n .. n + 3 of a row (at: the first one's place); vec: N is a multiple of 4
template <bool F32, bool NT = false>
SYM_DEV void store_quad(void* y, long long at, f32x4 f, int n, int N, bool vec) {
  if constexpr (F32) {
    float* o = reinterpret_cast<float*>(y) + at;
    if (vec) {
      if (n < N) {
        if constexpr (NT) __builtin_nontemporal_store(f, reinterpret_cast<f32x4*>(o));
        else *reinterpret_cast<f32x4*>(o) = f;
      }
    } else {
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (n + u < N) o[u] = f[u];
    }
  } else {
    bf16* o = reinterpret_cast<bf16*>(y) + at;
    bf16x4 v;
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = (bf16)f[u];
    if (vec) {
      if (n < N) *reinterpret_cast<bf16x4*>(o) = v;
    } else {
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (n + u < N) o[u] = v[u];
    }
  }
}

// Few rows per expert, many weights: a workgroup per CU walks units of OUT outputs (EPI_GLU: 8, their gate and up rows, else 16) of
// up to 16 rows of one expert: unit t, t + gridDim.x, ..  A wave holds its share of a unit's weights and rows in registers (KB
// steps of 64 elements, K = 64 NW KB); the next unit's are loaded while a unit is multiplied, so the weights stream without a
// gap from one expert to the next.  The waves sum a unit's parts in turn, one barrier a unit (two buffers).  A lane knows the
// segment of expert `lane` and the units up to its end; the rows' places are kept in LDS.  E <= 64, R <= WALK_ROWS.  Bound by HBM:
// the weights of 15 of 16 experts, gated 2 x 1536 x 2048, 32 rows, 189 MB 38.7 -> 32.7 us (5.8 TB/s), 62 of 64 679 MB 123.8 ->
// 104.6 (6.5 TB/s).
constexpr int WALK_ROWS = 512;

template <int NW, int KB, int EPI>
__global__ __launch_bounds__(64 * NW) void expert_walk_kernel(ExpertArgs a) {
  constexpr int OUT = EPI == EPI_GLU ? 8 : 16;
  static_assert(64 * NW >= WALK_ROWS, "a thread keeps one row's place");
  __shared__ f32x4 red[2][NW][64];
  __shared__ int rows[WALK_ROWS];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), j = lane & 15, hq = lane >> 4;
  const int K = 64 * NW * KB, N = a.N, tiles = (N + OUT - 1) / OUT, step = gridDim.x;
  const int begin = lane < a.E ? a.offsets[lane] : 0;
  const int count = lane < a.E ? max(0, min(a.offsets[lane + 1], a.R) - begin) : 0;
  int place = 0;
  if (threadIdx.x < a.R) place = a.src ? a.src[threadIdx.x] : threadIdx.x;
  const int units = (count + 15) / 16 * tiles;
  int end = units;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int v = __shfl_up(end, o, 64);
    if (lane >= o) end += v;
  }
  const int first = end - units, total = __builtin_amdgcn_readlane(end, 63);
  if ((int)blockIdx.x >= total) return;

  struct Unit {
    int e, r0, r1, n0;
    bool in;
  };
  // (past the last unit: one line for all lanes, so that a unit's wait never stands behind a branch)
  auto unit = [&](int t) {
    Unit u;
    u.in = t < total;
    if (!u.in) t = 0;
    u.e = __popcll(__ballot(end <= t));
    int rem = t - __builtin_amdgcn_readlane(first, u.e);
    u.r0 = __builtin_amdgcn_readlane(begin, u.e);
    u.r1 = u.r0 + __builtin_amdgcn_readlane(count, u.e);
    while (rem >= tiles) {
      rem -= tiles;
      u.r0 += 16;
    }
    u.n0 = rem * OUT;
    return u;
  };
  const unsigned kin = (unsigned)(4 * (j & 8) + 8 * hq) * 2;
  const char* Wb = reinterpret_cast<const char*>(a.W) + 128 * KB * wave;
  const char* xb = reinterpret_cast<const char*>(a.x) + 128 * KB * wave + 16 * hq;
  u32x4 w[2][KB][2];
  Pack8 xv[2][KB][2];
  auto load_w = [&](int b, const Unit& t) {
    const char* base = Wb + ((long long)t.e * (EPI == EPI_GLU ? 2 : 1) * N + t.n0) * K * 2;
#pragma unroll
    for (int l = 0; l < 2; ++l) {
      const int row = min((EPI == EPI_GLU ? 0 : 8 * l) + (j & 7), N - 1 - t.n0);
      const unsigned off = t.in ? (unsigned)(row * K) * 2 + kin : 0;
      const char* from = base + (EPI == EPI_GLU && l ? (long long)N * K * 2 : 0);
#pragma unroll
      for (int u = 0; u < KB; ++u) w[b][u][l] = ld_nt16(reinterpret_cast<const bf16*>(from + 128 * u + off));
    }
  };
  auto load_x = [&](int b, const Unit& t) {
    const char* from = xb + (long long)rows[min(t.r0 + j, t.r1 - 1)] * K * 2;
#pragma unroll
    for (int u = 0; u < KB; ++u)
#pragma unroll
      for (int k = 0; k < 2; ++k) xv[b][u][k].w = *reinterpret_cast<const u32x4*>(from + 128 * u + 64 * k);
  };
  auto multiply = [&](int b, const Unit& t, int turn) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < KB; ++u) {
      Pack8 f0, f1;
      f0.w = half_swap<0xc>(w[b][u][0], w[b][u][1]);
      f1.w = half_swap<0x3>(w[b][u][1], w[b][u][0]);
      acc = mfma16(f0.v, xv[b][u][0].v, acc);
      acc = mfma16(f1.v, xv[b][u][1].v, acc);      // lane: row j, outputs n0 + 4 hq + 0..3
    }
    red[b][wave][lane] = acc;
    __builtin_amdgcn_s_waitcnt(0xc07f);      // lgkmcnt(0): the next unit's loads stay in flight
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (wave != turn) return;
    f32x4 v = red[b][0][lane];
#pragma unroll
    for (int i = 1; i < NW; ++i) v += red[b][i][lane];
    if constexpr (EPI == EPI_GLU) {
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = silu(v[r]) * __shfl_down(v[r], 32, 64);
      if (hq >= 2) return;
    }
    if constexpr (EPI == EPI_RELU2)
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = relu2f(v[r]);
    const int n = t.n0 + 4 * hq;
    if (t.r0 + j < t.r1) store_quad<EPI == EPI_F32>(a.y, (long long)(t.r0 + j) * N + n, v, n, N, N % 4 == 0);
  };

  Unit cur = unit(blockIdx.x);
  load_w(0, cur);
  if (threadIdx.x < a.R) rows[threadIdx.x] = place;
  __builtin_amdgcn_s_waitcnt(0xc07f);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  load_x(0, cur);
  int t = blockIdx.x, turn = 0;
  while (true) {
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      if (!cur.in) return;
      t += step;
      const Unit next = unit(t);
      load_w(b ^ 1, next);
      load_x(b ^ 1, next);
      __builtin_amdgcn_sched_barrier(0);
      multiply(b, cur, turn);
      cur = next;
      turn = turn + 1 == NW ? 0 : turn + 1;
    }
  }
}

SYM_DEV int chunk_swz(int row) { return (row >> 1) & 7; }

// Tiles of up to 128 rows of an expert x 128 weight rows.  At a few dozen rows an expert it is a weight stream: workgroups start at
// different stages of K (first_chunk; in step -> so, us: 16 experts, gated 1536 x 2048, 192 rows 50.9 -> 45.9, 800 51.7 -> 46.8; 8 of
// 4096 x 4096 200 rows 132 -> 106; the persistent tiles, which share rows in their L2, do not gain).  Long rows that are no power
// of two apart, or so many that rounds of workgroups are out of step by themselves, do not gain either: 2048 x 3072 of 8 experts,
// gated 54.7 -> 56.7, 768 x 5120 73.2 -> 75.1, 16 of 4096 x 4096 198 -> 206.  The place is the weight columns', not the workgroup's:
// a row's sums are the same in every row tile and whatever other rows an expert or its neighbours have.  (About a hundred rows of
// an expert are no stream any more: 32 experts, gated 1024 x 4096, 3600 rows 171 -> 181.)
template <int BM, int BN, int WR, int WC, int EPI>
__global__ __launch_bounds__(64 * WR * WC) void expert_tile_kernel(ExpertArgs a) {
  constexpr int NWV = WR * WC, WN = BN / WC, MS = BM / WR / 16, NS = WN / 16;   // 16-row subtiles of a wave
  constexpr int AB = BM * 128, BB = BN * 128, STAGE = AB + BB;         // bytes of a stage
  constexpr int AL = BM / 8 / NWV, BL = BN / 8 / NWV;                  // direct loads (8 rows each) per wave and stage
  constexpr int OUT = EPI == EPI_GLU ? BN / 2 : BN, WO = OUT / WC, NO = WO / 16;   // outputs of a tile, of a wave; in 16s
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int K = a.K, N = a.N, nb = (N + OUT - 1) / OUT;
  int e = -1, r0 = 0, rows = 0, bx = 0;
  {
    int total = 0;
    for (int i = 0; i < a.E; ++i) total += (max(0, min(a.offsets[i + 1], a.R) - a.offsets[i]) + BM - 1) / BM;
    total *= nb;
    const int per = (total + 7) / 8, local = blockIdx.x >> 3;
    int slot = (blockIdx.x & 7) * per + local;
    if (local >= per || slot >= total) return;
    for (int i = 0; i < a.E; ++i) {
      const int s0 = a.offsets[i], s1 = min(a.offsets[i + 1], a.R), t = (max(0, s1 - s0) + BM - 1) / BM;
      if (slot < t * nb) {
        const int g = slot / (GN * t), in = slot - g * GN * t, w = min(GN, nb - GN * g), m = in / w;
        e = i;
        bx = GN * g + in - m * w;
        r0 = s0 + m * BM;
        rows = min(BM, s1 - r0);
        break;
      }
      slot -= t * nb;
    }
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, wr = wave / WC, wc = wave % WC;
  const int n0 = OUT * bx;
  const bf16* asrc[AL];
  const bf16* bsrc[BL];
#pragma unroll
  for (int i = 0; i < AL; ++i) {
    const int row = 8 * (NWV * i + wave) + (lane >> 3), ch = (lane & 7) ^ chunk_swz(row);
    const int p = r0 + min(row, rows - 1);          // rows past the segment re-read its last one (never stored)
    asrc[i] = reinterpret_cast<const bf16*>(a.x) + (long long)(a.src ? a.src[p] : p) * K + 8 * ch;
  }
#pragma unroll
  for (int i = 0; i < BL; ++i) {
    const int row = 8 * (NWV * i + wave) + (lane >> 3), ch = (lane & 7) ^ chunk_swz(row);
    const int n = EPI == EPI_GLU ? min(n0 + WO * (row / WN) + row % WO, N - 1) + (row % WN >= WO ? N : 0) : min(n0 + row, N - 1);
    bsrc[i] = reinterpret_cast<const bf16*>(a.W) + ((long long)e * (EPI == EPI_GLU ? 2 : 1) * N + n) * K + 8 * ch;
  }
  const unsigned int lds0 = lds_address(smem) + __builtin_amdgcn_readfirstlane(wave) * 1024;
  const int nk = K / 64;
  const int turn = K <= 2048 || ((K & (K - 1)) == 0 && a.E * nb < 1024) ? first_chunk(bx, nk, 0) : 0;
  auto stage = [&](int kt, int buf) {
    kt = kt + turn < nk ? kt + turn : kt + turn - nk;
    const unsigned int base = lds0 + buf * STAGE;
#pragma unroll
    for (int i = 0; i < AL; ++i) direct_load16(asrc[i] + kt * 64, base + NWV * i * 1024);
#pragma unroll
    for (int i = 0; i < BL; ++i) direct_load16(bsrc[i] + kt * 64, base + AB + NWV * i * 1024);
  };
  f32x4 acc[NS][MS];
#pragma unroll
  for (int i = 0; i < NS; ++i)
#pragma unroll
    for (int q = 0; q < MS; ++q) acc[i][q] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int j = lane & 15, hq = lane >> 4;
  stage(0, 0);
  for (int kt = 0; kt < nk; ++kt) {
    wait_direct_loads();
    __syncthreads();      // stage kt has landed for every wave, and every wave is done reading the other stage
    if (kt + 1 < nk) stage(kt + 1, (kt + 1) & 1);
    const char* A = smem + (kt & 1) * STAGE;
    const char* B = A + AB;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const int c = 4 * ks + hq;
      Pack8 bf[NS], af[MS];
#pragma unroll
      for (int i = 0; i < NS; ++i) {
        const int row = WN * wc + 16 * i + j;
        bf[i].u = *reinterpret_cast<const uint4*>(B + row * 128 + 16 * (c ^ chunk_swz(row)));
      }
#pragma unroll
      for (int q = 0; q < MS; ++q) {
        const int row = (BM / WR) * wr + 16 * q + j;
        af[q].u = *reinterpret_cast<const uint4*>(A + row * 128 + 16 * (c ^ chunk_swz(row)));
      }
#pragma unroll
      for (int i = 0; i < NS; ++i)
#pragma unroll
        for (int q = 0; q < MS; ++q) acc[i][q] = mfma16(bf[i].v, af[q].v, acc[i][q]);
    }
  }
  // lane (j, hq): output row 16 q + j of the wave's rows, columns 16 i + 4 hq + 0..3 of its columns
  const bool vec = (N & 3) == 0;
#pragma unroll
  for (int q = 0; q < MS; ++q) {
    const int m = (BM / WR) * wr + 16 * q + j;
    if (m >= rows) continue;
#pragma unroll
    for (int i = 0; i < NO; ++i) {
      const int n = n0 + WO * wc + 16 * i + 4 * hq;
      const long long at = (long long)(r0 + m) * N + n;
      f32x4 f = acc[i][q];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if constexpr (EPI == EPI_GLU) f[u] = silu(f[u]) * acc[i + NO][q][u];
        if constexpr (EPI == EPI_RELU2) f[u] = relu2f(f[u]);
      }
      store_quad<EPI == EPI_F32>(a.y, at, f, n, N, vec);
    }
  }
}

template <int BM, int BN, int WR, int WC, int EPI>
void launch_tile(const ExpertArgs& a, hipStream_t s) {
  constexpr int lds = 2 * (BM + BN) * 128, OUT = EPI == EPI_GLU ? BN / 2 : BN;
  const long long tiles = (long long)((a.N + OUT - 1) / OUT) * ((a.R + BM - 1) / BM + a.E);
  expert_tile_kernel<BM, BN, WR, WC, EPI><<<(unsigned)((tiles + 7) / 8 * 8), 64 * WR * WC, lds, s>>>(a);
}

template <int BM, int BN, int WR, int WC>
void launch_tiles(const ExpertArgs& a, hipStream_t s) {
  if (a.glu) launch_tile<BM, BN, WR, WC, EPI_GLU>(a, s);
  else if (a.relu2) launch_tile<BM, BN, WR, WC, EPI_RELU2>(a, s);
  else if (a.f32_out) launch_tile<BM, BN, WR, WC, EPI_F32>(a, s);
  else launch_tile<BM, BN, WR, WC, EPI_BF16>(a, s);
}

// Prompt steps with many rows an expert: one persistent workgroup a CU, 8 waves in 2 x 4, tiles of 256 rows x 256 weight rows (a
// wave: 128 x 64) and of 128 x 256 for what a segment leaves over.  K in stages of 64.  A wave reads its fragments half a stage
// ahead of their products, so a stage's LDS is free from its middle on, where its one barrier stands: the rows of the stage after
// next (two buffers) load behind it, the weight rows of that stage (three buffers) in front of it, all between products.  The
// stages run on over the tile boundaries: a tile's first two load while the last products and the epilogue of the one before run.
// Every XCD walks its run of the tiles whole ones first; the whole ones that would be left for a last partial round are cut in two.
// The gated epilogue's division is a product with v_rcp_f32's reciprocal: the matrix cores wait for it, and its error (1 ulp of fp32) is none
// of the result's (2048 x 2048 at 2048 rows, against 64 bits 0.001659324 of the norm either way, and at 4 to 64 experts of 768 to 14336
// outputs, gates of 0.1 to 8, the same to nine places too; 8192 x 2048 dense, 8100 rows 432 -> 417 us, 4096 x 1024, 4000 rows 64.8 ->
// 61.3).  Loads, reads and products stand in turns: all of an operand's loads at once 420 -> 447.
// LDS rows as in expert_tile_kernel.  K % 64 == 0, K >= PERSIST_K, x and an expert's weights below 2 GiB.
constexpr int PERSIST_K = 512, PERSIST_OP = 32 * 1024, PERSIST_LDS = 5 * PERSIST_OP;

struct ExpertTile {
  int e, r0, rows, n0, half;      // half: 128 rows at most
};

SYM_DEV int lanes_upto(int v, int lane) {      // inclusive sum over the lanes
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int w = __shfl_up(v, o, 64);
    if (lane >= o) v += w;
  }
  return v;
}

template <int EPI>
__global__ __launch_bounds__(512, 1) void expert_persist_kernel(ExpertArgs a) {
  constexpr int OUT = EPI == EPI_GLU ? 128 : 256, WO = OUT / 4, NO = WO / 16;      // outputs of a tile, of a wave; in 16s
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int K = a.K, N = a.N, nb = (N + OUT - 1) / OUT, nk = K / 64;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wr = wave >> 2, wc = wave & 3;

  // ---- this workgroup's tiles.  Whole and half row tiles of an expert; lane l: those of all experts up to its share of them
  auto segment = [&](int e, int& r0, int& r1, int& w, int& h) {
    r0 = a.offsets ? a.offsets[e] : 0, r1 = a.offsets ? max(r0, min(a.offsets[e + 1], a.R)) : a.R;      // (no offsets: all rows one's)
    const int left = (r1 - r0) & 255;
    w = (r1 - r0) / 256 + (left > 128), h = left > 0 && left <= 128;
  };
  const int share = (a.E + 63) / 64;
  int whole = 0, halves = 0;
  for (int e = lane * share; e < min((lane + 1) * share, a.E); ++e) {
    int r0, r1, w, h;
    segment(e, r0, r1, w, h);
    whole += w, halves += h;
  }
  whole = lanes_upto(whole, lane), halves = lanes_upto(halves, lane);
  const int wgs = gridDim.x >> 3, xcd = blockIdx.x & 7;      // (the grid is a multiple of 8)
  const int wtotal = __builtin_amdgcn_readlane(whole, 63) * nb, htotal = __builtin_amdgcn_readlane(halves, 63) * nb;
  const int wper = (wtotal + 7) / 8, hper = (htotal + 7) / 8;
  const int w0 = xcd * wper, wn = max(0, min(wper, wtotal - w0)), h0 = xcd * hper, hn = max(0, min(hper, htotal - h0));
  const int over = wn % wgs;      // (a half tile takes 5 / 9 of a whole one's time)
  const bool cut = over && 5 * ((2 * over + hn + wgs - 1) / wgs) < 9 + 5 * ((over + hn - 1) / wgs);
  const int wkeep = cut ? wn - over : wn, wcut = cut ? 2 * over : 0, count = wkeep + wcut + hn;
  auto find = [&](int s) {
    ExpertTile r;
    r.half = s >= wkeep;
    const bool rest = s >= wkeep + wcut;
    const int g = rest ? h0 + s - wkeep - wcut : w0 + (r.half ? wkeep + ((s - wkeep) >> 1) : s);
    const int upto = rest ? halves : whole, l = __builtin_popcountll(__ballot(upto * nb <= g));      // (some lane's sum lies above)
    int e = l * share, lo = l ? __builtin_amdgcn_readlane(upto, l - 1) : 0, s0, s1, w, h;
    segment(e, s0, s1, w, h);
    while ((lo + (rest ? h : w)) * nb <= g) {
      lo += rest ? h : w;
      segment(++e, s0, s1, w, h);
    }
    int m = w, n = g - lo * nb;
    if (!rest) {
      const int gr = n / (GN * w), in = n - gr * GN * w, cols = min(GN, nb - GN * gr);
      m = in / cols;
      n = GN * gr + in - m * cols;
    }
    r.e = e;
    r.r0 = s0 + 256 * m + (!rest && r.half ? 128 * ((s - wkeep) & 1) : 0);
    r.rows = min(r.half ? 128 : 256, s1 - r.r0);
    r.n0 = OUT * n;
    return r;
  };
  int slot = blockIdx.x >> 3;
  if (slot >= count) return;

  // ---- direct loads: instruction i of 4 covers rows 64 i + 8 wave + lane / 8 of an operand.  EPI_GLU: 32 gate rows and 32 up
  // rows of the same outputs in every 64, so that a pair meets in a wave.
  const int lrow = 8 * wave + (lane >> 3), lch = (lane & 7) ^ chunk_swz(lrow);
  int aoff[4], boff = 0, blast = 0;      // (weight rows past the expert's last re-read it)
  u32x4 xbuf = buffer_words(a.x, (long long)a.xrows * K * 2), wbuf;
  int ahalf = 0, kx = 0;      // of the tile being loaded; bytes of a row behind the stage to load
  auto bind = [&](const ExpertTile& t) {
    ahalf = t.half;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int p = t.r0 + min(64 * i + lrow, t.rows - 1);          // rows past the segment re-read its last one (never stored)
      aoff[i] = (a.src ? a.src[p] : p) * K * 2 + 16 * lch;
    }
    const int up = EPI == EPI_GLU ? (lrow >> 5) * N : 0;
    int row = t.n0 + (EPI == EPI_GLU ? lrow & 31 : lrow) + up, last = N - 1 + up;
    if (EPI == EPI_GLU && a.eights) row = 2 * t.n0 + 2 * (lrow & 24) + (lrow & 7) + 8 * (lrow >> 5), last = 2 * N - 1;
    boff = row * K * 2 + 16 * lch;
    blast = last * K * 2 + 16 * lch;
    const long long wrows = (EPI == EPI_GLU ? 2LL : 1LL) * N;
    wbuf = buffer_words(reinterpret_cast<const bf16*>(a.W) + t.e * wrows * K, wrows * K * 2);
  };
  const unsigned int lds0 = lds_address(smem) + wave * 1024;
  const int wstep = OUT / 4 * (EPI == EPI_GLU && a.eights ? 2 : 1) * K * 2;
  unsigned int afill = 0, bfill = 0;      // the buffers to fill
  auto load_a = [&](int i) {
    if (i < 2 || !ahalf) direct_buffer_load16(xbuf, aoff[i], kx, lds0 + afill + 8192 * i);
  };
  auto load_b = [&](int i) {
    direct_buffer_load16(wbuf, min(boff + i * wstep, blast), kx, lds0 + 2 * PERSIST_OP + bfill + 8192 * i);
  };
  ExpertTile cur = find(slot), next = cur;
  bool more = slot + wgs < count;
  if (more) next = find(slot + wgs);
  auto turn_b = [&](unsigned int b) { return b == 2 * PERSIST_OP ? 0u : b + PERSIST_OP; };
  auto loaded = [&]() {      // a stage's loads are out
    afill ^= PERSIST_OP;
    bfill = turn_b(bfill);
    kx += 128;
    if (kx == 2 * K) {
      kx = 0;
      if (more) bind(next);      // (behind the last tile: its own start again, into buffers that are not read any more)
    }
  };

  f32x4 acc[4][8];
  Pack8 f0[12], f1[12];      // the fragments of a stage's halves: 4 of weight rows, 8 of rows
  const int j = lane & 15, hq = lane >> 4;
  const int c0 = j * 128 + 16 * (hq ^ chunk_swz(j));      // of the first half; the second half's chunks are 64 bytes across
  unsigned int ard = 0, brd = 0;      // the buffers of the stage at hand
  auto fragment = [&](Pack8 (&f)[12], int c, unsigned int arow, int i) {
    if (i < 4) f[i].u = *reinterpret_cast<const uint4*>(smem + 2 * PERSIST_OP + brd + 8192 * wc + c + 2048 * i);
    else f[i].u = *reinterpret_cast<const uint4*>(smem + ard + arow + c + 2048 * (i - 4));
  };
  // one stage of a tile of 32 NQ rows; arow: where the wave's rows stand in a buffer, anext: in the next stage's
  auto stage = [&](auto start, auto nq, unsigned int arow, unsigned int anext, bool stores) __attribute__((always_inline)) {
    constexpr int NQ = decltype(nq)::value;
    int c1 = c0;
    asm volatile("v_xor_b32 %0, 64, %0" : "+v"(c1));      // (kept in a register it would cost another one's spill)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      load_b(i);
#pragma unroll
      for (int u = 0; u < 3; ++u)
        if (3 * i + u < 4 + NQ) fragment(f1, c1, arow, 3 * i + u);
#pragma unroll
      for (int q = 0; q < NQ; ++q) acc[i][q] = mfma16(f0[i].v, f0[4 + q].v, decltype(start)::value ? f32x4{0.f, 0.f, 0.f, 0.f} : acc[i][q]);
      __builtin_amdgcn_sched_barrier(0);
    }
    // every wave: the next stage has landed, this one's fragments are in registers
    if (stores) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(4 + 8 * NO) : "memory");
    else asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xc07f);      // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    ard ^= PERSIST_OP;
    brd = turn_b(brd);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      load_a(i);
#pragma unroll
      for (int u = 0; u < 3; ++u) fragment(f0, c0, anext, 3 * i + u);
#pragma unroll
      for (int q = 0; q < NQ; ++q) acc[i][q] = mfma16(f1[i].v, f1[4 + q].v, acc[i][q]);
      __builtin_amdgcn_sched_barrier(0);
    }
    loaded();
  };
  auto rows_at = [&](const ExpertTile& t) { return (unsigned int)(t.half ? 8192 : 16384) * wr; };
  const bool vec = (N & 3) == 0;
  bool stores = false;      // a whole tile's stores stand behind the loads that are waited for
  auto tile = [&](auto nq) __attribute__((always_inline)) {
    constexpr int NQ = decltype(nq)::value;
    const unsigned int arow = rows_at(cur), anext = rows_at(next);
    stage(std::true_type{}, nq, arow, arow, stores);
    for (int k = 1; k < nk; ++k) stage(std::false_type{}, nq, arow, k + 1 < nk ? arow : anext, false);
    // lane (j, hq): output row 16 q + j of the wave's rows, columns 16 i + 4 hq + 0..3 of its columns
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const int m = 16 * NQ * wr + 16 * q + j;
      if (m < cur.rows) {
#pragma unroll
        for (int i = 0; i < NO; ++i) {
          const int n = cur.n0 + WO * wc + 16 * i + 4 * hq;
          f32x4 v = acc[i][q];
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            if constexpr (EPI == EPI_GLU) v[u] = v[u] * __builtin_amdgcn_rcpf(1.f + __expf(-v[u])) * acc[i + NO][q][u];
            if constexpr (EPI == EPI_RELU2) v[u] = relu2f(v[u]);
          }
          // (fp32 rows go past the caches: a round of tiles writes twice what the L2 holds, and the operands stay there; 32400 rows,
          // 16 experts of 2048 x 1536: 233 -> 212 us.  The 16-bit rows of a gated product are read next: 350 -> 369 that way)
          store_quad<EPI == EPI_F32, EPI == EPI_F32>(a.y, (long long)(cur.r0 + m) * N + n, v, n, N, vec);
        }
      }
    }
    stores = NQ == 8 && vec && cur.rows == 256 && cur.n0 + OUT <= N;
  };

  bind(cur);
  wait_direct_loads();
#pragma unroll
  for (int s = 0; s < 2; ++s) {
#pragma unroll
    for (int i = 0; i < 4; ++i) load_b(i);
#pragma unroll
    for (int i = 0; i < 4; ++i) load_a(i);
    loaded();
  }
  if (ahalf) asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
  else asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
#pragma unroll
  for (int i = 0; i < 12; ++i) fragment(f0, c0, rows_at(cur), i);
  while (true) {
    if (cur.half) tile(std::integral_constant<int, 4>{});
    else tile(std::integral_constant<int, 8>{});
    if (!more) break;
    cur = next;
    slot += wgs;
    more = slot + wgs < count;
    if (more) next = find(slot + wgs);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // no load may land in LDS that is not this workgroup's any more
}

int cu_count() {
  int dev = 0, cus = 256;
  (void)hipGetDevice(&dev);
  (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  return cus;
}

template <int EPI>
void launch_persist(const ExpertArgs& a, int cus, hipStream_t s) {
  static const hipError_t once = hipFuncSetAttribute(reinterpret_cast<const void*>(&expert_persist_kernel<EPI>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, PERSIST_LDS);
  (void)once;
  constexpr int OUT = EPI == EPI_GLU ? 128 : 256;
  const long long tiles = (long long)((a.N + OUT - 1) / OUT) * ((a.R + 127) / 128 + a.E);
  const long long grid = std::min<long long>((tiles + 7) / 8 * 8, std::max(8, cus / 8 * 8));
  expert_persist_kernel<EPI><<<(unsigned)grid, 512, PERSIST_LDS, s>>>(a);
}

template <int NW, int NE>
void launch_route(const RouteArgs& a, hipStream_t s) {
  const int tiles = (a.T + 15) / 16;
  const size_t lds = (size_t)NW * NE * 256 * sizeof(float);
  if (a.resid) {
    const int room = (int)lds + 16 * (a.d + 8) * 2;      // (at most 32 + 64 KB)
    static const hipError_t once = hipFuncSetAttribute(reinterpret_cast<const void*>(&route_mfma_kernel<NW, NE, true, true>),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, 98304 + 1024);
    (void)once;
    route_mfma_kernel<NW, NE, true, true><<<1, 64 * NW, room, s>>>(a);
    return;
  }
  if (tiles == 1) route_mfma_kernel<NW, NE, true><<<1, 64 * NW, lds, s>>>(a);
  else route_mfma_kernel<NW, NE, false><<<tiles, 64 * NW, lds, s>>>(a);
}

template <int NE>
void launch_route_ne(const RouteArgs& a, hipStream_t s) {
  if (a.T <= 512 && NE <= 4) launch_route<16 / (NE > 2 ? 2 : 1), NE>(a, s);   // decode-sized: the width over more waves
  else launch_route<4, NE>(a, s);
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

bool route_mfma(const RouteArgs& a, int f32) {
  return !f32 && a.d % 32 == 0 && a.E <= 64 && a.k <= 64 && aligned16(a.x) && aligned16(a.Wr);
}

}  // namespace

bool route_norm_fits(const RouteArgs& a) {
  return route_mfma(a, 0) && a.T <= 16 && a.d % 512 == 0 && a.d <= 2048 && aligned16(a.resid) && aligned16(a.norm);
}

bool route_topk_runs(const RouteArgs& a, int f32) { return route_mfma(a, f32) && a.E <= 16 && a.d % 128 == 0; }

void launch_route_topk(const RouteArgs& a, int f32, hipStream_t s) {
  if (a.T <= 0) return;
  if (route_mfma(a, f32)) {
    if (a.runs) {
      if (a.d % 512 == 0) launch_route<16, 1>(a, s);
      else launch_route<4, 1>(a, s);
    } else if (a.E <= 16) launch_route_ne<1>(a, s);
    else if (a.E <= 32) launch_route_ne<2>(a, s);
    else launch_route_ne<4>(a, s);
    if (a.T <= 16) return;      // the single workgroup laid out the segments
  } else {
    const size_t lds = (size_t)a.E * sizeof(float);
    if (f32) route_rows_kernel<float><<<a.T, NT, lds, s>>>(a);
    else route_rows_kernel<bf16><<<a.T, NT, lds, s>>>(a);
  }
  const int R = a.T * a.k;
  expert_layout_kernel<<<(R + 4 * PLAN_NT - 1) / (4 * PLAN_NT), PLAN_NT, 3 * a.E * sizeof(int), s>>>(a.ids, R, a.E, a.k,
                                                                                                   a.offsets, a.dst, a.src);
}

template <int NW, int KB>
bool launch_walk(const ExpertArgs& a, int cus, hipStream_t s) {
  if (a.K != 64 * NW * KB) return false;
  const int tiles = a.glu ? (a.N + 7) / 8 : (a.N + 15) / 16;
  const long long most = (long long)tiles * std::min(a.R, a.E + a.R / 16);      // (units, at most)
  // (two small workgroups share a CU: 2048 x 512 of 64 experts, 32 rows, 19.7 -> 11.5 us; at 1536 wide one of 12 waves, 17.8 us
  // where one of 8 takes 18.3 and two 19.5)
  const int grid = (int)std::min<long long>(most, (NW == 8 ? 2 : 1) * cus);
  if (a.glu) expert_walk_kernel<NW, KB, EPI_GLU><<<grid, 64 * NW, 0, s>>>(a);
  else if (a.relu2) expert_walk_kernel<NW, KB, EPI_RELU2><<<grid, 64 * NW, 0, s>>>(a);
  else if (a.f32_out) expert_walk_kernel<NW, KB, EPI_F32><<<grid, 64 * NW, 0, s>>>(a);
  else expert_walk_kernel<NW, KB, EPI_BF16><<<grid, 64 * NW, 0, s>>>(a);
  return true;
}

bool expert_linear_mfma(const ExpertArgs& a, int f32) {
  return !f32 && a.K % 32 == 0 && aligned16(a.x) && aligned16(a.W) && aligned16(a.y);
}

// what the persistent tiles address: x and an expert's weights through a buffer's range, a lane's offset in it
static bool persist_fits(const ExpertArgs& a) {
  const long long top = 0x7fffffffLL;
  return a.K % 64 == 0 && a.K >= PERSIST_K && a.xrows * 2LL * a.K <= top && ((a.glu ? 2LL : 1LL) * a.N + 512) * 2 * a.K <= top;
}

const std::array<int, 4>& expert_walk_widths() {      // (64 NW KB of launch_expert_linear's forms)
  static const std::array<int, 4> widths = {512, 1536, 2048, 3072};
  return widths;
}

// The walk over many weights against a workgroup per 16 outputs, us: gated, 16 experts of 1536 x 2048, 4 / 16 / 32 / 128 rows 19.4 ->
// 12.5, 32.8 -> 26.1, 42.4 -> 39.3 (and 256 rows, where blocks of 16 read weights twice, 50.2 -> 62.9); 512 x 2048, 64 experts
// 32 rows 29.5 -> 24.7; 512 x 3072, 32 experts 38.3 -> 26.4; to fp32, 32 rows, 2048 x 1536 21.7 -> 17.7, 2048 x 2048 24.3 ->
// 20.2, 2048 x 512 of 64 experts 16.0 -> 11.5; narrow outputs do not fill it: 512 x 1536, 16 rows of 8 experts 5.0 -> 5.9, 1024 x
// 2048 11.7 -> 12.1, gated 1536 x 512 7.2 -> 8.0.
// Nor do few experts.  Of 1921 measured sizes that the lines above take (4 to 64 experts, 1 to 64 tokens), 98 are left to the
// weight stream, which the walk took 1.06 of; on the others it takes 0.84.  Its units come in rounds of a workgroup a CU: gated,
// between one and two rounds with rows enough to choose all experts (8 experts of 512 x 2048, 64 rows 10.5 -> 11.6; at 6 rows 4
// experts of 512 x 2048 0.90); 512 wide up to two rounds (4 experts, 2048 outputs, 10 rows 4.0 -> 4.7; 8 experts 8 rows 0.88);
// 2048 wide up to four (4 experts, 2048 outputs 9.0 -> 10.3, 8 experts 12 rows 11.9 -> 13.0; 16 experts 0.85).
// The widths: a wave holds a unit's weights and rows and the next unit's; at 4096 that alone is the 128 registers that a lane of
// sixteen waves has.  Other widths up to there are not instantiated.
static bool walks(const ExpertArgs& a, int cus) {
  const auto& widths = expert_walk_widths();
  if (a.E > 64 || a.R > WALK_ROWS || std::find(widths.begin(), widths.end(), a.K) == widths.end()) return false;
  const long long tiles = a.glu ? (a.N + 7) / 8 : (a.N + 15) / 16, units = a.E * tiles;
  if (a.glu) return a.K >= 1536 && !(units > cus && units <= 2 * cus && a.R >= 2 * a.E);
  if (a.N < 1536) return false;
  if (a.K == 512) return std::min(a.R, a.E) * tiles > 2 * cus;
  return a.K != 2048 || units > 4 * cus || 2 * a.R < 3 * a.E;
}

// Persistent tiles against those of 128, us: 16 experts, gated 1536 x 2048 and 2048 x 1536, at 96 rows each 43.9 -> 46.0 and 29.0 ->
// 30.5, 128 62.9 -> 52.2 and 35.2 -> 31.8, 512 124 -> 112 and 76 -> 77, 2025 446 -> 360 and 276 -> 212; 8 experts, gated 14336 x
// 4096 and 4096 x 14336, at 64 rows 374 -> 420 and 244 -> 256, 128 511 -> 452 and 311 -> 270, 2048 3740 -> 3018 and 2160 -> 1650
// (1.28 and 1.17 PFLOP/s); 64 experts, 2048 x 1024 at 128 rows 110 -> 83.  Where the gated tiles fill 0.7 to 1 round of the CUs,
// most of them get a second half tile: 16 experts of 256 rows (0.75 rounds) 73 -> 80, of 224 65 -> 56, of 288 90 -> 88.
// They have to be many: below 0.3 rounds the small ones, four times as many, are ahead (8 experts of 128 rows, 2048 x 1536 28.0 ->
// 34.1, of 375 rows, 512 x 2048 31.0 -> 49.7; from there 0.82 on average, 2054 sizes of 4 to 64 experts, and below it 1.09 on 529).
// Widths below 1024 pay a tile's start and end over few stages: 512, 2048 outputs, 16 experts of 1250 rows 1.06 to 1.11, 64 experts
// 0.70, gated 0.8 to 0.96 from one round on; 512 outputs of 2025 rows 40.5 -> 48.3.
static bool persists(const ExpertArgs& a, int per, int cus) {
  if (!persist_fits(a) || a.N < 256) return false;
  const long long cols = (a.N + 255) / 256 * (a.glu ? 2 : 1), full = cols * (a.R / 256);
  const long long tiles = (a.glu ? (a.N + 127) / 128 : cols) * a.E * std::max(1, (per + 255) / 256);
  if (a.K < 1024) return per >= 1024 && a.N >= 1024 && tiles >= (a.glu ? 1 : 2) * cus;
  return per >= 128 && 10 * tiles >= 3 * cus && (!a.glu || 10 * full <= 7 * cus || full >= cus);
}

// A dense gated projection of many rows is one expert's: rounds of tiles that the XCDs' workgroups take (a half one 5 / 9 of a whole
// one), as the kernel deals them out.  Its tiles run at 1.2 to 1.3 PFLOP/s and save the launch that multiplies; against the library's
// product and that launch it is ahead where its rounds are full to 0.6, from 4096 wide on, where the library's are better, to 0.8.
// us, library / tiles (rounds' fill): 8192 x 2048 at 400 rows 38.9 / 33.8 (0.70), 513 43.1 / 47.4 (0.50), 600 45.5 / 46.8 (0.59), 700 49.9 /
// 47.8 (0.68), 1000 64.9 / 56.2, 1530 99 / 84.5, 2600 189 / 153, 8100 462 / 444; 5632 x 2048 at 800 42.3 / 46.5 (0.54), 1000 58 / 47
// (0.67), 8100 404 / 305; 1536 x 6144 at 1800 69.1 / 69.7 (0.59), 3000 102 / 117 (0.55); 14336 x 4096 at 400 103 / 107 (0.68), 700 158 / 160
// (0.77), 1000 204 / 204 (0.85), 2600 586 / 506, 8100 1399 / 1412; 11008 x 4096 at 1530 314 / 236, 8100 1229 / 1104.
bool dense_glu_pays(long long M, long long N, long long K, int cus) {
  if (M <= 256 || N < 256 || K < 1024) return false;
  const long long cols = (N + 127) / 128, left = M % 256, wgs = std::max(1, cus / 8);
  const long long w = (cols * (M / 256 + (left > 128)) + 7) / 8, h = left > 0 && left <= 128 ? (cols + 7) / 8 : 0;      // an XCD's, whole and half
  const long long over = w % wgs, halves = (over + h + wgs - 1) / wgs, uncut = over ? 9 + 5 * (halves - 1) : 5 * halves;
  const long long ninths = 9 * (w / wgs) + (over ? std::min(uncut, 5 * ((2 * over + h + wgs - 1) / wgs)) : uncut);
  // fill: M cols / 256 whole tiles' work over 8 wgs workgroups, against the rounds
  return 9 * 10 * M * cols >= (K >= 4096 ? 8 : 6) * 256 * 8 * wgs * ninths;
}

// (weights whose rows come by eights, in prompt steps of four layers, us: 8192 x 2048, 420 rows 554 -> 510, 1500 1146 -> 1085, 8000 3694 ->
// 3542; 14336 x 4096, 1100 rows 2172 -> 2113, 2600 4512 -> 4186, 8100 10944 -> 10881)
bool launch_dense_glu(const ExpertArgs& a, hipStream_t s) {
  const int cus = cu_count();
  if (!expert_linear_mfma(a, 0) || !persist_fits(a) || !dense_glu_pays(a.R, a.N, a.K, cus)) return false;
  launch_persist<EPI_GLU>(a, cus, s);
  return true;
}

// The form that a call takes by its sizes: 0 all shapes, 1 weight stream, 2 / 3 tiles of 128 / 256, 4 the walk.
// Stream or tile, measured at 16 experts, 4 rows each on average: [gate | up] of 1536 x 2048 46.0 us on both, 2048 x 1536 23.9
// against 28.8; at 16 rows each 53 against 46.6 and 33 against 28.7.
int expert_linear_form(const ExpertArgs& a, bool mfma, int cus) {
  const int per = (a.R + a.E - 1) / a.E;      // rows per expert if they are spread evenly
  const bool stream = mfma && a.E <= 65535, tile = mfma && a.K % 64 == 0;
  if (stream && (per <= 8 || !tile)) return per <= 8 && walks(a, cus) ? 4 : 1;
  if (tile) return persists(a, per, cus) ? 3 : 2;
  return 0;
}

// Returns the form used; impl < 0: expert_linear_form's.  A form that does not take the sizes gives way: 4 to 1, 3 to 2.
int launch_expert_linear(const ExpertArgs& a, int f32, int impl, hipStream_t s) {
  if (a.R <= 0) return 0;
  const bool mfma = expert_linear_mfma(a, f32), stream = mfma && a.E <= 65535, tile = mfma && a.K % 64 == 0;
  const int per = (a.R + a.E - 1) / a.E, cus = cu_count();
  if (impl < 0) impl = expert_linear_form(a, mfma, cus);
  if (impl == 4) {
    if (mfma && a.E <= 64 && a.R <= WALK_ROWS &&
        (launch_walk<8, 1>(a, cus, s) || launch_walk<12, 2>(a, cus, s) || launch_walk<16, 2>(a, cus, s) || launch_walk<16, 3>(a, cus, s)))
      return 4;
    impl = 1;
  }
  if (impl == 1 && stream) {
    const int deep = a.K / 512;               // 64-element steps of each of 8 waves
    if (per <= 8 && a.glu) {
      // (both rows of a pair take twice the registers: 4 waves, 2 steps: 37.7 us, 8 waves: 38.5 with 2 steps and 43 with 4, at
      // 32 rows, 16 x 2 x 1536 x 2048 with 14 experts chosen)
      expert_stream_kernel<1, 4, 2, EPI_GLU><<<dim3((a.N + 15) / 16, a.E), 256, 0, s>>>(a);
    } else if (per <= 8) {
      // widths of 1536 to 2016: every wave has 3 steps or 4, and with 4 in flight those of 3 would load them one by one (16
      // experts, 32 rows, 2048 outputs, us, 4 -> 3 in flight: 1536 28.6 -> 23.6, 1568 29.5 -> 24.9, 1792 30.4 -> 28.2, 2016
      // 35.8 -> 32.5)
      if (deep == 3) launch_stream<1, 8, 3>(a, s);
      else launch_stream<1, 8, 4>(a, s);
    } else if (per <= 24) {
      launch_stream<2, 4, 2>(a, s);
    } else {
      launch_stream<4, 4, 2>(a, s);
    }
    return 1;
  }
  if (impl == 3 && !(tile && persist_fits(a))) impl = 2;
  if (impl == 2 && tile) {
    launch_tiles<128, 128, 2, 2>(a, s);
    return 2;
  }
  if (impl == 3 && tile) {
    if (a.glu) launch_persist<EPI_GLU>(a, cus, s);
    else if (a.relu2) launch_persist<EPI_RELU2>(a, cus, s);
    else if (a.f32_out) launch_persist<EPI_F32>(a, cus, s);
    else launch_persist<EPI_BF16>(a, cus, s);
    return 3;
  }
  if (a.glu || a.f32_out) return -1;      // (the binding has refused it)
  launch_grouped_linear(a.x, a.W, a.offsets, a.E, a.R, a.N, a.K, a.y, f32, s, a.src, a.relu2);
  return 0;
}
