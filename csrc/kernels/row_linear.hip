// Linear layers of a few rows (decode steps, the logits of a prompt step's last rows): y = f(x) . W^T with x [M][K] of
// M <= 16 rows, W [N][K] bf16 row-major, fp32 accumulation on v_mfma_f32_16x16x32_bf16.
//
// The weights are read once, so the kernel is a weight stream: a workgroup owns a tile of 16 or 8 weight rows (two tiles
// for a gated pair), its waves split K, every wave has a chunk of weight loads in flight while it multiplies the chunk
// before, and the partial sums meet in LDS.  W is the A operand (its rows the tile's rows), x the B operand (its rows the
// columns); x is read straight from the L2, which all workgroups share.  (Past 16 rows that traffic passes the weights':
// 32 rows of 2048 x 8192 take 22 us against the library's 19, so those stay there.)
//
// What a neighbouring launch did is done here: the squared ReLU of the input (XF), and silu(gate) * up of a projection
// whose rows are [gate | up] (EPI_GLU: a workgroup computes both rows of its outputs).
#include "common.h"
#include "hybrid_launchers.h"

namespace {

enum { EPI_BF16 = 0, EPI_F32 = 1, EPI_GLU = 2 };

struct Args {
  const bf16* x;
  long long ldx;
  const bf16* W;
  void* out;
  long long ldo;
  int M, N, K;  // EPI_GLU: N outputs, W has 2 N rows
};

SYM_DEV void relu_squared(Pack8& x) {
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float v = fmaxf((float)x.h[j], 0.f);
    x.h[j] = (bf16)(v * v);
  }
}

// Lane (m = lane & 15, h) holds outputs 4 h .. 4 h + 3 of row m of the tile at n0; N is a multiple of 4.
template <int RH, int EPI>
SYM_DEV void store_rows(const Args& a, int n0, int lane, f32x4 v, f32x4 u) {
  const int m = lane & 15, n = n0 + 4 * (lane >> 4);
  if constexpr (EPI == EPI_GLU) {
    // the two projections are rounded to bf16 first, as separate launches leave them
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = silu((float)(bf16)v[r]) * (float)(bf16)u[r];
  }
  if (m >= a.M || 4 * (lane >> 4) >= RH || n >= a.N) return;
  if constexpr (EPI == EPI_F32) {
    *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(a.out) + m * a.ldo + n) = v;
  } else {
    bf16x4 b;
#pragma unroll
    for (int r = 0; r < 4; ++r) b[r] = (bf16)v[r];
    *reinterpret_cast<bf16x4*>(reinterpret_cast<bf16*>(a.out) + m * a.ldo + n) = b;
  }
}

// A lane's registers from the lane 8 further in its row of 16, in the banks of MASK only (0x3: lanes 0-7, 0xc: 8-15).
template <int MASK>
SYM_DEV u32x4 half_swap(u32x4 keep, u32x4 from) {
  u32x4 r;
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = __builtin_amdgcn_update_dpp(keep[i], from[i], 0x128 /* row_ror:8 */, 0xf, MASK, false);
  return r;
}

// RT: weight tiles of a workgroup.  RH: weight rows of a tile, 16 or 8.  U: 64-deep k blocks of a chunk.  Every wave has
// the same number of whole chunks.
//
// One load instruction reads 128 contiguous bytes (a 64-deep k block) of each of 8 weight rows: lanes 0-7 of each row of 16
// lanes hold the block's first 32-deep step, lanes 8-15 its second.  Two such loads (rows 0-7, rows 8-15) become the two
// steps' A operands by exchanging halves, 4 v_mov_dpp each.  With RH = 8 there is one load, and rows 8-15 of the product
// are dropped.
template <int RT, int RH, int NW, int U, int EPI, bool XF>
__global__ __launch_bounds__(NW * 64) void row_linear_kernel(Args a) {
  constexpr int LD = RH / 8;  // loads of a block
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, h = lane >> 4;
  const int n0 = blockIdx.x * (EPI == EPI_GLU ? RH : RH * RT);

  // rows past the end repeat the last one; their products are not stored
  unsigned wo[RT][LD];
  const char* wb[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    const int first = EPI == EPI_GLU ? n0 : n0 + RH * rt;
    const int base = min(first, a.N - 1);
    wb[rt] = reinterpret_cast<const char*>(a.W + (long long)(base + (EPI == EPI_GLU ? rt * a.N : 0)) * a.K);
#pragma unroll
    for (int l = 0; l < LD; ++l)
      wo[rt][l] = (unsigned)((min(first + 8 * l + (r16 & 7), a.N - 1) - base) * a.K + 4 * (r16 & 8) + 8 * h) * 2;
  }
  const char* xb = reinterpret_cast<const char*>(a.x);
  const unsigned xo = (unsigned)(min(r16, a.M - 1) * a.ldx + 8 * h) * 2;

  f32x4 acc[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) acc[rt] = f32x4{0.f, 0.f, 0.f, 0.f};

  u32x4 w[2][U][RT][LD];
  Pack8 xv[U][2];
  auto load_w = [&](int b, int blk) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int l = 0; l < LD; ++l) w[b][u][rt][l] = ld_nt16(reinterpret_cast<const bf16*>(wb[rt] + 128 * (blk + u) + wo[rt][l]));
  };
  auto load_x = [&](int blk) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int t = 0; t < 2; ++t) xv[u][t].w = *reinterpret_cast<const u32x4*>(xb + 128 * (blk + u) + 64 * t + xo);
  };
  auto multiply = [&](int b) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if constexpr (XF) {
#pragma unroll
        for (int t = 0; t < 2; ++t) relu_squared(xv[u][t]);
      }
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        Pack8 f0, f1;
        const u32x4 lo = w[b][u][rt][0], hi = w[b][u][rt][LD - 1];
        f0.w = LD == 2 ? half_swap<0xc>(lo, hi) : lo;
        f1.w = half_swap<0x3>(hi, lo);
        acc[rt] = mfma16(f0.v, xv[u][0].v, acc[rt]);
        acc[rt] = mfma16(f1.v, xv[u][1].v, acc[rt]);
      }
    }
  };
  // The loads of a chunk stand ahead of the products of the one before (the scheduler, left alone, moves them behind to
  // save registers), and the last chunk's successor is itself, read again: behind a branch every wait would drain all
  // loads.
  const int per = (a.K >> 6) / NW, s0 = wid * per;
  load_w(0, s0);
  if (per <= U) {  // one chunk
    load_x(s0);
    __builtin_amdgcn_sched_barrier(0);
    multiply(0);
  } else {
    const int end = s0 + per, last = end - U;
    for (int s = s0; s < end; s += 2 * U) {
      load_x(s);
      load_w(1, min(s + U, last));
      __builtin_amdgcn_sched_barrier(0);
      multiply(0);
      if (s + U >= end) break;
      __builtin_amdgcn_sched_barrier(0);
      load_x(s + U);
      load_w(0, min(s + 2 * U, last));
      __builtin_amdgcn_sched_barrier(0);
      multiply(1);
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  __shared__ f32x4 red[NW][RT][64];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) red[wid][rt][lane] = acc[rt];
  __syncthreads();
  if (wid >= (EPI == EPI_GLU ? 1 : RT)) return;
  auto sum = [&](int rt) {
    f32x4 v = red[0][rt][lane];
#pragma unroll
    for (int i = 1; i < NW; ++i) v += red[i][rt][lane];
    return v;
  };
  store_rows<RH, EPI>(a, n0 + RH * wid, lane, sum(wid), EPI == EPI_GLU ? sum(RT - 1) : f32x4{});
}

// Any K up to SMALL_K (low-rank factors): one wave per 16-row tile, 32 deep a step; lanes past K multiply zeros.
constexpr int SMALL_K = 256;

template <int EPI, bool XF>
__global__ __launch_bounds__(64) void row_linear_small_kernel(Args a) {
  constexpr int RT = EPI == EPI_GLU ? 2 : 1;
  const int lane = threadIdx.x, r16 = lane & 15, h = lane >> 4, n0 = blockIdx.x * 16;
  const bf16* wr = a.W + (long long)min(n0 + r16, a.N - 1) * a.K + 8 * h;
  const bf16* xr = a.x + min(r16, a.M - 1) * a.ldx + 8 * h;
  f32x4 acc[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) acc[rt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int k = 0; k < a.K; k += 32) {
    const bool in = k + 8 * h < a.K;  // K is a multiple of 8
    Pack8 x, w;
    x.u = in ? *reinterpret_cast<const uint4*>(xr + k) : make_uint4(0, 0, 0, 0);
    if constexpr (XF) relu_squared(x);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      w.u = in ? *reinterpret_cast<const uint4*>(wr + (long long)rt * a.N * a.K + k) : make_uint4(0, 0, 0, 0);
      acc[rt] = mfma16(w.v, x.v, acc[rt]);
    }
  }
  store_rows<16, EPI>(a, n0, lane, acc[0], acc[RT - 1]);
}

template <int RT, int RH, int NW, int U, int EPI, bool XF>
bool run(const Args& a, hipStream_t s) {
  if (a.K % (64 * NW * U)) return false;
  constexpr int rows = EPI == EPI_GLU ? RH : RH * RT;
  row_linear_kernel<RT, RH, NW, U, EPI, XF><<<(a.N + rows - 1) / rows, NW * 64, 0, s>>>(a);
  return true;
}

// Tile by the number of outputs (us at 8 rows, other weights read in between; the library and the launch it replaces in
// brackets):
//   up to 3071: 8-row tiles, so that 2048 outputs are 256 workgroups (2048 x 2048 4.8, 16-row tiles 5.5 [8.5]; 2048 x 4096
//   7.3 / 9.0 [11.5]; 2048 x 8192 with the squared ReLU 11.9 / 15.2 [15.6])
//   16-row tiles from there (17688 x 2048 21.9, 8-row tiles 23.9 [49.6]; 4096 x 14336 24.8 / 33 [27.2])
//   two 16-row tiles that share x from 24576 (32768 x 2048 to fp32 32.1, one tile 35.4 [35.3])
// Gated pairs are two tiles as well (8192 x 2048 17.2 [20.1], 14336 x 4096 49.2 [67.2]).  Four blocks a chunk where they
// are all of a wave's share, else two (more bytes in flight cost waves); four waves where K does not divide by eight's.
template <int EPI, bool XF>
bool by_shape(const Args& a, hipStream_t s) {
  if (a.K <= SMALL_K) {
    row_linear_small_kernel<EPI, XF><<<(a.N + 15) / 16, 64, 0, s>>>(a);
    return true;
  }
  if constexpr (EPI == EPI_GLU) {
    return run<2, 16, 4, 4, EPI, XF>(a, s) || run<2, 16, 4, 1, EPI, XF>(a, s);
  } else {
    const bool whole = a.K <= 64 * 8 * 4;
    if (a.N < 3072 && ((whole && run<1, 8, 8, 4, EPI, XF>(a, s)) || run<1, 8, 8, 2, EPI, XF>(a, s))) return true;
    if (a.N >= 24576 && run<2, 16, 4, 4, EPI, XF>(a, s)) return true;
    return (whole && run<1, 16, 8, 4, EPI, XF>(a, s)) || run<1, 16, 8, 2, EPI, XF>(a, s) || run<1, 16, 4, 1, EPI, XF>(a, s);
  }
}

}  // namespace

bool launch_row_linear(const void* x, long long ldx, const void* W, void* out, long long ldo, int M, int N, int K, int f32_out,
                       int relu2, int glu, hipStream_t s) {
  const Args a{(const bf16*)x, ldx, (const bf16*)W, out, ldo, M, N, K};
  return glu ? by_shape<EPI_GLU, false>(a, s) : f32_out ? by_shape<EPI_F32, false>(a, s)
         : relu2 ? by_shape<EPI_BF16, true>(a, s) : by_shape<EPI_BF16, false>(a, s);
}
