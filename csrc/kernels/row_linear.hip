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

// RT: weight tiles of a workgroup.  RH: weight rows of a tile, 16 or 8.  U: 64-deep k blocks of a chunk.  Every wave has
// the same number of whole chunks.
//
// One load instruction reads 128 contiguous bytes (a 64-deep k block) of each of 8 weight rows: lanes 0-7 of each row of 16
// lanes hold the block's first 32-deep step, lanes 8-15 its second.  Two such loads (rows 0-7, rows 8-15) become the two
// steps' A operands by exchanging halves, 4 v_mov_dpp each.  With RH = 8 there is one load, and rows 8-15 of the product
// are dropped.
//
// M8: RH = 8 and at most 8 rows of x, which then are read like the weights.  One product of the two registers as they are
// holds the first step's result in its upper left quarter and the second's in its lower right one (the others mix the steps
// and are dropped): half the x traffic, which is twice the weights' otherwise, half the matrix products and no exchange.
template <int RT, int RH, int NW, int U, int EPI, bool XF, bool M8 = false>
__global__ __launch_bounds__(NW * 64) void row_linear_kernel(Args a) {
  static_assert(!M8 || (RH == 8 && RT == 1 && EPI != EPI_GLU), "M8: one tile of 8 rows");
  constexpr int LD = RH / 8;  // loads of a block
  constexpr int XL = M8 ? 1 : 2;
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
  const unsigned xo = (unsigned)(min(M8 ? r16 & 7 : r16, a.M - 1) * a.ldx + (M8 ? 4 * (r16 & 8) : 0) + 8 * h) * 2;

  f32x4 acc[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) acc[rt] = f32x4{0.f, 0.f, 0.f, 0.f};

  u32x4 w[2][U][RT][LD];
  Pack8 xv[U][XL];
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
      for (int t = 0; t < XL; ++t) xv[u][t].w = *reinterpret_cast<const u32x4*>(xb + 128 * (blk + u) + 64 * t + xo);
  };
  auto multiply = [&](int b) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if constexpr (XF) {
#pragma unroll
        for (int t = 0; t < XL; ++t) relu_squared(xv[u][t]);
      }
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        Pack8 f0, f1;
        if constexpr (M8) {
          f0.w = w[b][u][rt][0];
          acc[rt] = mfma16(f0.v, xv[u][0].v, acc[rt]);
          continue;
        }
        const u32x4 lo = w[b][u][rt][0], hi = w[b][u][rt][LD - 1];
        f0.w = LD == 2 ? half_swap<0xc>(lo, hi) : lo;
        f1.w = half_swap<0x3>(hi, lo);
        acc[rt] = mfma16(f0.v, xv[u][0].v, acc[rt]);
        acc[rt] = mfma16(f1.v, xv[u][XL - 1].v, acc[rt]);
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
    if constexpr (M8) {  // lane 40 on: the second step's part
#pragma unroll
      for (int i = 0; i < NW; ++i) v += red[i][rt][(lane + 40) & 63];
    }
    return v;
  };
  store_rows<RH, EPI>(a, n0 + RH * wid, lane, sum(wid), EPI == EPI_GLU ? sum(RT - 1) : f32x4{});
}

// Many tiles: x stays in registers.  A workgroup's waves hold their shares of x (KB 64-deep blocks each, K = 64 NW KB) and walk
// the 16-row tiles blockIdx.x, + gridDim.x, ..  Read per tile, x costs up to as much L2 traffic as the weights cost HBM.  The
// next tile's weights are in flight while a tile is multiplied (two tiles ahead is slower, 8 rows of 8192 x 2048 gated 13.8 ->
// 14.7 us: what the last tile reads for nothing grows); the waves sum a tile's parts in turn, and one barrier a tile (two
// buffers) keeps them together.  EPI_GLU: 8 gate rows and the 8 up rows of the same outputs are one tile, so a pair meets
// across the halves of the result.
template <int NW, int KB, int EPI, bool XF>
__global__ __launch_bounds__(NW * 64) void row_linear_walk_kernel(Args a) {
  constexpr int OUT = EPI == EPI_GLU ? 8 : 16;
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, h = lane >> 4;
  const int tiles = (a.N + OUT - 1) / OUT, step = gridDim.x;
  __shared__ f32x4 red[2][NW][64];

  const char* xb = reinterpret_cast<const char*>(a.x) + 128 * KB * wid + (min(r16, a.M - 1) * a.ldx + 8 * h) * 2;
  const char* Wb = reinterpret_cast<const char*>(a.W) + 128 * KB * wid;
  const unsigned kin = (unsigned)(4 * (r16 & 8) + 8 * h) * 2;
  u32x4 w[2][KB][2];
  Pack8 xv[KB][2];
  // (past the last tile: one line for all, so that a tile's wait never stands behind a branch)
  auto load_w = [&](int b, int t) {
    const bool in = t < tiles;
    const int n0 = in ? t * OUT : 0;
    const char* base = Wb + (long long)n0 * a.K * 2;
#pragma unroll
    for (int l = 0; l < 2; ++l) {
      const int row = min((EPI == EPI_GLU ? 0 : 8 * l) + (r16 & 7), a.N - 1 - n0);
      const unsigned off = in ? (unsigned)(row * a.K) * 2 + kin : 0;
      const char* src = base + (EPI == EPI_GLU && l ? (long long)a.N * a.K * 2 : 0);
#pragma unroll
      for (int u = 0; u < KB; ++u) w[b][u][l] = ld_nt16(reinterpret_cast<const bf16*>(src + 128 * u + off));
    }
  };
  auto tile = [&](int b, int t, int turn) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < KB; ++u) {
      Pack8 f0, f1;
      f0.w = half_swap<0xc>(w[b][u][0], w[b][u][1]);
      f1.w = half_swap<0x3>(w[b][u][1], w[b][u][0]);
      acc = mfma16(f0.v, xv[u][0].v, acc);
      acc = mfma16(f1.v, xv[u][1].v, acc);
    }
    red[b][wid][lane] = acc;
    __builtin_amdgcn_s_waitcnt(0xc07f);      // lgkmcnt(0): the next tile's loads stay in flight
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (wid != turn) return;
    auto sum = [&](int from) {
      f32x4 v = red[b][0][from];
#pragma unroll
      for (int i = 1; i < NW; ++i) v += red[b][i][from];
      return v;
    };
    if constexpr (EPI == EPI_GLU) {
      f32x4 v = sum(lane), up;
#pragma unroll
      for (int r = 0; r < 4; ++r) up[r] = __shfl_down(v[r], 32, 64);
      store_rows<8, EPI>(a, t * OUT, lane, v, up);
    } else {
      store_rows<16, EPI>(a, t * OUT, lane, sum(lane), f32x4{});
    }
  };
  int t = blockIdx.x, turn = 0;
  load_w(0, t);
#pragma unroll
  for (int u = 0; u < KB; ++u)
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      xv[u][k].w = *reinterpret_cast<const u32x4*>(xb + 128 * u + 64 * k);
      if constexpr (XF) relu_squared(xv[u][k]);
    }
  while (true) {
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      if (t >= tiles) return;
      load_w(b ^ 1, t + step);
      __builtin_amdgcn_sched_barrier(0);
      tile(b, t, turn);
      t += step;
      turn = turn + 1 == NW ? 0 : turn + 1;
    }
  }
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

template <int NW, int KB, int EPI, bool XF>
bool walk(const Args& a, hipStream_t s) {
  if (a.K != 64 * NW * KB) return false;
  constexpr int OUT = EPI == EPI_GLU ? 8 : 16;
  const int tiles = (a.N + OUT - 1) / OUT;
  row_linear_walk_kernel<NW, KB, EPI, XF><<<tiles < 256 ? tiles : 256, NW * 64, 0, s>>>(a);
  return true;
}

template <int RT, int RH, int NW, int U, int EPI, bool XF, bool M8 = false>
bool run(const Args& a, hipStream_t s) {
  if (a.K % (64 * NW * U)) return false;
  constexpr int rows = EPI == EPI_GLU ? RH : RH * RT;
  row_linear_kernel<RT, RH, NW, U, EPI, XF, M8><<<(a.N + rows - 1) / rows, NW * 64, 0, s>>>(a);
  return true;
}

// Tile by the number of outputs (us at 8 rows, other weights read in between; the library and the launch it replaces in
// brackets):
//   up to 3071: 8-row tiles, so that 2048 outputs are 256 workgroups (2048 x 2048 4.8, 16-row tiles 5.5 [8.5]).  M8, as one
//   chunk where a wave's share is at most 8 blocks, else two blocks a chunk (x read twice / M8 at 1 and at 8 rows: 2048 x 4096
//   6.5 / 5.6 and 7.8 / 6.8; 2048 x 8192 9.9 / 9.3 and 12.2 / 12.0, with the squared ReLU 11.5 / 10.6 and 12.8 / 12.3)
//   the walk from 4097 on, where some workgroup has a second tile (8-row or 16-row tiles one by one / walk: 17440 x 2048 21.7 /
//   16.5, 6144 x 2048 10.2 / 8.8, 32768 x 2048 to fp32 32.1 / 27.3, 28672 x 4096 50.7 / 38.6 = 6.1 TB/s; 4096 x 2048 7.8 / 7.6
//   at 16 rows, 6.6 / 6.9 at 2), of the widths that are written out below; 1536 wide always (its other form has four waves of
//   one block a chunk: 2048 outputs 5.5 / 4.6)
//   16-row tiles between the two and for other widths (8-row tiles 3072 x 2048 at 16 rows 7.6, 6.6); two that share x from 24576
// Gated pairs walk (8192 x 2048 18.1 / 13.9, 1024 x 2048 7.9 / 5.9, 14336 x 4096 50.6 / 39.4).  Four blocks a chunk where they are
// all of a wave's share, else two (more bytes in flight cost waves); four waves where K does not divide by eight's.
template <int EPI, bool XF>
bool by_shape(const Args& a, hipStream_t s) {
  if (a.K <= SMALL_K) {
    row_linear_small_kernel<EPI, XF><<<(a.N + 15) / 16, 64, 0, s>>>(a);
    return true;
  }
  const bool walks = EPI == EPI_GLU ? a.K >= 2048 : a.N > 4096 || a.K == 1536;
  if (walks && (walk<8, 3, EPI, XF>(a, s) || walk<16, 2, EPI, XF>(a, s) || walk<8, 6, EPI, XF>(a, s) || walk<8, 8, EPI, XF>(a, s)))
    return true;
  if constexpr (EPI == EPI_GLU) {
    return run<2, 16, 4, 4, EPI, XF>(a, s) || run<2, 16, 4, 1, EPI, XF>(a, s);
  } else {
    const int per = a.K / (64 * 8);  // blocks of each of eight waves
    if (a.N < 3072 && a.M <= 8 &&
        ((per <= 4 && run<1, 8, 8, 4, EPI, XF, true>(a, s)) || (per <= 8 && run<1, 8, 8, 8, EPI, XF, true>(a, s)) ||
         run<1, 8, 8, 2, EPI, XF, true>(a, s)))
      return true;
    const bool whole = per <= 4;
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
