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
#include "row_units.h"

#include <type_traits>

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
// a launch's problems (blockIdx.y), of the same sizes and strides, these many bytes apart; rows past 16 by blockIdx.z
struct Problems {
  Args a;
  long long dx, dw, dout;
};
template <int EPI>
SYM_DEV Args problem(const Problems& ps) {
  Args a = ps.a;
  const int y = blockIdx.y, z = blockIdx.z;
  a.x = reinterpret_cast<const bf16*>(reinterpret_cast<const char*>(a.x) + y * ps.dx) + 16 * z * a.ldx;
  a.W = reinterpret_cast<const bf16*>(reinterpret_cast<const char*>(a.W) + y * ps.dw);
  a.out = reinterpret_cast<char*>(a.out) + y * ps.dout + 16 * z * a.ldo * (EPI == EPI_F32 ? 4 : 2);
  a.M = min(16, a.M - 16 * z);
  return a;
}

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

// RT: weight tiles of a workgroup.  RH: weight rows of a tile, 16 or 8.  Every wave has the same number of whole blocks, UK deep
// each: four load instructions a tile.
//
// Four load instructions read a block: 256 contiguous bytes of 16 rows (RH 8: 512 of 8), and quad_transpose makes four operands of
// them.  x is read the same way.  What bounds the launch is what a CU takes in, x among it (16 rows of 2048 x 8192: 256 KB of x
// behind 128 KB of weights); while neighbouring lanes read different rows, that went at 37 bytes a ns.
// With RH = 8, lanes 0-7 of 16 hold an operand's first 128 of k, lanes 8-15 its second, which a half_swap brings to the rows' own
// lanes for the second product; rows 8-15 of the products are dropped.
//
// EPI_F32 sums each 128 of k apart (32768 x 2048, two waves of 1024: off by 1.9e-7 of the result in one chain, 8.7e-8 so, 8192 x 2048 1.3e-7
// and 8.3e-8, 2048 x 14336 at 16 rows 3.7e-7 and 1.2e-7; in the same time).
//
// M8: RH = 8 and at most 8 rows of x, which then are read like the weights.  One product of the two registers as they are
// holds the first half's result in its upper left quarter and the second's in its lower right one (the others mix the halves
// and are dropped): half the x traffic, which is twice the weights' otherwise, half the matrix products and no exchange.
//
// More: what a launch does beside its product.  RowRide: row work that the product does not read, by the workgroups behind its tiles (a
// decode step's rotation or convolution beside the feed-forward's second product; launches of 4.7 us each, most of it latency).
struct Nothing {};
SYM_DEV void ride(const RowRide& r, int wg, int threads) {
  const int row = wg / r.per_row, part = wg - row * r.per_row;
  const int first = part * threads + (int)threadIdx.x;
  if (r.conv.out) {
    if (first < r.conv.C) conv_silu_save<bf16>(r.conv, row, first);
  } else {
    qkv_rope_row<bf16>(r.rope, row, first, threads * r.per_row);
  }
}

template <int RT, int RH, int NW, int EPI, bool XF, bool M8 = false, typename More = Nothing>
__global__ __launch_bounds__(NW * 64) void row_linear_kernel(Problems ps, More more) {
  const Args a = problem<EPI>(ps);
  if constexpr (std::is_same<More, RowRide>::value) {
    constexpr int out = EPI == EPI_GLU ? RH : RH * RT;
    const int tiles = (a.N + out - 1) / out;
    if ((int)blockIdx.x >= tiles) return ride(more, blockIdx.x - tiles, NW * 64);
  }
  static_assert(!M8 || (RH == 8 && RT == 1 && EPI != EPI_GLU), "M8: one tile of 8 rows");
  constexpr int UK = RH == 16 ? 128 : 256;
  constexpr int XL = RH == 16 || M8 ? 1 : 2;      // x: 128-deep (M8: 256-deep) parts of a block
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0 = blockIdx.x * (EPI == EPI_GLU ? RH : RH * RT);
  // the lane's row among those of load 0 (load i: i rows on) and its bytes in a row of a block, of a tile of 16 and of 8 rows
  const int row16 = lane & 12, row8 = lane & 4;
  const unsigned in16 = 16 * ((lane & 3) + 4 * (lane >> 4)), in8 = in16 + 32 * (lane & 8);

  // rows past the end repeat the last one; their products are not stored
  unsigned wo[RT][4], xo[4];
  const char* wb[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    const int first = EPI == EPI_GLU ? n0 : n0 + RH * rt;
    const int base = min(first, a.N - 1);
    wb[rt] = reinterpret_cast<const char*>(a.W + (long long)(base + (EPI == EPI_GLU ? rt * a.N : 0)) * a.K);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      wo[rt][i] = (unsigned)((min(first + (RH == 16 ? row16 : row8) + i, a.N - 1) - base) * a.K) * 2 + (RH == 16 ? in16 : in8);
  }
  const char* xb = reinterpret_cast<const char*>(a.x);
#pragma unroll
  for (int i = 0; i < 4; ++i) xo[i] = (unsigned)(min((M8 ? row8 : row16) + i, a.M - 1) * a.ldx) * 2 + (M8 ? in8 : in16);

  f32x4 acc[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) acc[rt] = f32x4{0.f, 0.f, 0.f, 0.f};

  u32x4 w[2][RT][4], xv[2][XL][4];
  // (x first: it comes from the L2, and is turned while the weights are on their way)
  auto load = [&](int b, int blk) {
#pragma unroll
    for (int t = 0; t < XL; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) xv[b][t][i] = *reinterpret_cast<const u32x4*>(xb + 2 * UK * blk + 256 * t + xo[i]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int i = 0; i < 4; ++i) w[b][rt][i] = ld_nt16(reinterpret_cast<const bf16*>(wb[rt] + 2 * UK * blk + wo[rt][i]));
  };
  // parts (EPI_F32, whose sums are the result): each block's sum apart
  auto multiply = [&](int b, auto parts) {
    constexpr bool PARTS = decltype(parts)::value;
    Pack8 f[XL][4];
#pragma unroll
    for (int t = 0; t < XL; ++t) {
      u32x4(&x)[4] = xv[b][t];
      quad_transpose(x[0], x[1], x[2], x[3]);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        f[t][i].w = x[i];
        if constexpr (XF) relu_squared(f[t][i]);
      }
    }
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      u32x4(&v)[4] = w[b][rt];
      quad_transpose(v[0], v[1], v[2], v[3]);
      f32x4 sum = PARTS ? f32x4{0.f, 0.f, 0.f, 0.f} : acc[rt], half = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        Pack8 p;
        p.w = v[i];
        sum = mfma16(p.v, f[0][i].v, sum);
        if constexpr (XL == 2) {
          p.w = half_swap<0x3>(v[i], v[i]);
          f32x4& to = EPI == EPI_F32 ? half : sum;
          to = mfma16(p.v, f[1][i].v, to);
        }
      }
      if constexpr (XL == 2 && EPI == EPI_F32) sum += half;
      acc[rt] = PARTS ? acc[rt] + sum : sum;
    }
  };
  // The loads of a block stand ahead of the products of the one before (the scheduler, left alone, moves them behind to
  // save registers), and the last block's successor is itself, read again: behind a branch every wait would drain all
  // loads.
  const int per = a.K / UK / NW, s0 = wid * per, last = s0 + per - 1;
  load(0, s0);
  __builtin_amdgcn_sched_barrier(0);
  constexpr std::integral_constant<bool, EPI == EPI_F32> parts;
  if (per == 1) {
    multiply(0, std::false_type());
  } else {
    for (int s = s0; s <= last; s += 2) {
      load(1, min(s + 1, last));
      __builtin_amdgcn_sched_barrier(0);
      multiply(0, parts);
      if (s == last) break;
      __builtin_amdgcn_sched_barrier(0);
      load(0, min(s + 2, last));
      __builtin_amdgcn_sched_barrier(0);
      multiply(1, parts);
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  __shared__ f32x4 red[NW][RT][64];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) red[wid][rt][lane] = acc[rt];
  __syncthreads();
  auto sum = [&](int rt) {
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      f32x4 part = red[i][rt][lane];
      if constexpr (M8) part += red[i][rt][(lane + 40) & 63];      // lane 40 on: the second half's
      v = i ? v + part : part;
    }
    return v;
  };
  for (int rt = wid; rt < (EPI == EPI_GLU ? 1 : RT); rt += NW)
    store_rows<RH, EPI>(a, n0 + RH * rt, lane, sum(rt), EPI == EPI_GLU ? sum(RT - 1) : f32x4{});
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
__global__ __launch_bounds__(64) void row_linear_small_kernel(Problems ps) {
  const Args a = problem<EPI>(ps);
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

// Up to 16 outputs of many rows into fp32 (step sizes and gates of a prompt step): 16 rows a workgroup, whose waves take the 128-deep
// blocks of K in turn, read as row_linear_kernel reads them, two in flight, and meet in LDS.  What a CU takes in bounds it: 16 x 2048 at
// 300 / 1530 / 8100 rows 4.4 / 4.5 / 7.1 us (neighbouring lanes on different rows 5.5 / 5.6 / 9.4; the library 5.5 / 5.3 / 21.1, behind a
// prompt step's other launches 10.5 at 1530), 16 x 1024 3.5 / 3.6 / 5.0 (4.3 / 4.3 / 9.7); 4096 deep it is behind, 6.7 / 6.8 (6.2 / 6.3).
constexpr int NARROW_WAVES = 8;

__global__ __launch_bounds__(64 * NARROW_WAVES) void narrow_linear_kernel(Args a) {
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r16 = lane & 15, h = lane >> 4;
  const int m0 = 16 * blockIdx.x, blocks = a.K / 128, in = 8 * ((lane & 3) + 4 * h);
  const bf16 *xr[4], *wr[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    xr[i] = a.x + min(m0 + (lane & 12) + i, a.M - 1) * a.ldx + in;
    wr[i] = a.W + (long long)min((lane & 12) + i, a.N - 1) * a.K + in;
  }
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int b = wid; b < blocks; b += 2 * NARROW_WAVES) {
    u32x4 x[2][4], w[2][4];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int k = 128 * min(b + u * NARROW_WAVES, blocks - 1);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        x[u][i] = *reinterpret_cast<const u32x4*>(xr[i] + k);
        w[u][i] = *reinterpret_cast<const u32x4*>(wr[i] + k);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      if (b + u * NARROW_WAVES >= blocks) break;
      quad_transpose(x[u][0], x[u][1], x[u][2], x[u][3]);
      quad_transpose(w[u][0], w[u][1], w[u][2], w[u][3]);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        Pack8 p, q;
        p.w = w[u][i], q.w = x[u][i];
        acc = mfma16(p.v, q.v, acc);
      }
      settle(acc);
    }
  }
  settle(acc);
  __shared__ f32x4 red[NARROW_WAVES][64];
  red[wid][lane] = acc;
  __syncthreads();
  if (wid) return;
#pragma unroll
  for (int i = 1; i < NARROW_WAVES; ++i) acc += red[i][lane];
  const int m = m0 + r16, n = 4 * h;      // N is a multiple of 4
  if (m < a.M && n < a.N) *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(a.out) + m * a.ldo + n) = acc;
}

// what a launch does: its problems, how many, and work beside them or null
struct Job {
  const Problems& ps;
  int count;
  const RowRide* beside;
  bool plain() const { return count == 1 && !beside && ps.a.M <= 16; }
  dim3 grid(int tiles) const { return dim3(tiles, count, (ps.a.M + 15) / 16); }
};

template <int NW, int KB, int EPI, bool XF>
bool walk(const Job& j, hipStream_t s) {
  const Args& a = j.ps.a;
  if (a.K != 64 * NW * KB || !j.plain()) return false;
  constexpr int OUT = EPI == EPI_GLU ? 8 : 16;
  const int tiles = (a.N + OUT - 1) / OUT;
  row_linear_walk_kernel<NW, KB, EPI, XF><<<tiles < 256 ? tiles : 256, NW * 64, 0, s>>>(a);
  return true;
}

template <int RT, int RH, int NW, int EPI, bool XF, bool M8>
bool run(const Job& j, hipStream_t s) {
  const Args& a = j.ps.a;
  if (a.K % ((RH == 16 ? 128 : 256) * NW)) return false;
  constexpr int rows = EPI == EPI_GLU ? RH : RH * RT;
  const int tiles = (a.N + rows - 1) / rows;
  if (!j.beside) {
    row_linear_kernel<RT, RH, NW, EPI, XF, M8><<<j.grid(tiles), NW * 64, 0, s>>>(j.ps, Nothing{});
    return true;
  }
  if constexpr (EPI == EPI_BF16 && XF) {
    if (j.beside) {
      RowRide r = *j.beside;
      r.per_row = r.conv.out ? (r.conv.C + NW * 64 - 1) / (NW * 64) : 2;
      row_linear_kernel<RT, RH, NW, EPI, XF, M8, RowRide><<<tiles + r.per_row * r.rows, NW * 64, 0, s>>>(j.ps, r);
      return true;
    }
  }
  return false;
}

// With `waves` waves if these divide K's blocks, else with another number of them
template <int RT, int RH, int EPI, bool XF, bool M8 = false>
bool run_waves(const Job& j, int waves, hipStream_t s) {
  switch (waves) {
    case 8: if (run<RT, RH, 8, EPI, XF, M8>(j, s)) return true; break;
    case 6: if (run<RT, RH, 6, EPI, XF, M8>(j, s)) return true; break;
    case 2: if (run<RT, RH, 2, EPI, XF, M8>(j, s)) return true; break;
    default: break;
  }
  if (run<RT, RH, 4, EPI, XF, M8>(j, s)) return true;
  if constexpr (RH == 8)
    if (run<RT, RH, 7, EPI, XF, M8>(j, s) || run<RT, RH, 6, EPI, XF, M8>(j, s) || run<RT, RH, 5, EPI, XF, M8>(j, s) ||
        run<RT, RH, 3, EPI, XF, M8>(j, s))
      return true;
  return run<RT, RH, 2, EPI, XF, M8>(j, s);      // (RH 16: takes every K, an even number of blocks)
}

// Tile by the number of outputs (us; before / now: rows of neighbouring lanes / of lane quads, at 1, 8, 16 rows):
//   up to 2048: 8-row tiles, so that 2048 outputs are 256 workgroups.  Up to 8 blocks of K a wave each, then four waves (2048 x
//   2048 3.9, 4.5, 5.2 / 4.0, 4.2, 4.8; x 4096 5.5, 6.6, 8.4 / 5.4, 5.6, 7.2; x 14336 12.7, 15.7, 21.6 / 11.6, 12.4, 16.7); M8
//   with eight where their shares would lie 4 KB apart (2048 x 8192, 8 rows: four 8.9, eight 8.8, before 10.3; x 16384 19.4,
//   16.7, 18.1); squared ReLUs, of which every workgroup takes all, with eight or six (9 to 16 rows of 2048 x 8192 four 13.3, eight
//   12.7, before 12.6; 512 x 8192 12.9, 11.5, 11.9; 264 x 3072 four 6.4, six 6.0, before 6.2; 1 to 8 of 512 x 4096 5.4, 5.1, 5.3)
//   from 2049 on 16-row tiles, RT of them sharing x: 1 or 2 while that is one round of the 256 CUs (2560 x 2048 4.9, 6.2, 7.7 /
//   4.9, 5.0, 5.2 (8-row tiles 5.0, 5.2, 7.5); 4096 x 2048 6.4, 6.6, 7.5 / 5.2, 5.3, 5.6; 6144 x 2048 8.3, 8.5, 9.0 / 6.9, 6.9,
//   7.1 (RT 1: 7.5, 7.7, 8.1); 8192 x 4096 13.7, 14.1, 15.5 / 13.3, 12.9, 12.7), then 2 or 3 by the rounds, whose cost is
//   a tile's each and half a tile's for x (10240 x 2048 RT 2 / 3 10.8 / 9.3 [before 11.6]; 17440 16.0 / 14.7 [16.0]; 32768
//   23.0 / 26 [27.1])
//   past 40960 outputs rounds run into each other: three only while they are at most 6, full to 7 / 8 (73728 x 2048 walk / three 51.0,
//   53.4, 55.3 / 49.2, 49.9, 52.1), else the walk of 2048 (50304: 36.9, 37.3, 39.1 / 39.7, 39.9, 41.0), and one, for more rows two
//   (100352 x 1024 one / two / three 36.2, 38.4, 44.8 / 37.1, 37.9, 40.8 / 39.7, 41.4, 44.0)
//   one from 8192 deep on (8192 x 8192 23.8, 27.4, 33.0 / 23.4, 23.3, 25.6; RT 2 28.7, 29.1, 29.6), where K has eight or four shares: two
//   waves of one tile have too few loads out (32768 x 9472 at 1, 16 rows 108.8, 122.4, so 92.0, 94.2, before 91.8, 137.6)
//   the walk where many tiles of few blocks, or of many, pass: 12288 x 1536 walk / tiles 8.5 / 8.8, 32768 x 1536 16.9 / 19.2 (8192 x
//   1536 at 1, 16 rows 6.4, 7.5 / 6.9, 6.9), 28672 x 4096 37.9 / 40.2, against 16384 x 4096 23.6 / 22.6; 12288 x 3072 even
//   (its widths are those that it is written out for: its waves hold their shares of x and of two tiles in registers, so a K needs a
//   number of waves and blocks of its own; others, as 2304, take the tiles at every size)
// Waves of 16-row tiles: a block each up to 8 in one round (12288 x 1024, RT 3: eight 6.2, two 6.9); then four (two of RT 3), eight
// from 8192 deep on (3000 x 8192 12.4 / 11.4).  Where more rounds cover a wait, one for 8 blocks, at least two (32768 x 2048 two /
// four 23.0 / 23.7, 16384 x 4096 four / two 22.6 / 25; gated 8192 x 1024 two / eight 7.7 / 9.3), four for 4 blocks.
// Gated pairs are two tiles of 16 outputs' (1024 x 1024 4.4, 4.8, 5.0 / 4.2, 4.3, 4.3; 8192 x 8192 56, 57, 59 / 45, 46, 47).  Of the
// walk's widths they are where they come near whole rounds (8192 x 2048 12.7, 13.0, 13.6 / 12.6, 12.6, 12.8; 4096 x 4096 14.0 to
// 15.9 / 12.2 to 12.5; but 4360 x 2048 9.9 / 10.7, 6144 x 4096, three rounds of the walk, 19.3 / 20.7, 14336 x 4096 38.7 / 41.1), with
// few outputs for more than 8 rows (512 x 4096 at 1, 16 rows 8.6, 10.7 / 9.4, 9.5).
template <int EPI, bool XF>
bool by_shape(const Job& j, hipStream_t s) {
  const Args& a = j.ps.a;
  if (a.K <= SMALL_K) {
    if (j.beside) return false;
    row_linear_small_kernel<EPI, XF><<<j.grid((a.N + 15) / 16), 64, 0, s>>>(j.ps);
    return true;
  }
  const int tiles = (a.N + 15) / 16, blocks = a.K / 128;
  bool walks;
  if constexpr (EPI == EPI_GLU) {
    const bool near = (tiles > 128 && tiles <= 256) || (tiles > 384 && tiles <= 512) || (tiles <= 128 && a.M > 8);
    walks = a.K == 3072 || ((a.K == 2048 || a.K == 4096) && !near);
  } else {
    walks = ((a.K == 1536 || a.K == 3072) && a.N > 8192) || (a.K == 1536 && a.N > 4096 && a.M <= 4) || (a.K == 4096 && a.N > 16384);
  }
  if (walks && !j.plain()) return false;
  if (walks && (walk<8, 3, EPI, XF>(j, s) || walk<8, 6, EPI, XF>(j, s) || walk<8, 8, EPI, XF>(j, s))) return true;
  auto waves = [&](int rt, int wgs) {
    const bool one = wgs <= 256;
    if (blocks <= (one ? 8 : 4)) return blocks;
    if (blocks >= 64) return 8;
    return one && rt < 3 ? 4 : blocks <= 20 ? 2 : 4;
  };
  if constexpr (EPI == EPI_GLU) {
    if (walks && walk<16, 2, EPI, XF>(j, s)) return true;
    return run_waves<2, 16, EPI, XF>(j, waves(2, tiles), s);
  } else {
    if (a.N <= 2048 && a.K % 256 == 0) {
      const int deep = a.K / 256;
      const int most = XF ? (deep % 8 ? 6 : 8) : a.M <= 8 && deep % 32 == 0 ? 8 : 4, shares = deep <= 8 ? deep : most;
      if (a.M <= 8 ? run_waves<1, 8, EPI, XF, true>(j, shares, s) : run_waves<1, 8, EPI, XF>(j, shares, s))
        return true;
    }
    const int two = (tiles + 1) / 2, three = (tiles + 2) / 3;
    if (tiles <= 256 || (blocks >= 64 && blocks % 4 == 0)) return run_waves<1, 16, EPI, XF>(j, waves(1, tiles), s);
    const int rounds2 = (two + 255) / 256, rounds3 = (three + 255) / 256;
    if (two > 1280 && (rounds3 > 6 || 8 * three < 7 * 256 * rounds3)) {
      if (a.K == 2048 && !j.plain()) return false;
      if (walk<16, 2, EPI, XF>(j, s)) return true;
      if (a.K > 512 && (a.M <= 4 || (a.M <= 8 && 10 * two < 9 * 256 * rounds2))) return run_waves<1, 16, EPI, XF>(j, waves(1, tiles), s);
    } else if (two > 256 && 7 * rounds3 < 5 * rounds2) {
      return run_waves<3, 16, EPI, XF>(j, waves(3, three), s);
    }
    return run_waves<2, 16, EPI, XF>(j, waves(2, two), s);
  }
}

}  // namespace

void launch_narrow_linear(const void* x, long long ldx, const void* W, float* out, long long ldo, int M, int N, int K, hipStream_t s) {
  const Args a{(const bf16*)x, ldx, (const bf16*)W, out, ldo, M, N, K};
  narrow_linear_kernel<<<(M + 15) / 16, 64 * NARROW_WAVES, 0, s>>>(a);
}

bool launch_row_linear(const void* x, long long ldx, const void* W, void* out, long long ldo, int M, int N, int K, int f32_out,
                       int relu2, int glu, hipStream_t s) {
  const Problems ps{{(const bf16*)x, ldx, (const bf16*)W, out, ldo, M, N, K}, 0, 0, 0};
  const Job j{ps, 1, nullptr};
  return glu ? by_shape<EPI_GLU, false>(j, s) : f32_out ? by_shape<EPI_F32, false>(j, s)
         : relu2 ? by_shape<EPI_BF16, true>(j, s) : by_shape<EPI_BF16, false>(j, s);
}

bool launch_row_linear_many(const void* x, long long ldx, long long dx, const void* W, long long dw, void* out, long long ldo, long long dout,
                            int count, int M, int N, int K, hipStream_t s) {
  const Problems ps{{(const bf16*)x, ldx, (const bf16*)W, out, ldo, M, N, K}, dx, dw, dout};
  return by_shape<EPI_BF16, false>(Job{ps, count, nullptr}, s);
}

bool launch_row_linear_beside(const void* x, long long ldx, const void* W, void* out, long long ldo, int M, int N, int K, const RowRide& r,
                              hipStream_t s) {
  const Problems ps{{(const bf16*)x, ldx, (const bf16*)W, out, ldo, M, N, K}, 0, 0, 0};
  return by_shape<EPI_BF16, true>(Job{ps, 1, &r}, s);
}
