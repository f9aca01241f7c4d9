// Gated delta rule: a linear recurrence whose state [N x P] (fp32, per sequence and head) is corrected towards every new
// key / value pair,
//
//     S <- diag(g_t) S;   u_t = beta_t (v_t - S^T k_t);   S <- S + k_t u_t^T;   o_t = S^T q_t
//
//     beta_t = sigmoid(bz_t),   log g_t = -exp(A_log) softplus(dz_t + dt_bias)     per head, or per head and key channel
//
// q, k fp32 (unit vectors: see conv_silu_qkv), v in the activation dtype; decays, step sizes, states and sums fp32.  A run
// of rows (one sequence's tokens of a step) starts from its state slot (or zero at position 0) and ends in it; each (slot,
// head, column) is read and written by one lane group of one workgroup.
//
// Two forms:
//
// 1. Token by token (decode steps, the 32-bit model): grid (P / columns, heads, runs).  A wave's lanes are PCOLS value
//    columns x SLICES slices of the key channels, the slices in neighbouring lanes: S^T k sits on the serial path of every
//    token, and a sum over neighbouring lanes is two or three cross-lane adds on the vector unit (no LDS round trip).  The
//    vectors that all columns share are staged through LDS for CH tokens at a time, the next batch's loads in flight.
//
// 2. Chunked (prompt steps): with chunks of C = 32 tokens, G_i the running sum of log g inside the chunk and S_0 the state
//    in front of it,
//        u_i = beta_i (v_i - (k_i e^(G_i))^T S_0 - sum_{j < i} Akk_ij u_j),      Akk_ij = sum_n k_i k_j e^(G_i - G_j)
//        o_i = (q_i e^(G_i))^T S_0 + sum_{j <= i} Aqk_ij u_j                      (every exponent <= 0: nothing overflows)
//        S_C = e^(G_C) S_0 + sum_j (k_j e^(G_C - G_j)) u_j^T
//    delta_chunk_prep_kernel (one workgroup per chunk and head, all chunks at once) evaluates Akk, Aqk and T = (I +
//    diag(beta) Akk)^-1 diag(beta) by forward substitution.  One decay per head: the scores are matrix products, times
//    e^(G_i - G_j).  Decays per channel: inside the two diagonal 16 x 16 tiles the exponents of differences are taken per
//    (i, j, channel) on the vector unit; the tile below them factors at the end of the first half, e^(G_i - G_15) e^(G_15 -
//    G_j), both exponents <= 0, and is a matrix product again.
//    delta_chunk_scan_kernel (grid (P / 64, heads, runs)) then walks a run's chunks with
//        R = V - Kt S,   U = T R,   O = Qt S + Aqk U,   S <- D S + Kh^T U
//    as fp32 matrix products (v_mfma_f32_16x16x4_f32; in bf16 parts up to 128 key channels of the bf16 model).  A wave owns 16 value columns and ALL of N: its state stays in
//    accumulator registers for the whole run, and since an accumulator's rows are 4 (lane / 16) + r and a B operand's
//    contraction index is lane / 16, register r of the state IS the B operand of a step that contracts over the rows
//    4 g + r (the A operand is read in the same order: one 16-byte LDS read feeds four steps).  The same holds for R and U.
//    Four waves multiply, four others stage the next chunk (loads, exponentials, LDS) on the same SIMDs meanwhile.
#include "attn_tiles.h"
#include "bf16_parts.h"
#include "common.h"
#include "hybrid_launchers.h"
#include "walk_places.h"

namespace {

constexpr int NT = 256;
constexpr float LOG2E = 1.4426950408889634f;

SYM_DEV float softplus_exact(float v) { return fmaxf(v, 0.f) + log1pf(expf(-fabsf(v))); }
SYM_DEV float sigmoidf(float v) { return 1.f / (1.f + expf(-v)); }

template <int CTRL>
SYM_DEV float dpp_add(float v) {
  return v + __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xf, 0xf, true));
}
// sum over groups of 4 or 8 neighbouring lanes (quad_perm xor 1, xor 2, then the half row mirrored)
template <int SLICES>
SYM_DEV float slice_sum(float v) {
  v = dpp_add<0xB1>(v);
  v = dpp_add<0x4E>(v);
  if (SLICES == 8) v = dpp_add<0x141>(v);
  return v;
}

// NPL: state entries per lane (>= ceil(N / SLICES)); CH: tokens staged per batch
template <typename T, bool CHANNEL, int NPL, int CH, int SLICES>
__global__ __launch_bounds__(NT) void delta_scan_kernel(DeltaRuleArgs a) {
  extern __shared__ float lds[];
  constexpr int PCOLS = 64 / SLICES;
  constexpr int NPAD = NPL * SLICES;
  constexpr int LROW = SLICES * (NPL + 4);           // slices 16 bytes apart in bank space
  constexpr int EPT = (CH * NPAD + NT - 1) / NT;     // staged (token, channel) entries per thread
  constexpr int ASZ = CHANNEL ? CH * LROW : CH;
  constexpr int BUF = 2 * CH * LROW + ASZ + CH;      // q, k, decays, step sizes
  const int N = a.N, P = a.P;
  const int h = blockIdx.y, run = blockIdx.z;
  const int s0 = a.cu_q ? a.cu_q[run] : run, s1 = a.cu_q ? a.cu_q[run + 1] : run + 1;
  if (s1 <= s0) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int ns = lane & (SLICES - 1), pc = lane / SLICES;
  const int p = blockIdx.x * (PCOLS * (NT / 64)) + wave * PCOLS + pc;
  const bool pin = p < P;
  const int n0 = ns * NPL, l0 = ns * (NPL + 4);
  const int pr = a.prev_row[s0];
  const int sv = a.save_slot[s1 - 1];
  const long long gn = (long long)a.G * N;
  const float* q = a.q + (long long)(h / a.hpg) * N;
  const float* k = a.k + (long long)(h / a.hpg) * N;
  const T* v = reinterpret_cast<const T*>(a.v) + (long long)h * P + p;
  const float rate = expf(a.A_log[h]);
  float rq[EPT], rk[EPT], rz[EPT], vn[CH], rb = 0.f, rd = 0.f;
  auto fetch = [&](int t0) {
    const int nt = min(CH, s1 - t0);
#pragma unroll
    for (int u = 0; u < EPT; ++u) {
      const int i = threadIdx.x + NT * u;
      const int tt = i / NPAD, n = i - tt * NPAD;
      const bool in = tt < nt && n < N;
      const long long r = t0 + tt;
      rq[u] = in ? q[r * gn + n] : 0.f;
      rk[u] = in ? k[r * gn + n] : 0.f;
      if (CHANNEL) rz[u] = in ? a.dz[r * a.ldd + (long long)h * N + n] + a.dt_bias[(long long)h * N + n] : 0.f;
    }
    if (threadIdx.x < CH) {
      const bool in = (int)threadIdx.x < nt;
      const long long r = t0 + threadIdx.x;
      rb = in ? a.bz[r * a.ldb + h] : 0.f;
      if (!CHANNEL) rd = in ? a.dz[r * a.ldd + h] + a.dt_bias[h] : 0.f;
    }
#pragma unroll
    for (int tt = 0; tt < CH; ++tt)
      vn[tt] = tt < nt && pin ? (float)v[(long long)(t0 + tt) * a.H * P] : 0.f;
  };
  auto commit = [&](float* buf) {
    float* qS = buf;
    float* kS = buf + CH * LROW;
    float* aS = kS + CH * LROW;
    float* bS = aS + ASZ;
#pragma unroll
    for (int u = 0; u < EPT; ++u) {
      const int i = threadIdx.x + NT * u;
      const int tt = i / NPAD, n = i - tt * NPAD;
      if (tt < CH) {
        const int o = tt * LROW + (n / NPL) * (NPL + 4) + n % NPL;
        qS[o] = rq[u];
        kS[o] = rk[u];
        if (CHANNEL) aS[o] = expf(-rate * softplus_exact(rz[u]));   // (padding channels: k = q = 0, the state stays 0)
      }
    }
    if (threadIdx.x < CH) {
      bS[threadIdx.x] = sigmoidf(rb);
      if (!CHANNEL) aS[threadIdx.x] = expf(-rate * softplus_exact(rd));
    }
  };
  fetch(s0);
  float S[NPL];
  const bool old = pr <= -2 && pin;
  const float* st = a.state + (old ? (long long)(-(pr + 2)) * a.state_stride + (long long)h * N * P + p : 0);
#pragma unroll
  for (int i = 0; i < NPL; ++i) S[i] = old && n0 + i < N ? st[(long long)(n0 + i) * P] : 0.f;
  int flip = 0;
  for (int t0 = s0; t0 < s1; t0 += CH, flip ^= 1) {
    const int nt = min(CH, s1 - t0);
    float* buf = lds + flip * BUF;
    commit(buf);
    float vr[CH], po[CH];
#pragma unroll
    for (int tt = 0; tt < CH; ++tt) vr[tt] = vn[tt];
    __syncthreads();   // this batch is in LDS; every thread has finished the batch before the last (same buffer)
    if (t0 + CH < s1) fetch(t0 + CH);
    const float* qS = buf;
    const float* kS = buf + CH * LROW;
    const float* aS = kS + CH * LROW;
    const float* bS = aS + ASZ;
#pragma unroll
    for (int tt = 0; tt < CH; ++tt) {
      po[tt] = 0.f;
      if (tt < nt) {
        const float4* q4 = reinterpret_cast<const float4*>(qS + tt * LROW + l0);
        const float4* k4 = reinterpret_cast<const float4*>(kS + tt * LROW + l0);
        const float4* a4 = reinterpret_cast<const float4*>(aS + tt * LROW + l0);
        const float at = CHANNEL ? 0.f : aS[tt];
        float d0 = 0.f, d1 = 0.f, d2 = 0.f, d3 = 0.f;
#pragma unroll
        for (int i = 0; i < NPL / 4; ++i) {
          const float4 kv = k4[i];
          float4 av;
          if (CHANNEL) av = a4[i];
          else av = make_float4(at, at, at, at);
          S[4 * i + 0] *= av.x, S[4 * i + 1] *= av.y, S[4 * i + 2] *= av.z, S[4 * i + 3] *= av.w;
          d0 += S[4 * i + 0] * kv.x, d1 += S[4 * i + 1] * kv.y, d2 += S[4 * i + 2] * kv.z, d3 += S[4 * i + 3] * kv.w;
        }
        const float u = bS[tt] * (vr[tt] - slice_sum<SLICES>((d0 + d1) + (d2 + d3)));
        float o0 = 0.f, o1 = 0.f, o2 = 0.f, o3 = 0.f;
#pragma unroll
        for (int i = 0; i < NPL / 4; ++i) {
          const float4 kv = k4[i], qv = q4[i];
          S[4 * i + 0] += kv.x * u, S[4 * i + 1] += kv.y * u, S[4 * i + 2] += kv.z * u, S[4 * i + 3] += kv.w * u;
          o0 += S[4 * i + 0] * qv.x, o1 += S[4 * i + 1] * qv.y, o2 += S[4 * i + 2] * qv.z, o3 += S[4 * i + 3] * qv.w;
        }
        po[tt] = (o0 + o1) + (o2 + o3);
      }
    }
#pragma unroll
    for (int tt = 0; tt < CH; ++tt) po[tt] = slice_sum<SLICES>(po[tt]);
    if (ns == 0 && pin)
#pragma unroll
      for (int tt = 0; tt < CH; ++tt)
        if (tt < nt) a.out[((long long)(t0 + tt) * a.H + h) * P + p] = po[tt];
  }
  if (sv >= 0 && pin) {
    float* so = a.state + (long long)sv * a.state_stride + (long long)h * N * P + p;
#pragma unroll
    for (int i = 0; i < NPL; ++i)
      if (n0 + i < N) so[(long long)(n0 + i) * P] = S[i];
  }
}

// ---- chunked form ------------------------------------------------------------------------------------------------
constexpr int C = 32;            // tokens per chunk
constexpr int LC = C + 4;        // LDS pitch of a [.][C] matrix
// scratch per (row, head): row of T [C] | row of Aqk [C] | G: N key channels, or one value in four
SYM_DEV int ws_cols(bool channel, int N) { return 2 * C + (channel ? N : 4); }

// v_mfma_f32_16x16x4_f32: lane l holds A[l % 16][l / 16], B[l / 16][l % 16], D[4 (l / 16) + r][l % 16] in register r
SYM_DEV f32x4 mfma4(float x, float y, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(x, y, c, 0, 0, 0); }
SYM_DEV f32x4 lds4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
SYM_DEV f32x4 exp2_neg(f32x4 v) {       // 2^v for exponents that are <= 0 where they matter
  f32x4 r;
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = __builtin_amdgcn_exp2f(fminf(v[i], 0.f));
  return r;
}

// grid (64-row tiles x 2 chunks, heads); NN: 16-channel tiles (N <= 16 NN)
template <bool CHANNEL, int NN>
__global__ __launch_bounds__(NT) void delta_chunk_prep_kernel(DeltaRuleArgs a) {
  extern __shared__ float lds[];
  constexpr int NP = 16 * NN, LD = NP + 4;
  constexpr int TSTEP = NT / NP, EPT = C / TSTEP;      // a thread stages channel n of the tokens tt0, tt0 + TSTEP, ..
  const int N = a.N;
  const int h = blockIdx.y, tile = blockIdx.x >> 1, sub = blockIdx.x & 1;
  const int seq = a.tiles[2 * tile], off = a.tiles[2 * tile + 1];
  const int q0 = a.cu_q[seq], qlen = a.cu_q[seq + 1] - q0;
  if (off >= qlen) return;                     // padding tile
  const int nt = min(C, qlen - off - C * sub);
  if (nt <= 0) return;
  const long long r0 = q0 + off + C * sub;
  float* kS = lds;                             // [C][LD]
  float* qS = kS + C * LD;                     // [C][LD]
  float* GS = qS + C * LD;                     // CHANNEL: [C][LD], else [C]
  float* XS = GS + (CHANNEL ? C * LD : C);     // [2 halves of the channels][Akk, Aqk][C][LC]
  float* bS = XS + 4 * C * LC;                 // [C]
  float* LS = XS;                              // afterwards: [C][LC] beta_i Akk_ij below the diagonal
  float* TS = XS + 2 * C * LC;                 // [C][LC]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int n = tid % NP, tt0 = tid / NP;
  const int gn = a.G * N;
  const float rate2 = expf(a.A_log[h]) * LOG2E;
  {
    const float* k = a.k + (r0 + tt0) * gn + (h / a.hpg) * N + n;
    const float* q = a.q + (r0 + tt0) * gn + (h / a.hpg) * N + n;
    const float* dz = CHANNEL ? a.dz + (r0 + tt0) * a.ldd + h * N + n : nullptr;
    const float db = CHANNEL && n < N ? a.dt_bias[h * N + n] : 0.f;
    float rk[EPT], rq[EPT], rz[EPT];
#pragma unroll
    for (int u = 0; u < EPT; ++u) {
      const bool in = tt0 + TSTEP * u < nt && n < N;
      rk[u] = in ? k[(long long)TSTEP * u * gn] : 0.f;
      rq[u] = in ? q[(long long)TSTEP * u * gn] : 0.f;
      if (CHANNEL) rz[u] = in ? dz[TSTEP * u * a.ldd] : 0.f;
    }
#pragma unroll
    for (int u = 0; u < EPT; ++u) {
      const int o = (tt0 + TSTEP * u) * LD + n;
      kS[o] = rk[u];
      qS[o] = rq[u];
      if (CHANNEL) GS[o] = tt0 + TSTEP * u < nt && n < N ? -rate2 * softplus_exact(rz[u] + db) : 0.f;
    }
  }
  if (tid < C) {
    const bool in = tid < nt;
    bS[tid] = in ? sigmoidf(a.bz[(r0 + tid) * a.ldb + h]) : 0.f;
    if (!CHANNEL) {
      float g = in ? -rate2 * softplus_exact(a.dz[(r0 + tid) * a.ldd + h] + a.dt_bias[h]) : 0.f;
#pragma unroll
      for (int o = 1; o < C; o <<= 1) {        // running sum over the chunk's tokens
        const float up = __shfl_up(g, o, 64);
        if (tid >= o) g += up;
      }
      GS[tid] = g;
    }
  }
  __syncthreads();
  const int wc = ws_cols(CHANNEL, N);
  float* ws = a.ws + (r0 * a.H + h) * wc;      // row stride H * wc
  const long long wrow = (long long)a.H * wc;
  if (CHANNEL) {
    if (tid < NP) {
      float g[C];
#pragma unroll
      for (int tt = 0; tt < C; ++tt) g[tt] = GS[tt * LD + tid];
#pragma unroll
      for (int tt = 1; tt < C; ++tt) g[tt] += g[tt - 1];
#pragma unroll
      for (int tt = 0; tt < C; ++tt) {
        GS[tt * LD + tid] = g[tt];
        if (tt < nt && tid < N) ws[tt * wrow + 2 * C + tid] = g[tt];
      }
    }
    __syncthreads();
  } else if (tid < nt) {
    ws[tid * wrow + 2 * C] = GS[tid];
  }
  // scores.  A wave takes one half of the channels (half) of Akk or Aqk (kind) for the matrix products
  constexpr int NH = NN > 1 ? NN / 2 : 1;      // 16-channel tiles per half
  const int half = wave >> 1, kind = wave & 1;
  const int col = lane & 15, g = lane >> 4;
  {
    const float* iS = kind ? qS : kS;
    f32x4 d00 = {0.f, 0.f, 0.f, 0.f}, d10 = d00, d11 = d00;
    if (NN > 1 || half == 0) {
#pragma unroll
      for (int t = 0; t < NH; ++t) {
        const int c = 16 * (half * NH + t) + 4 * g;
        f32x4 i1 = lds4(iS + (16 + col) * LD + c);
        f32x4 j0 = lds4(kS + col * LD + c);
        if (CHANNEL) {
          const f32x4 mid = lds4(GS + 15 * LD + c);
          i1 = i1 * exp2_neg(lds4(GS + (16 + col) * LD + c) - mid);
          j0 = j0 * exp2_neg(mid - lds4(GS + col * LD + c));
#pragma unroll
          for (int r = 0; r < 4; ++r) d10 = mfma4(i1[r], j0[r], d10);
        } else {
          const f32x4 i0 = lds4(iS + col * LD + c), j1 = lds4(kS + (16 + col) * LD + c);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            d00 = mfma4(i0[r], j0[r], d00);
            d10 = mfma4(i1[r], j0[r], d10);
            d11 = mfma4(i1[r], j1[r], d11);
          }
        }
      }
    }
    float* X = XS + (half * 2 + kind) * C * LC;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      X[(16 + 4 * g + r) * LC + col] = d10[r];
      if (!CHANNEL) {
        X[(4 * g + r) * LC + col] = d00[r];
        X[(16 + 4 * g + r) * LC + 16 + col] = d11[r];
      }
    }
  }
  if (CHANNEL) {
    // diagonal tiles: wave (half, tile), a 2 x 2 block of (i, j) per lane, both kinds
    const int dt = wave & 1, ib = lane >> 3, jb = lane & 7;
    const int i0 = 16 * dt + 2 * ib, j0 = 16 * dt + 2 * jb;
    float kk[2][2] = {{0.f, 0.f}, {0.f, 0.f}}, qk[2][2] = {{0.f, 0.f}, {0.f, 0.f}};
    if (jb <= ib && (NN > 1 || half == 0)) {
#pragma unroll 2
      for (int c = 16 * NH * half; c < 16 * NH * (half + 1); c += 4) {
        f32x4 ki[2], qi[2], kj[2], gi[2], gj[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          ki[e] = lds4(kS + (i0 + e) * LD + c);
          qi[e] = lds4(qS + (i0 + e) * LD + c);
          gi[e] = lds4(GS + (i0 + e) * LD + c);
          kj[e] = lds4(kS + (j0 + e) * LD + c);
          gj[e] = lds4(GS + (j0 + e) * LD + c);
        }
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
          for (int f = 0; f < 2; ++f) {
            const f32x4 w = kj[f] * exp2_neg(gi[e] - gj[f]);    // (above the diagonal: clamped, never used)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              kk[e][f] += ki[e][r] * w[r];
              qk[e][f] += qi[e][r] * w[r];
            }
          }
      }
    }
    float* X = XS + half * 2 * C * LC;
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
      for (int f = 0; f < 2; ++f) {
        X[(i0 + e) * LC + j0 + f] = kk[e][f];
        X[C * LC + (i0 + e) * LC + j0 + f] = qk[e][f];
      }
  }
  __syncthreads();
  // the halves meet; Akk goes on as beta_i Akk_ij (the threads hold their sums across a barrier: LS lies on XS)
  float lv[C * C / NT];
#pragma unroll
  for (int u = 0; u < C * C / NT; ++u) {
    const int i = (tid + NT * u) / C, j = (tid + NT * u) % C;
    const int o = i * LC + j;
    float w = 1.f;
    if (!CHANNEL) w = __builtin_amdgcn_exp2f(fminf(GS[i] - GS[j], 0.f));
    const bool stored = !(i < 16 && j >= 16);
    lv[u] = j < i ? bS[i] * w * (XS[o] + XS[2 * C * LC + o]) : 0.f;
    const float av = stored && j <= i ? w * (XS[C * LC + o] + XS[3 * C * LC + o]) : 0.f;
    if (i < nt) ws[i * wrow + C + j] = av;
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < C * C / NT; ++u) LS[(tid + NT * u) / C * LC + (tid + NT * u) % C] = lv[u];
  __syncthreads();
  // T = (I + L)^-1 diag(beta): thread c solves column c by forward substitution
  if (tid < C) {
    float t[C];
#pragma unroll
    for (int i = 0; i < C; ++i) {
      float s0 = i == tid ? bS[i] : 0.f, s1 = 0.f;
#pragma unroll
      for (int j = 0; j < i; ++j) {
        const float l = LS[i * LC + j];
        if (j & 1) s1 -= l * t[j];
        else s0 -= l * t[j];
      }
      t[i] = s0 + s1;
      TS[i * LC + tid] = t[i];
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < C * C / NT; ++u) {
    const int i = (tid + NT * u) / C, c = (tid + NT * u) % C;
    if (i < nt) ws[i * wrow + c] = TS[i * LC + c];
  }
}

// grid (P / (16 MW), heads, runs): waves 0 .. MW - 1 multiply (16 value columns each), as many more stage.  NN: 16-row tiles of
// the state (N <= 16 NN); NBUF: LDS stages (two where they fit).  With four and four a multiplying and a staging wave share a
// SIMD, and their times all but add up (68 us alone and 42 alone, 95 together); two and two have a SIMD each.
template <typename T, bool CHANNEL, int NN, int NBUF, int MW>
__global__ __launch_bounds__(128 * MW) void delta_chunk_scan_kernel(DeltaRuleArgs a) {
  extern __shared__ float lds[];
  constexpr int NT = 64 * MW;                  // staging threads
  constexpr int NP = 16 * NN;                  // padded key channels
  constexpr int LD = NP + 4;
  constexpr int TSTEP = NT / NP, EPT = C / TSTEP;      // a staging thread owns channel n of the tokens tt0, tt0 + TSTEP, ..
  constexpr int oQ = C * LD, oH = 2 * C * LD, oT = oH + NP * LC, oA = oT + C * LC, oD = oA + C * LC, STAGE = oD + NP;
  const int N = a.N, P = a.P;
  const int h = blockIdx.y, run = blockIdx.z;
  const int s0 = a.cu_q[run], s1 = a.cu_q[run + 1];
  if (s1 <= s0) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int chunks = (s1 - s0 + C - 1) / C;
  const int wc = ws_cols(CHANNEL, N);
  const long long wrow = (long long)a.H * wc;
  if (wave >= MW) {
    // ---- staging waves -----------------------------------------------------------------------------------------
    const int tid = threadIdx.x - NT, n = tid % NP, tt0 = tid / NP;
    const bool nin = n < N;
    const int gn = a.G * N;
    const float* k = a.k + (long long)(s0 + tt0) * gn + (h / a.hpg) * N + n;
    const float* q = a.q + (long long)(s0 + tt0) * gn + (h / a.hpg) * N + n;
    const float* wsh = a.ws + (long long)s0 * wrow + (long long)h * wc;
    const float* G = wsh + tt0 * wrow + 2 * C + (CHANNEL ? n : 0);
    const int mj = tid % C, mt = tid / C;      // the [C][C] matrices: column mj of the rows mt, mt + NT / C, ..
    const float* M = wsh + mt * wrow + mj;
    constexpr int MSTEP = NT / C, MPT = C / MSTEP;
    // a chunk waits in registers until its stage is free; at sizes where that does not fit (one stage), it is loaded a few
    // rows at a time instead
    constexpr bool AHEAD = NBUF == 2;
    constexpr int EB = AHEAD ? EPT : 4;
    float rk[EB], rq[EB], rg[EB], gl, rt[MPT], ra[MPT];
    auto fetch = [&](int c, int u0) {
      const int t0 = c * C, nt = min(C, s1 - s0 - t0);
      const float* kc = k + (long long)t0 * gn;
      const float* qc = q + (long long)t0 * gn;
      const float* Gc = G + t0 * wrow;
#pragma unroll
      for (int e = 0; e < EB; ++e) {
        const int u = u0 + e;
        const bool row = tt0 + TSTEP * u < nt;
        rk[e] = row && nin ? kc[(long long)TSTEP * u * gn] : 0.f;
        rq[e] = row && nin ? qc[(long long)TSTEP * u * gn] : 0.f;
        rg[e] = row && (nin || !CHANNEL) ? Gc[TSTEP * u * wrow] : 0.f;
      }
      if (u0) return;
      gl = nin || !CHANNEL ? wsh[(long long)(t0 + nt - 1) * wrow + 2 * C + (CHANNEL ? n : 0)] : 0.f;
      const float* Mc = M + t0 * wrow;
#pragma unroll
      for (int u = 0; u < MPT; ++u) {
        const bool in = mt + MSTEP * u < nt && mj < nt;
        rt[u] = in ? Mc[MSTEP * u * wrow] : 0.f;
        ra[u] = in ? Mc[MSTEP * u * wrow + C] : 0.f;
      }
    };
    auto put = [&](float* st, int u0) {
#pragma unroll
      for (int e = 0; e < EB; ++e) {
        const int tt = tt0 + TSTEP * (u0 + e);
        const float eg = __builtin_amdgcn_exp2f(rg[e]);
        st[tt * LD + n] = rk[e] * eg;
        st[oQ + tt * LD + n] = rq[e] * eg;
        st[oH + n * LC + tt] = rk[e] * __builtin_amdgcn_exp2f(fminf(gl - rg[e], 0.f));   // (rows past the run's end: k = 0)
      }
    };
    auto stash = [&](float* st, int c) {
      if (AHEAD) {
        put(st, 0);
      } else {
#pragma unroll 1
        for (int u0 = 0; u0 < EPT; u0 += EB) {
          fetch(c, u0);
          put(st, u0);
        }
      }
      if (tt0 == 0) st[oD + n] = __builtin_amdgcn_exp2f(gl);
#pragma unroll
      for (int u = 0; u < MPT; ++u) {
        st[oT + (mt + MSTEP * u) * LC + mj] = rt[u];
        st[oA + (mt + MSTEP * u) * LC + mj] = ra[u];
      }
    };
    if (AHEAD) fetch(0, 0);
    stash(lds, 0);
    if (AHEAD && chunks > 1) fetch(1, 0);
    __syncthreads();                           // chunk 0 is staged
    for (int c = 0; c < chunks; ++c) {
      if (NBUF == 1) __syncthreads();          // chunk c has been read
      if (c + 1 < chunks) {
        stash(lds + (NBUF == 2 ? ((c + 1) & 1) * STAGE : 0), c + 1);
        if (AHEAD && c + 2 < chunks) fetch(c + 2, 0);
      }
      __syncthreads();                         // chunk c + 1 is staged (two stages: and chunk c has been read)
    }
    return;
  }
  // ---- multiplying waves -----------------------------------------------------------------------------------------
  const int col = lane & 15, g = lane >> 4;
  const int p = blockIdx.x * 16 * MW + wave * 16 + col;
  const bool pin = p < P;
  const int pr = a.prev_row[s0];
  const int sv = a.save_slot[s1 - 1];
  const long long hp = (long long)a.H * P;
  const T* v = reinterpret_cast<const T*>(a.v) + (long long)s0 * hp + (long long)h * P;
  float* out = a.out + (long long)s0 * hp + (long long)h * P;
  const int vo = (int)sizeof(T) * (4 * g * (int)hp + p), oo = 4 * (4 * g * (int)hp + p);      // (launch_delta_rule bounds H P)
  float vn[8];
  auto fetch_v = [&](int c) {
    const __amdgpu_buffer_rsrc_t bv = chunk_rows(v + (long long)c * C * hp, sizeof(T) * hp, min(C, s1 - s0 - c * C), (int)sizeof(T) * P);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int off = pin ? vo + (16 * (i >> 2) + (i & 3)) * (int)(sizeof(T) * hp) : NO_PLACE;
      if constexpr (sizeof(T) == 2) vn[i] = (float)__builtin_bit_cast(bf16, __builtin_amdgcn_raw_buffer_load_b16(bv, off, 0, 0));
      else vn[i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(bv, off, 0, 0));
    }
  };
  f32x4 S[NN];
  const bool old = pr <= -2 && pin;
  const float* st0 = a.state + (old ? (long long)(-(pr + 2)) * a.state_stride + (long long)h * N * P + p : 0);
#pragma unroll
  for (int t = 0; t < NN; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int n = 16 * t + 4 * g + r;
      S[t][r] = old && n < N ? st0[(long long)n * P] : 0.f;
    }
  fetch_v(0);
  __syncthreads();                             // chunk 0 is staged
  for (int c = 0; c < chunks; ++c) {
    const float* st = lds + (NBUF == 2 ? (c & 1) * STAGE : 0);
    const float* Kt = st + col * LD + 4 * g;
    const float* Qt = st + oQ + col * LD + 4 * g;
    const float* Kh = st + oH + col * LC + 4 * g;
    const float* Tm = st + oT + col * LC + 4 * g;
    const float* Aq = st + oA + col * LC + 4 * g;
    const float* D = st + oD + 4 * g;
    // One multiplying wave a SIMD: every LDS read stands a step ahead of the products that take it (left to the compiler each
    // was waited for, more time than the products: 17 chunks of 8 heads x 128 x 256, 3 runs, 110 us; 88 this way).
    f32x4 x[2][4];
    auto load = [&](int t) {
      x[t & 1][0] = lds4(Kt + 16 * t), x[t & 1][1] = lds4(Kt + 16 * LD + 16 * t);
      x[t & 1][2] = lds4(Qt + 16 * t), x[t & 1][3] = lds4(Qt + 16 * LD + 16 * t);
    };
    load(0);
    const f32x4 V0 = {vn[0], vn[1], vn[2], vn[3]}, V1 = {vn[4], vn[5], vn[6], vn[7]};
    if (c + 1 < chunks) fetch_v(c + 1);
    f32x4 K0 = {0.f, 0.f, 0.f, 0.f}, K1 = K0, O0 = K0, O1 = K0, m[6], d[2], kh[2][2];
#pragma unroll
    for (int t = 0; t < NN; ++t) {
      if (t + 1 < NN) {
        load(t + 1);
      } else {
        m[0] = lds4(Tm), m[1] = lds4(Tm + 16 * LC), m[2] = lds4(Tm + 16 * LC + 16);
        m[3] = lds4(Aq), m[4] = lds4(Aq + 16 * LC), m[5] = lds4(Aq + 16 * LC + 16);
      }
      d[t & 1] = lds4(D + 16 * t);
      __builtin_amdgcn_sched_barrier(0);
      const f32x4(&y)[4] = x[t & 1];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        K0 = mfma4(y[0][r], S[t][r], K0);
        K1 = mfma4(y[1][r], S[t][r], K1);
        O0 = mfma4(y[2][r], S[t][r], O0);
        O1 = mfma4(y[3][r], S[t][r], O1);
      }
      if (t) S[t - 1] *= d[(t - 1) & 1];       // (its products are out)
      __builtin_amdgcn_sched_barrier(0);
    }
    S[NN - 1] *= d[(NN - 1) & 1];
    kh[0][0] = lds4(Kh), kh[0][1] = lds4(Kh + 16);
    __builtin_amdgcn_sched_barrier(0);
    const f32x4 R0 = V0 - K0, R1 = V1 - K1;
    f32x4 U0 = {0.f, 0.f, 0.f, 0.f}, U1 = U0;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      U0 = mfma4(m[0][r], R0[r], U0);
      U1 = mfma4(m[1][r], R0[r], U1);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) U1 = mfma4(m[2][r], R1[r], U1);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      O0 = mfma4(m[3][r], U0[r], O0);
      O1 = mfma4(m[4][r], U0[r], O1);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) O1 = mfma4(m[5][r], U1[r], O1);
#pragma unroll
    for (int t = 0; t < NN; ++t) {
      if (t + 1 < NN) kh[(t + 1) & 1][0] = lds4(Kh + 16 * (t + 1) * LC), kh[(t + 1) & 1][1] = lds4(Kh + 16 * (t + 1) * LC + 16);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int r = 0; r < 4; ++r) S[t] = mfma4(kh[t & 1][0][r], U0[r], S[t]);
#pragma unroll
      for (int r = 0; r < 4; ++r) S[t] = mfma4(kh[t & 1][1][r], U1[r], S[t]);
    }
    const int nt = min(C, s1 - s0 - c * C);
    const __amdgpu_buffer_rsrc_t bo = chunk_rows(out + (long long)c * C * hp, 4 * hp, nt, 4 * P);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(O0[r]), bo, pin ? oo + r * 4 * (int)hp : NO_PLACE, 0, 0);
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(O1[r]), bo, pin ? oo + (16 + r) * 4 * (int)hp : NO_PLACE, 0, 0);
    }
    if (NBUF == 1) __syncthreads();            // chunk c has been read
    __syncthreads();                           // chunk c + 1 is staged (two stages: and chunk c has been read)
  }
  if (sv >= 0 && pin) {
    float* so = a.state + (long long)sv * a.state_stride + (long long)h * N * P + p;
#pragma unroll
    for (int t = 0; t < NN; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int n = 16 * t + 4 * g + r;
        if (n < N) so[(long long)n * P] = S[t][r];
      }
  }
}

// The same walk on v_mfma_f32_16x16x32_bf16, for up to 128 key channels in the bf16 model: the fp32 products were what bound it (8 x
// 128 x 256: 224 of 32 cycles a chunk and wave).  State, keys, queries and corrections go in as three bf16 parts, six terms a
// product; T R and Aqk U, a tenth, stay fp32 products, their matrices straight from the scratch, a chunk ahead.
// A B operand's contraction index is 8 (lane / 16) + j and an accumulator's rows 4 (lane / 16) + r: with the contraction in the
// order j < 4: 4 g + j, else 16 + 4 g + j - 4, two accumulator tiles are a B operand.  Keys and queries lie in LDS in that order
// along a row, so that an A operand is one 16-byte read; the last product takes the keys' tokens as its contraction, by LDS transpose reads.
// One decay per head: rows and corrections are scaled behind the products (E = 2^(G_i), W = 2^(G_C - G_i)) and the keys serve both;
// decays per channel: k 2^G, q 2^G and k 2^(G_C - G) are staged.  NB: 32-channel blocks (N <= 32 NB, N a multiple of 8).
// What is left is the chain of a chunk, its products a third (4000 tokens in one run, us a chunk: 2.5; without the products of the
// state 1.8, without staging 2.4).  256 registers a lane: with more allowed the compiler keeps a part in AGPRs (348 -> 396).
// Prep and walk, fp32 products / parts, 8 x 128 x 256, us: one decay per head 3 runs of 510 91 / 62, 8 of 1000 222 / 162, one of
// 4000 529 / 355, of 100 35 / 26; per channel 108 / 87, 290 / 217, 567 / 420, 45 / 38.  Error against 64 bits no larger (rms of the outputs
// 2.2e-7 / 2.1e-7 at 510 rows, 3.8e-7 / 3.2e-7 with slow decays).
// An infinity or NaN of the state or a value ends as NaN in its own column from its chunk on, as with fp32 products, which meet 0 x
// infinity in T and Aqk.
template <bool CHANNEL, int NB, int MW>
__global__ __launch_bounds__(128 * MW, 4 / MW) void delta_chunk_parts_kernel(DeltaRuleArgs a, int unit) {
  constexpr int ST = 64 * MW;                            // staging threads
  constexpr int NP = 32 * NB, LQ = NP + 8;               // LQ: bf16 pitch of a [C][NP] matrix
  constexpr int PART = C * LQ, oQ = 3 * PART, oH = CHANNEL ? 6 * PART : 0, MATS = CHANNEL ? 3 : 2;
  constexpr int FS = CHANNEL ? NP : 2 * C + 4;           // floats: 2^(G_C) per channel, or E | W | 2^(G_C)
  constexpr int STAGE = MATS * 3 * PART * 2 + FS * 4;    // bytes
  static_assert(STAGE % 16 == 0 && 2 * STAGE <= 160 * 1024, "two stages");
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int N = a.N, P = a.P;
  const WalkPlace at = walk_place(unit);
  const int slab = at.slab, h = at.head, run = at.run;
  const int s0 = a.cu_q[run], s1 = a.cu_q[run + 1];
  if (s1 <= s0) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int chunks = (s1 - s0 + C - 1) / C;
  const int wc = ws_cols(CHANNEL, N);
  const long long wrow = (long long)a.H * wc;
  const float* ws = a.ws + (long long)s0 * wrow + (long long)h * wc;
  if (wave >= MW) {
    // ---- staging waves: thread (token tt0, 8 channels from c8), TSTEP tokens apart -----------------------------------
    constexpr int GR = NP / 8, TSTEP = ST / GR, PASS = (C + TSTEP - 1) / TSTEP;
    const int tid = threadIdx.x - ST, c8 = 8 * (tid % GR), tt0 = tid / GR;
    const bool nin = c8 < N && tt0 < C;
    const int gn = a.G * N;
    const float* k = a.k + (long long)s0 * gn + (h / a.hpg) * N;
    const float* q = a.q + (long long)s0 * gn + (h / a.hpg) * N;
    const int at = 32 * (c8 / 32) + 8 * (c8 % 16 / 4) + 4 * (c8 % 32 / 16);      // the 4 from c8; the 4 behind them 8 on
    int ko[PASS], go[PASS];
#pragma unroll
    for (int u = 0; u < PASS; ++u) {
      const int tt = tt0 + TSTEP * u;
      ko[u] = nin ? 4 * (tt * gn + c8) : NO_PLACE;
      go[u] = nin ? 4 * (tt * (int)wrow + 2 * C + c8) : NO_PLACE;
    }
    f32x4 rk[PASS][2], rq[PASS][2], rg[CHANNEL ? PASS : 1][2], gl[2];
    float g1 = 0.f, glast = 0.f;
    auto fetch = [&](int c) {
      const int t0 = c * C, nt = min(C, s1 - s0 - t0);
      const __amdgpu_buffer_rsrc_t bk = chunk_rows(k + (long long)t0 * gn, 4LL * gn, nt, 4 * N);
      const __amdgpu_buffer_rsrc_t bq = chunk_rows(q + (long long)t0 * gn, 4LL * gn, nt, 4 * N);
      const __amdgpu_buffer_rsrc_t bg = chunk_rows(ws + t0 * wrow, 4 * wrow, nt, 4 * wc);
#pragma unroll
      for (int u = 0; u < PASS; ++u)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          rk[u][i] = row16f(bk, ko[u] + (nin ? 16 * i : 0));
          rq[u][i] = row16f(bq, ko[u] + (nin ? 16 * i : 0));
          if constexpr (CHANNEL) rg[u][i] = row16f(bg, go[u] + (nin ? 16 * i : 0));
        }
      const float* last = ws + (t0 + nt - 1) * wrow + 2 * C;
      if constexpr (CHANNEL) {
#pragma unroll
        for (int i = 0; i < 2; ++i) gl[i] = nin ? lds4(last + c8 + 4 * i) : f32x4{0.f, 0.f, 0.f, 0.f};
      } else {
        g1 = tid < C ? __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(bg, 4 * (tid * (int)wrow + 2 * C), 0, 0)) : 0.f;
        glast = last[0];
      }
    };
    auto put = [&](bf16* m, int tt, f32x4 lo, f32x4 hi, auto wide) {
      const Parts x = split<decltype(wide)::value>(lo, hi);
      auto half = [&](int part, bf16x8 v) {
        Pack8 w;
        w.v = v;
        bf16* to = m + part * PART + tt * LQ + at;
        *reinterpret_cast<uint2*>(to) = make_uint2(w.u.x, w.u.y);
        *reinterpret_cast<uint2*>(to + 8) = make_uint2(w.u.z, w.u.w);
      };
      half(0, x.h), half(1, x.m), half(2, x.l);
    };
    auto stash = [&](int c) {
      bf16* st = reinterpret_cast<bf16*>(smem + (c & 1) * STAGE);
      float* fs = reinterpret_cast<float*>(st + MATS * 3 * PART);
#pragma unroll
      for (int u = 0; u < PASS; ++u) {
        const int tt = tt0 + TSTEP * u;
        if (tt >= C) break;
        if constexpr (CHANNEL) {
          f32x4 e[2], w[2];
#pragma unroll
          for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              e[i][r] = __builtin_amdgcn_exp2f(rg[u][i][r]);
              w[i][r] = __builtin_amdgcn_exp2f(fminf(gl[i][r] - rg[u][i][r], 0.f));      // (rows past the run's end: k = 0)
            }
          put(st, tt, rk[u][0] * e[0], rk[u][1] * e[1], std::false_type());
          put(st + oQ, tt, rq[u][0] * e[0], rq[u][1] * e[1], std::true_type());
          put(st + oH, tt, rk[u][0] * w[0], rk[u][1] * w[1], std::false_type());
        } else {
          put(st, tt, rk[u][0], rk[u][1], std::false_type());
          put(st + oQ, tt, rq[u][0], rq[u][1], std::true_type());
        }
      }
      if constexpr (CHANNEL) {
        if (tt0 == 0)
#pragma unroll
          for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) fs[c8 + 4 * i + r] = __builtin_amdgcn_exp2f(gl[i][r]);
      } else if (tid < C) {
        fs[tid] = __builtin_amdgcn_exp2f(g1);
        fs[C + tid] = __builtin_amdgcn_exp2f(fminf(glast - g1, 0.f));
        if (tid == 0) fs[2 * C] = __builtin_amdgcn_exp2f(glast);
      }
    };
    fetch(0);
    stash(0);
    if (chunks > 1) fetch(1);
    __syncthreads();                           // chunk 0 is staged
    for (int c = 0; c < chunks; ++c) {
      if (c + 1 < chunks) {
        stash(c + 1);
        if (c + 2 < chunks) fetch(c + 2);
      }
      __syncthreads();                         // chunk c + 1 is staged, chunk c has been read
    }
    return;
  }
  // ---- multiplying waves -----------------------------------------------------------------------------------------
  const int col = lane & 15, g = lane >> 4;
  const int p = slab * 16 * MW + wave * 16 + col;
  const bool pin = p < P;
  const int pr = a.prev_row[s0];
  const int sv = a.save_slot[s1 - 1];
  const long long hp = (long long)a.H * P;
  const bf16* v = reinterpret_cast<const bf16*>(a.v) + (long long)s0 * hp + (long long)h * P;
  float* out = a.out + (long long)s0 * hp + (long long)h * P;
  const int vo = 2 * (4 * g * (int)hp + p), oo = 4 * (4 * g * (int)hp + p);      // (launch_delta_rule bounds H P)
  float vn[8];
  auto fetch_v = [&](int c) {
    const __amdgpu_buffer_rsrc_t bv = chunk_rows(v + (long long)c * C * hp, 2 * hp, min(C, s1 - s0 - c * C), 2 * P);
#pragma unroll
    for (int i = 0; i < 8; ++i)
      vn[i] = (float)__builtin_bit_cast(bf16, __builtin_amdgcn_raw_buffer_load_b16(bv, pin ? vo + (16 * (i >> 2) + (i & 3)) * 2 * (int)hp : NO_PLACE, 0, 0));
  };
  // T and Aqk: rows col, 16 + col; a row's 4 from 4 g, 16 + 4 g (rows past the run's end and what lies above the diagonal: 0)
  f32x4 m[6];
  auto fetch_m = [&](int c) {
    const __amdgpu_buffer_rsrc_t bm = chunk_rows(ws + (long long)c * C * wrow, 4 * wrow, min(C, s1 - s0 - c * C), 8 * C);
    const int o = 4 * (col * (int)wrow + 4 * g), o16 = o + 64 * (int)wrow;
    m[0] = row16f(bm, o), m[1] = row16f(bm, o16), m[2] = row16f(bm, o16 + 64);
    m[3] = row16f(bm, o + 4 * C), m[4] = row16f(bm, o16 + 4 * C), m[5] = row16f(bm, o16 + 4 * C + 64);
  };
  f32x4 S[2 * NB];
  const bool old = pr <= -2 && pin;
  const float* st0 = a.state + (old ? (long long)(-(pr + 2)) * a.state_stride + (long long)h * N * P + p : 0);
#pragma unroll
  for (int t = 0; t < 2 * NB; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int n = 16 * t + 4 * g + r;
      S[t][r] = old && n < N ? st0[(long long)n * P] : 0.f;
    }
  fetch_v(0);
  fetch_m(0);
  __syncthreads();                             // chunk 0 is staged
  for (int c = 0; c < chunks; ++c) {
    const bf16* st = reinterpret_cast<const bf16*>(smem + (c & 1) * STAGE);
    const float* fs = reinterpret_cast<const float*>(st + MATS * 3 * PART);
    const bf16* Kr = st + col * LQ + 8 * g;
    // (one multiplying wave a SIMD: LDS reads stand a step ahead of the products that take them)
    bf16x8 f[2][2][3][2];                      // of a block's turn: keys, queries; parts; row tiles
    auto load = [&](int b) {
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int part = 0; part < 3; ++part)
#pragma unroll
          for (int i = 0; i < 2; ++i)
            f[b & 1][x][part][i] = *reinterpret_cast<const bf16x8*>(Kr + x * oQ + part * PART + 16 * i * LQ + 32 * b);
    };
    load(0);
    const f32x4 V0 = {vn[0], vn[1], vn[2], vn[3]}, V1 = {vn[4], vn[5], vn[6], vn[7]};
    if (c + 1 < chunks) fetch_v(c + 1);
    f32x4 e[2], w[2];                          // one decay per head: of the rows 4 g + r, 16 + 4 g + r
    float dh = 1.f;
    if constexpr (!CHANNEL) {
#pragma unroll
      for (int i = 0; i < 2; ++i) e[i] = lds4(fs + 16 * i + 4 * g), w[i] = lds4(fs + C + 16 * i + 4 * g);
      dh = fs[2 * C];
    }
    f32x4 K[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}}, O[2] = {K[0], K[0]};
    Parts s = split<true>(S[0], S[1]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      if (b + 1 < NB) load(b + 1);
      f32x4 d[2];
      if constexpr (CHANNEL) d[0] = lds4(fs + 32 * b + 4 * g), d[1] = lds4(fs + 32 * b + 16 + 4 * g);
      Parts next = s;
      if (b + 1 < NB) next = split<true>(S[2 * b + 2], S[2 * b + 3]);
#pragma unroll
      for (int term = 0; term < 6; ++term) {   // the smallest terms first
        constexpr int mine[6] = {0, 2, 1, 1, 0, 0};
        const bf16x8 sp = term == 0 ? s.l : term == 2 || term == 4 ? s.m : s.h;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          K[i] = mfma16(f[b & 1][0][mine[term]][i], sp, K[i]);
          O[i] = mfma16(f[b & 1][1][mine[term]][i], sp, O[i]);
        }
      }
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        if constexpr (CHANNEL) S[2 * b + i] *= d[i];
        else S[2 * b + i] *= dh;
      }
      s = next;
      __builtin_amdgcn_sched_barrier(0);
    }
    // keys of the last product: 16 channels of the tokens 4 g .. + 3 and 16 + 4 g .. + 3
    const char* Ht = reinterpret_cast<const char*>(st + oH + (4 * g + (col >> 2)) * LQ) + 16 * (col & 3);
    bf16x8 kh[2][3];
    auto load_h = [&](int t) {
#pragma unroll
      for (int part = 0; part < 3; ++part) {
        const char* at = Ht + part * PART * 2 + 64 * (t >> 1) + 8 * (t & 1);
        Pack8 x;
        const uint2 lo = read_tr(at), hi = read_tr(at + 32 * LQ);
        x.u = make_uint4(lo.x, lo.y, hi.x, hi.y);
        kh[t & 1][part] = x.v;
      }
    };
    load_h(0);
    if constexpr (!CHANNEL) {
#pragma unroll
      for (int i = 0; i < 2; ++i) K[i] *= e[i], O[i] *= e[i];
    }
    const f32x4 R0 = V0 - K[0], R1 = V1 - K[1];
    f32x4 U0 = {0.f, 0.f, 0.f, 0.f}, U1 = U0;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      U0 = mfma4(m[0][r], R0[r], U0);
      U1 = mfma4(m[1][r], R0[r], U1);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) U1 = mfma4(m[2][r], R1[r], U1);
    const Parts u = CHANNEL ? split<true>(U0, U1) : split<true>(U0 * w[0], U1 * w[1]);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      O[0] = mfma4(m[3][r], U0[r], O[0]);
      O[1] = mfma4(m[4][r], U0[r], O[1]);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) O[1] = mfma4(m[5][r], U1[r], O[1]);
    if (c + 1 < chunks) fetch_m(c + 1);
#pragma unroll
    for (int t = 0; t < 2 * NB; ++t) {
      if (t + 1 < 2 * NB) load_h(t + 1);
      __builtin_amdgcn_sched_barrier(0);
      const bf16x8(&x)[3] = kh[t & 1];
      S[t] = mfma16(x[0], u.l, S[t]);
      S[t] = mfma16(x[2], u.h, S[t]);
      S[t] = mfma16(x[1], u.m, S[t]);
      S[t] = mfma16(x[1], u.h, S[t]);
      S[t] = mfma16(x[0], u.m, S[t]);
      S[t] = mfma16(x[0], u.h, S[t]);
    }
    const int nt = min(C, s1 - s0 - c * C);
    const __amdgpu_buffer_rsrc_t bo = chunk_rows(out + (long long)c * C * hp, 4 * hp, nt, 4 * P);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(O[i][r]), bo, pin ? oo + (16 * i + r) * 4 * (int)hp : NO_PLACE, 0, 0);
    __syncthreads();                           // chunk c + 1 is staged, chunk c has been read
  }
  if (sv >= 0 && pin) {
    float* so = a.state + (long long)sv * a.state_stride + (long long)h * N * P + p;
#pragma unroll
    for (int t = 0; t < 2 * NB; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int n = 16 * t + 4 * g + r;
        if (n < N) so[(long long)n * P] = S[t][r];
      }
  }
}

void raise_lds(const void* f) { hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024); }

template <typename T, bool CHANNEL, int NPL, int CH, int SLICES>
void launch_serial(const DeltaRuleArgs& a, hipStream_t s) {
  const int cols = (64 / SLICES) * (NT / 64);
  const int lrow = SLICES * (NPL + 4);
  const size_t lds = (size_t)2 * (2 * CH * lrow + (CHANNEL ? CH * lrow : CH) + CH) * sizeof(float);
  static bool raised = false;
  if (!raised && lds > 64 * 1024) raise_lds(reinterpret_cast<const void*>(&delta_scan_kernel<T, CHANNEL, NPL, CH, SLICES>));
  raised = true;
  delta_scan_kernel<T, CHANNEL, NPL, CH, SLICES><<<dim3((a.P + cols - 1) / cols, a.H, a.runs), NT, lds, s>>>(a);
}

template <typename T, bool CHANNEL>
void serial(const DeltaRuleArgs& a, hipStream_t s) {
  const int need = (a.N + 3) / 4;
  if (a.T == a.runs) {        // one token per run: the state's traffic is the launch
    if (need <= 4) launch_serial<T, CHANNEL, 4, 1, 4>(a, s);
    else if (need <= 8) launch_serial<T, CHANNEL, 8, 1, 4>(a, s);
    else if (need <= 16) launch_serial<T, CHANNEL, 16, 1, 4>(a, s);
    else if (need <= 32) launch_serial<T, CHANNEL, 32, 1, 4>(a, s);
    else launch_serial<T, CHANNEL, 64, 1, 4>(a, s);
    return;
  }
  if (need <= 4) launch_serial<T, CHANNEL, 4, 16, 4>(a, s);
  else if (need <= 8) launch_serial<T, CHANNEL, 8, 16, 4>(a, s);
  else if (need <= 16) launch_serial<T, CHANNEL, 8, 16, 8>(a, s);
  else if (need <= 32) launch_serial<T, CHANNEL, 16, 16, 8>(a, s);
  else launch_serial<T, CHANNEL, 32, 8, 8>(a, s);      // N <= 256 (checked by the op layer)
}

template <typename T, bool CHANNEL, int NN, int MW>
void launch_scan(const DeltaRuleArgs& a, hipStream_t s) {
  constexpr int NP = 16 * NN, LD = NP + 4;
  constexpr int STAGE = 2 * C * LD + NP * LC + 2 * C * LC + NP;
  constexpr int NBUF = 2 * STAGE * (int)sizeof(float) <= 160 * 1024 ? 2 : 1;
  static const bool raised = (raise_lds(reinterpret_cast<const void*>(&delta_chunk_scan_kernel<T, CHANNEL, NN, NBUF, MW>)), true);
  (void)raised;
  const dim3 grid((a.P + 16 * MW - 1) / (16 * MW), a.H, a.runs);
  delta_chunk_scan_kernel<T, CHANNEL, NN, NBUF, MW><<<grid, 128 * MW, (size_t)NBUF * STAGE * sizeof(float), s>>>(a);
}

template <bool CHANNEL, int NB, int MW>
void launch_parts(const DeltaRuleArgs& a, hipStream_t s) {
  constexpr int lds = 2 * ((CHANNEL ? 9 : 6) * C * (32 * NB + 8) * 2 + (CHANNEL ? 32 * NB : 2 * C + 4) * 4);
  static const bool raised = (raise_lds(reinterpret_cast<const void*>(&delta_chunk_parts_kernel<CHANNEL, NB, MW>)), true);
  (void)raised;
  const int slabs = (a.P + 16 * MW - 1) / (16 * MW);
  const long long total = (long long)slabs * a.H * a.runs;
  delta_chunk_parts_kernel<CHANNEL, NB, MW><<<dim3(slabs, a.H, a.runs), 128 * MW, lds, s>>>(a, walk_unit(total, slabs));
}

template <typename T, bool CHANNEL, int NN>
void launch_chunks(const DeltaRuleArgs& a, hipStream_t s) {
  constexpr int LD = 16 * NN + 4;
  const size_t prep = (size_t)((CHANNEL ? 3 : 2) * C * LD + 4 * C * LC + 2 * C) * sizeof(float);
  static const bool raised = (raise_lds(reinterpret_cast<const void*>(&delta_chunk_prep_kernel<CHANNEL, NN>)), true);
  (void)raised;
  delta_chunk_prep_kernel<CHANNEL, NN><<<dim3(2 * a.ntiles, a.H), NT, prep, s>>>(a);
  // 32 columns a workgroup while those are at most one a CU (256) and runs are long enough that the first chunk's staging, which
  // half as many waves do, is not what counts; else 64 (8 heads x 128 x 256, us with 32 / with 64 columns: 3 runs of 512 tokens
  // 76 / 88, 5 runs 146 / 87, one of 4000 498 / 639, 3 runs of 200 40.7 / 40.3, of 60 17.6 / 14.9; in parts, prep included, 5 runs of
  // 512 109 / 71, 8 of 20 25 / 20, 3 of 200 37.6 / 38.1)
  const bool narrow = NN <= 8 && (long long)((a.P + 31) / 32) * a.H * a.runs <= 256 && a.T >= 8LL * C * a.runs;
  if constexpr (sizeof(T) == 2 && NN <= 8) {
    const auto a16 = [](const void* p) { return (uintptr_t)p % 16 == 0; };
    // (whole groups of 8 channels in 16-byte loads; a chunk's rows at 32-bit offsets)
    if (a.N % 8 == 0 && a16(a.q) && a16(a.k) && a16(a.ws) && (long long)a.H * (2 * C + a.N) <= 1 << 22 && (long long)a.G * a.N <= 1 << 22)
      return narrow ? launch_parts<CHANNEL, (NN + 1) / 2, 2>(a, s) : launch_parts<CHANNEL, (NN + 1) / 2, 4>(a, s);
  }
  if constexpr (NN <= 8) {
    if (narrow) return launch_scan<T, CHANNEL, NN, 2>(a, s);
  }
  launch_scan<T, CHANNEL, NN, 4>(a, s);
}

template <typename T, bool CHANNEL>
void chunked(const DeltaRuleArgs& a, hipStream_t s) {
  const int nn = (a.N + 15) / 16;
  if (nn <= 1) launch_chunks<T, CHANNEL, 1>(a, s);
  else if (nn <= 2) launch_chunks<T, CHANNEL, 2>(a, s);
  else if (nn <= 4) launch_chunks<T, CHANNEL, 4>(a, s);
  else if (nn <= 8) launch_chunks<T, CHANNEL, 8>(a, s);
  else launch_chunks<T, CHANNEL, 16>(a, s);
}

}  // namespace

int launch_delta_rule(const DeltaRuleArgs& a, int channel, int f32, int impl, hipStream_t s) {
  if (a.runs <= 0 || a.T <= 0) return 1;
  const bool chunk = impl == 0 && a.tiles && a.ntiles > 0 && a.ws && a.cu_q && (long long)a.H * a.P <= 1 << 23;      // (32-bit places in a chunk)
  if (f32) {
    if (chunk) channel ? chunked<float, true>(a, s) : chunked<float, false>(a, s);
    else channel ? serial<float, true>(a, s) : serial<float, false>(a, s);
  } else {
    if (chunk) channel ? chunked<bf16, true>(a, s) : chunked<bf16, false>(a, s);
    else channel ? serial<bf16, true>(a, s) : serial<bf16, false>(a, s);
  }
  return chunk ? 0 : 1;
}
