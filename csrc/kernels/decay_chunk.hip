// Chunked form of the decaying recurrences of decay_scan.hip for prompt steps in bf16:
//
//     S_t = diag(a_t) S_(t-1) + b_t k_t v_t^T,     o_t = q_scale S_t^T q_t (+ skip_h v_t)          S [N x P] fp32
//
// mode 0: a per key channel, b = 1 (gated linear attention); mode 1: a per head, b the step size (state-space layers).
// Token by token a state costs 4 N P vector operations a token on the serial path (8100 tokens in 8 prompts: 1656 us at
// 8 heads x 128 x 256, 1345 us at 64 x 128 x 64).  With chunks of C = 32 tokens, G_i the running sum of log2 a inside the
// chunk and S_0 the state in front of it,
//     o_i = (q_i 2^(G_i))^T S_0 + sum_{j <= i} A_ij v_j,     A_ij = b_j sum_n q_in k_jn 2^(G_in - G_jn)
//     S_C = 2^(G_C) S_0 + sum_j (k_j 2^(G_C - G_j) b_j) v_j^T                 (every exponent <= 0: nothing overflows)
// is matrix products; a run's chunks are walked in order, few long runs in segments at once (a segment's state from 0 and its decays
// first, then each segment from the states in front of it).
//
// Precision: q, k and v are bf16, so they are exact operands of v_mfma_f32_16x16x32_bf16, which accumulates in fp32.  An
// fp32 operand (the state, a scaled vector, the scores) is used as the sum of three bf16 parts (bf16_parts.h).
//
// Work split: grid (P / 64, heads, runs or segments), waves of 16 value columns with all of N or half of it: the state stays in accumulator registers
// for the whole run.  An accumulator's rows are 4 (lane / 16) + r, a B operand's contraction index is 8 (lane / 16) + j; with
// the contraction taken in the order j < 4: 4 g + j, else 16 + 4 g + j - 4, two accumulator tiles ARE a B operand, and the A
// operand is read in the same order (two 8-byte LDS reads).  The same holds for the values and, computed transposed, for the
// scores.  The next chunk's rows are loaded while the current one is multiplied (two LDS stages, one barrier a chunk).
// One or two waves a SIMD: what a chunk costs is its vector instructions and every wait that nothing covers.  8100 tokens in 8
// runs, us: 8 heads x 128 x 256 300 -> 228, 64 x 128 x 64 258 -> 200 with pairs rounded at once, rows through a buffer's range,
// k turned by LDS transpose reads instead of 2-byte stores (a third of the time in bank conflicts) and reads a step ahead.
#include "attn_tiles.h"
#include "bf16_parts.h"
#include "hybrid_launchers.h"
#include "walk_places.h"

#include <algorithm>

namespace {

constexpr int NT = 256;
constexpr int C = 32;             // tokens per chunk
constexpr int LT = C + 4;         // LDS pitch of a [.][C] matrix
constexpr float LOG2E = 1.4426950408889634f;

SYM_DEV float softplus_exact(float v) { return fmaxf(v, 0.f) + log1pf(expf(-fabsf(v))); }
// A token's log2 decay, no lower than -256: 2^-256 is 0 in fp32 like everything below, and the chunk's sums stay finite where
// a token forgets all (a pre-activation or bias of -inf, an infinite rate), so differences behind it are no inf - inf.  NaN
// stays NaN.
template <typename F>
SYM_DEV F log_decay(F v) { return v < (F)-256 ? (F)-256 : v; }
SYM_DEV float pow2(float v) { return __builtin_amdgcn_exp2f(v); }
SYM_DEV f32x4 mfma4(float x, float y, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(x, y, c, 0, 0, 0); }
SYM_DEV f32x4 lds4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }

SYM_DEV bf16 row2(__amdgpu_buffer_rsrc_t r, int off) {
  return __builtin_bit_cast(bf16, __builtin_amdgcn_raw_buffer_load_b16(r, off, 0, 0));
}

// inclusive sums over lanes 0 .. 31, in the vector unit
template <int CTRL>
SYM_DEV double lanes_before(double v) {      // (lanes without one: 0)
  const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
  const unsigned int lo = __builtin_amdgcn_update_dpp(0, (int)u, CTRL, 0xf, 0xf, false);
  const unsigned int hi = __builtin_amdgcn_update_dpp(0, (int)(u >> 32), CTRL, 0xf, 0xf, false);
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}
SYM_DEV double prefix32(double v, int lane) {
  v += lanes_before<0x111>(v);               // row_shr 1, 2, 4, 8
  v += lanes_before<0x112>(v);
  v += lanes_before<0x114>(v);
  v += lanes_before<0x118>(v);
  const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
  const unsigned int lo = __builtin_amdgcn_readlane((int)u, 15), hi = __builtin_amdgcn_readlane((int)(u >> 32), 15);
  return lane < 16 ? v : v + __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// mode 0's scratch, a block per chunk and head: the bf16 parts of q_i 2^(G_i) | those of k_i 2^(G_C - G_i), each 3 [C][NP] | A fp32
// [C][C] | 2^(G_C) fp32 [NP], as the walk keeps it in LDS: 16-byte pieces of a row are exchanged by its number (row_turn, score_turn), so that
// reads along the rows and LDS transpose reads meet no bank twice; rows and channels past the end are 0.  Bytes, in whole KB.  The parts
// are formed here once, not by every slab's workgroup in the walk, which only copies (8 heads x 128 x 256, walk, us: 8 runs of 612 to
// 1546 tokens 195 -> 178, one of 7900 870 -> 782; the launch that forms them stays at 81).
constexpr int chunk_block(int NP) { return (6 * C * NP * 2 + C * C * 4 + NP * 4 + 1023) / 1024 * 1024; }
inline int padded(int N) { return N <= 32 ? 32 : N <= 64 ? 64 : 128; }
template <int NP>
SYM_DEV int row_turn(int row) { return (((row & 7) << 1) | ((row >> 3) & 1)) & (NP / 8 - 1); }
SYM_DEV int score_turn(int row) { return (row >> 1) & 7; }
// a run's first block: runs need no more than a block past their rows' share
SYM_DEV long long first_block(int s0, int run) { return (s0 >> 5) + run; }
__host__ __device__ inline int ws_cols(int N) { return C + 2 * N; }      // (floats a row and head that a caller's scratch has at least)

// ---- mode 0: decays and scores A of every chunk, grid (64-row tiles x 2 chunks, heads) ----------------------------------
// G is held as a pair of floats: what counts are its differences, and once a few tokens of a chunk forget hard, G is in the
// hundreds and a float's differences of the tokens behind them keep few digits (a tenth of the tokens at -100 with tau 1: 9e-6
// of the output's norm from G alone, the token walk 1e-7).  Inside the four 8 x 8 tiles on the diagonal the exponents of
// differences are taken per (i, j, channel) on the vector unit; the tiles below them factor at the end of the columns,
// 2^(G_i - G_15) 2^(G_15 - G_j) for rows 16 .. (G_7 and G_23 for rows 8 .. of each half), both exponents <= 0, and are matrix
// products.  Bound by the vector unit, the per-pair exponents before all: 8100 tokens, 8 heads of 128 channels 140 -> 90 us from
// 16 x 16 diagonal tiles.
template <int NN>
__global__ __launch_bounds__(NT) void decay_chunk_prep_kernel(DecayScanArgs a) {
  constexpr int NP = 16 * NN, LD = NP + 4;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  float* kS = reinterpret_cast<float*>(smem);  // [C][LD]
  float* qS = kS + C * LD;                     // [C][LD]
  float* GS = qS + C * LD;                     // [C][LD] G: high part
  float* LS = GS + C * LD;                     // [C][LD] low part
  float* XS = kS;                              // [4][C][LT] partial scores, when the others have been read
  static_assert(LT <= LD, "the partial scores fit");
  const int N = a.N, h = blockIdx.y, tile = blockIdx.x >> 1, sub = blockIdx.x & 1;
  const int seq = a.tiles[2 * tile], off = a.tiles[2 * tile + 1];
  const int q0 = a.cu_q[seq], qlen = a.cu_q[seq + 1] - q0;
  if (off >= qlen) return;                     // padding tile
  const int nt = min(C, qlen - off - C * sub);
  if (nt <= 0) return;
  const long long r0 = q0 + off + C * sub;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const bf16* q = reinterpret_cast<const bf16*>(a.q) + r0 * a.ldq + (h / a.hpg) * N;
  const bf16* k = reinterpret_cast<const bf16*>(a.k) + r0 * a.ldk + (h / a.hpg) * N;
  const bf16* dz = reinterpret_cast<const bf16*>(a.dz) + r0 * a.ldd + (long long)h * N;
  const float* db = a.dbias + (long long)h * N;
  const float scale = -LOG2E / a.tau;
  // every load is in flight before the first is waited for
  constexpr int EL = C * NP / NT;
  static_assert(C * NP % NT == 0 && NT % 2 == 0, "whole elements a thread");
  bf16 kv[EL], qv[EL], zv[EL];
  float bv[EL];
#pragma unroll
  for (int e = 0; e < EL; ++e) {
    const int i = tid + NT * e, tt = min(i / NP, nt - 1), n = min(i % NP, N - 1);
    zv[e] = dz[tt * a.ldd + n];
    bv[e] = db[n];
    kv[e] = k[tt * a.ldk + n];
    qv[e] = q[tt * a.ldq + n];
  }
#pragma unroll
  for (int e = 0; e < EL; ++e) {
    const int i = tid + NT * e, tt = i / NP, n = i % NP;
    const bool in = tt < nt && n < N;
    GS[tt * LD + n] = in ? log_decay(scale * softplus_exact(-((float)zv[e] + bv[e]))) : 0.f;
    kS[tt * LD + n] = in ? (float)kv[e] : 0.f;
    qS[tt * LD + n] = in ? (float)qv[e] : 0.f;
  }
  __syncthreads();
  char* const ws = reinterpret_cast<char*>(a.ws) + ((first_block(q0, seq) + off / C + sub) * a.H + h) * chunk_block(NP);
  if (tid < NP) {
    double g = 0.;
#pragma unroll 8
    for (int tt = 0; tt < C; ++tt) {
      g += (double)GS[tt * LD + tid];
      const float hi = (float)g;
      GS[tt * LD + tid] = hi;
      LS[tt * LD + tid] = (float)(g - (double)hi);
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < (C * NP / 8 + NT - 1) / NT; ++u) {      // (G stands still past the run's end, so the last row's is G_C)
    const int i = tid + NT * u;
    if (C * NP / 8 % NT && i >= C * NP / 8) break;
    const int tt = i / (NP / 8), ch = i % (NP / 8), at = tt * LD + 8 * ch, end = (C - 1) * LD + 8 * ch;
    f32x4 x[2], y[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const f32x4 gi = lds4(GS + at + 4 * e), li = lds4(LS + at + 4 * e), gc = lds4(GS + end + 4 * e), lc = lds4(LS + end + 4 * e);
      const f32x4 qi = lds4(qS + at + 4 * e), ki = lds4(kS + at + 4 * e);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        x[e][r] = qi[r] * pow2(gi[r]);
        y[e][r] = ki[r] * pow2((gc[r] - gi[r]) + (lc[r] - li[r]));
      }
    }
    const Parts sx = split(x[0], x[1]), sy = split(y[0], y[1]);
    bf16* to = reinterpret_cast<bf16*>(ws) + tt * NP + 8 * (ch ^ row_turn<NP>(tt));
    *reinterpret_cast<bf16x8*>(to) = sx.h;
    *reinterpret_cast<bf16x8*>(to + C * NP) = sx.m;
    *reinterpret_cast<bf16x8*>(to + 2 * C * NP) = sx.l;
    *reinterpret_cast<bf16x8*>(to + 3 * C * NP) = sy.h;
    *reinterpret_cast<bf16x8*>(to + 4 * C * NP) = sy.m;
    *reinterpret_cast<bf16x8*>(to + 5 * C * NP) = sy.l;
  }
  float* const scores = reinterpret_cast<float*>(ws + 6 * C * NP * 2);
  if (tid < NP) scores[C * C + tid] = tid < N ? pow2(GS[(C - 1) * LD + tid]) : 0.f;
  const int col = lane & 15, g = lane >> 4;
  // rows 16 .., columns .. 15: the waves take the channel tiles in turn
  f32x4 d = {0.f, 0.f, 0.f, 0.f};
  for (int t = wave; t < NN; t += 4) {
    const int c = 16 * t + 4 * g;
    const f32x4 mh = lds4(GS + 15 * LD + c), gi = lds4(GS + (16 + col) * LD + c), gj = lds4(GS + col * LD + c);
    const f32x4 ml = lds4(LS + 15 * LD + c), li = lds4(LS + (16 + col) * LD + c), lj = lds4(LS + col * LD + c);
    const f32x4 qi = lds4(qS + (16 + col) * LD + c), kj = lds4(kS + col * LD + c);
#pragma unroll
    for (int r = 0; r < 4; ++r)
      d = mfma4(qi[r] * pow2((gi[r] - mh[r]) + (li[r] - ml[r])), kj[r] * pow2((mh[r] - gj[r]) + (ml[r] - lj[r])), d);
  }
  // rows 8 .. of each half, columns .. 7 of it: the same product, both halves in the diagonal blocks of one tile
  f32x4 d8 = {0.f, 0.f, 0.f, 0.f};
  const int low = (col & 7) + 16 * (col >> 3), mid = 16 * (col >> 3) + 7;
  for (int t = wave; t < NN; t += 4) {
    const int c = 16 * t + 4 * g;
    const f32x4 mh = lds4(GS + mid * LD + c), gi = lds4(GS + (low + 8) * LD + c), gj = lds4(GS + low * LD + c);
    const f32x4 ml = lds4(LS + mid * LD + c), li = lds4(LS + (low + 8) * LD + c), lj = lds4(LS + low * LD + c);
    const f32x4 qi = lds4(qS + (low + 8) * LD + c), kj = lds4(kS + low * LD + c);
#pragma unroll
    for (int r = 0; r < 4; ++r)
      d8 = mfma4(qi[r] * pow2((gi[r] - mh[r]) + (li[r] - ml[r])), kj[r] * pow2((mh[r] - gj[r]) + (ml[r] - lj[r])), d8);
  }
  // the four 8 x 8 on the diagonal: a 2 x 2 block of (i, j) per lane, the waves take a quarter of the channels each
  constexpr int NQ = NP / 4;
  const int ib = (lane >> 2) & 3, jb = lane & 3;
  const int i0 = 8 * g + 2 * ib, j0 = 8 * g + 2 * jb;
  float s[2][2] = {{0.f, 0.f}, {0.f, 0.f}};
  if (jb <= ib) {
#pragma unroll 2
    for (int c = NQ * wave; c < NQ * (wave + 1); c += 4) {
      f32x4 qi[2], gi[2], li[2], kj[2], gj[2], lj[2];
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        qi[e] = lds4(qS + (i0 + e) * LD + c);
        gi[e] = lds4(GS + (i0 + e) * LD + c);
        li[e] = lds4(LS + (i0 + e) * LD + c);
        kj[e] = lds4(kS + (j0 + e) * LD + c);
        gj[e] = lds4(GS + (j0 + e) * LD + c);
        lj[e] = lds4(LS + (j0 + e) * LD + c);
      }
#pragma unroll
      for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int f = 0; f < 2; ++f)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            s[e][f] += qi[e][r] * (kj[f][r] * pow2((gi[e][r] - gj[f][r]) + (li[e][r] - lj[f][r])));
    }
  }
  __syncthreads();                             // (the rows have been read: their place takes the partial scores)
#pragma unroll
  for (int r = 0; r < 4; ++r) XS[(wave * C + 16 + 4 * g + r) * LT + col] = d[r];
  if ((col >> 3) == (g >> 1))
#pragma unroll
    for (int r = 0; r < 4; ++r) XS[(wave * C + 16 * (g >> 1) + 8 + 4 * (g & 1) + r) * LT + low] = d8[r];
#pragma unroll
  for (int e = 0; e < 2; ++e)
#pragma unroll
    for (int f = 0; f < 2; ++f) XS[(wave * C + i0 + e) * LT + j0 + f] = s[e][f];
  __syncthreads();
#pragma unroll
  for (int u = 0; u < C * C / NT; ++u) {
    const int i = (tid + NT * u) / C, j = (tid + NT * u) % C;
    const float* x = XS + i * LT + j;
    const float v = j <= i ? (x[0] + x[C * LT]) + (x[2 * C * LT] + x[3 * C * LT]) : 0.f;
    scores[i * C + 4 * ((j >> 2) ^ score_turn(i)) + (j & 3)] = i < nt ? v : 0.f;
  }
}

// ---- segments of runs ------------------------------------------------------------------------------------------------------
// Runs too few to give every CU a workgroup (mode 1: two) are cut: as many segments as there are workgroups for, none longer than it
// must be, the same number of chunks in each of a run's but for one.  All workgroups find the same from the same lengths.
constexpr int SEGMENTS_MAX = 16;      // (and fewer runs than that: a row of 16 lanes holds them)

// Segments that a step's walks have workgroups for; 0: whole runs.  The walk of the states is 2 / 5 of a walk, and a launch and the
// states in front of a segment cost about 4 chunks (mode 1, with two workgroups a CU: 8).  Walks, us, whole / in segments: 8 heads x 128 x
// 256, one run of 130 tokens 19 / 19.5, of 300 33 / 20.5, of 7900 782 / 183, 2 of 300 36 / 27, 4 of 175 30 / 32, 4 of 500 74 / 66,
// 6 of 1000 140 / 165; 64 x 128 x 64, one of 130 21 / 25, of 300 36 / 30, of 7900 776 / 218, 2 of 300 37 / 36, 2 of 1000 105 / 68,
// 3 of 267 37 / 39, 4 of 500 75 / 77.
int walk_segments(int mode, long long T, long long runs, long long H, long long P) {
  const long long per = H * ((P + 63) / 64);
  const long long n = std::min<long long>(SEGMENTS_MAX, (mode == 0 ? 256 : 512) / per);
  if (mode > 1 || runs < 1 || n < 2 * runs) return 0;
  return T >= (mode == 0 ? 96 * runs + 384 * runs * runs / n : 128 * runs + 768 * runs * runs / n) ? (int)n : 0;
}

struct Segment {
  int run, from, to;            // chunks of the run
  int place, of, item0;         // its number among the run's, how many these are, the run's first item
};

SYM_DEV int row_total(int v) {      // over a row of 16 lanes
  v += __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x141, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x140, 0xf, 0xf, true);
  return __builtin_amdgcn_readfirstlane(v);
}

SYM_DEV bool find_segment(const int* cu_q, int runs, int items, int item, Segment& s) {
  const int lane = threadIdx.x & 15;
  const int n = lane < runs ? (max(0, cu_q[lane + 1] - cu_q[lane]) + C - 1) / C : 0;
  auto pieces = [&](int len) { return (int)((unsigned)(n + len - 1) / (unsigned)len); };
  int lo = max(2, (row_total(n) + items - 1) / items), hi = lo;      // the shortest that are no more than `items`
  while (row_total(pieces(hi)) > items) hi *= 2;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (row_total(pieces(mid)) > items) lo = mid + 1;
    else hi = mid;
  }
  const int k = pieces(hi);
  int upto = k;
  upto += __builtin_amdgcn_update_dpp(0, upto, 0x111, 0xf, 0xf, false);
  upto += __builtin_amdgcn_update_dpp(0, upto, 0x112, 0xf, 0xf, false);
  upto += __builtin_amdgcn_update_dpp(0, upto, 0x114, 0xf, 0xf, false);
  upto += __builtin_amdgcn_update_dpp(0, upto, 0x118, 0xf, 0xf, false);
  const int run = __builtin_popcountll(__ballot(upto <= item) & 0xffff);
  if (run >= runs) return false;
  const int chunks = __builtin_amdgcn_readlane(n, run);
  s.run = run, s.of = __builtin_amdgcn_readlane(k, run);
  s.item0 = __builtin_amdgcn_readlane(upto, run) - s.of;
  s.place = item - s.item0;
  s.from = chunks * s.place / s.of, s.to = chunks * (s.place + 1) / s.of;
  return true;
}

// bytes of LDS of a walk: two stages, mode 1's sums, the parts that waves hand over
constexpr int scan_lds(int mode, int NB, int HV) {
  const int NP = 32 * NB;
  return 2 * (mode == 0 ? chunk_block(NP) : 2 * C * (NP + 8) * 2) + (mode == 1 ? 8 * HV * 3 * C * 4 : 0) + (HV - 1) * 16 * 4 * HV * 128;
}

// ---- the walk ------------------------------------------------------------------------------------------------------------
// NB: 32-channel blocks of the state (N <= 32 NB).  HV: 2 where two waves share 16 columns, each with half of N: the parts of the
// state, which are formed anew for every chunk, and the staging are most of the vector work, and with a wave a SIMD (mode 0's LDS
// leaves one workgroup a CU) nothing covers the waits.  Each of the two finishes one of the chunk's row tiles and hands its part of the
// other over in LDS; it is read behind the chunk's barrier and stored a chunk later (8 heads x 128 x 256, us: 8 runs of 1012 tokens 210
// -> 197, 2 of 750 101 -> 92; 64 x 128 x 64, 2 of 750, 84.5 -> 80.5).  256 registers a lane: with more allowed the
// compiler keeps a part in AGPRs, which was slower.
// WALK: WHOLE runs, grid z their number; or, where the runs are few (walk_segments), segments of them: the STATES that all segments but
// a run's last add up from 0 (the first: from the run's state), with their channels' decays, then the SEGMENTS themselves, each from the
// states in front of it.
enum { WHOLE, STATES, SEGMENTS };

template <int MODE, int NB, int HV, int WALK>
__global__ __launch_bounds__(NT * HV, 2) void decay_chunk_scan_kernel(DecayScanArgs a, int unit) {
  constexpr int TH = NT * HV, NWV = 4 * HV, NBW = NB / HV, TI = 2 / HV;
  constexpr int NP = 32 * NB, LQ = MODE == 0 ? NP : NP + 8;   // LQ: bf16 pitch of a [C][NP] matrix
  constexpr int PL = MODE == 0 ? 3 : 1;                 // bf16 parts of the staged vectors
  constexpr int oK = PL * C * LQ, oF = oK + PL * C * LQ;      // in bf16: q | k, a part behind the other
  constexpr int STAGE = MODE == 0 ? chunk_block(NP) : oF * 2; // bytes; behind oF in mode 0: A | 2^(G_C)
  constexpr int SUMS = MODE == 1 ? 2 * NWV * 3 * C : 0; // floats, mode 1: G | its low part | b of 2 NWV chunks
  static_assert(STAGE % 16 == 0, "stages start at multiples of 16 bytes");
  static_assert(2 * STAGE + SUMS * 4 + (HV - 1) * 16 * NWV * 128 == scan_lds(MODE, NB, HV), "the launch's LDS");
  extern __shared__ __attribute__((aligned(16))) char smem[];
  float* const sums = reinterpret_cast<float*>(smem + 2 * STAGE);
  f32x4* const given = reinterpret_cast<f32x4*>(smem + 2 * STAGE + SUMS * 4);      // [2][NWV][64]
  const int N = a.N, P = a.P;
  const WalkPlace at = walk_place(unit);
  const int slab = at.slab, h = at.head;
  Segment seg{at.run, 0, 0, 0, 1, 0};
  if constexpr (WALK != WHOLE)
    if (!find_segment(a.cu_q, a.runs, a.segments, at.run, seg)) return;
  const int run = seg.run, q0 = a.cu_q[run];
  const int s0 = WALK == WHOLE ? q0 : q0 + C * seg.from, s1 = WALK == WHOLE ? a.cu_q[run + 1] : min(a.cu_q[run + 1], q0 + C * seg.to);
  if (s1 <= s0 || (WALK == STATES && seg.place + 1 == seg.of)) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), col = lane & 15, g = lane >> 4;
  const int hf = HV == 2 ? wave >> 2 : 0, ch0 = 32 * NBW * hf;      // the wave's channels
  const int p = slab * 64 + (wave & 3) * 16 + col;
  const bool pin = p < P;
  const int chunks = (s1 - s0 + C - 1) / C;
  const int pr = a.prev_row[q0], sv = a.save_slot[s1 - 1];      // (a save_slot in the middle of a run is no one's)
  const bf16* q = reinterpret_cast<const bf16*>(a.q) + s0 * a.ldq + (h / a.hpg) * N;
  const bf16* k = reinterpret_cast<const bf16*>(a.k) + s0 * a.ldk + (h / a.hpg) * N;
  const bf16* v = reinterpret_cast<const bf16*>(a.v) + s0 * a.ldv + (long long)h * P;
  const bf16* dt = reinterpret_cast<const bf16*>(a.dz) + s0 * a.ldd + h;          // mode 1
  const char* block = MODE == 0 ? reinterpret_cast<const char*>(a.ws) + ((first_block(q0, run) + seg.from) * a.H + h) * STAGE : nullptr;
  float* out = a.out + ((long long)s0 * a.H + h) * P;
  const long long orow = (long long)a.H * P;
  const int ldv = (int)a.ldv * 2, ldo = (int)orow * 4;                            // (decay_chunk_takes bounds them)
  const int vo = pin ? 4 * g * ldv + 2 * p : NO_PLACE, oo = pin ? (4 * g + 16 * hf) * ldo + 4 * p : NO_PLACE;

  // staging, mode 0: the chunk's block as it lies, by direct loads; mode 1: thread (token tt, 8 channels from c8), PASS tokens apart
  constexpr int GR = NP / 8, TSTEP = TH / GR, PASS = (C + TSTEP - 1) / TSTEP;
  const int c8 = 8 * (tid % GR), tt0 = tid / GR;
  const bool nin = c8 < N && tt0 < C;                   // (N is a multiple of 8)
  Pack8 rq[PASS], rk[PASS];
  bf16 vn[8];
  int qo[PASS], ko[PASS];
#pragma unroll
  for (int u = 0; u < PASS; ++u) {
    const int tt = tt0 + TSTEP * u;
    qo[u] = nin ? tt * (int)a.ldq * 2 + 2 * c8 : NO_PLACE;
    ko[u] = nin ? tt * (int)a.ldk * 2 + 2 * c8 : NO_PLACE;
  }
  const unsigned int lds0 = lds_address(smem) + wave * 1024;
  auto fetch = [&](int c) {
    if constexpr (MODE == 0) {
      const u32x4 from = buffer_words(block + (long long)c * a.H * STAGE, STAGE);
#pragma unroll
      for (int i = 0; i < (STAGE / 1024 + NWV - 1) / NWV; ++i)
        if (NWV * i + wave >= (WALK == STATES ? oK * 2 / 1024 : 0) && NWV * i + wave < STAGE / 1024)
          direct_buffer_load16(from, 16 * lane, 1024 * (NWV * i + wave), lds0 + (c & 1) * STAGE + 1024 * NWV * i);
    } else {
      const int t0 = c * C, nt = min(C, s1 - s0 - t0);
      const __amdgpu_buffer_rsrc_t bq = chunk_rows(q + t0 * a.ldq, a.ldq * 2, nt, N * 2);
      const __amdgpu_buffer_rsrc_t bk = chunk_rows(k + t0 * a.ldk, a.ldk * 2, nt, N * 2);
#pragma unroll
      for (int u = 0; u < PASS; ++u)
        if (WALK != STATES) rq[u].u = row16(bq, qo[u]);
#pragma unroll
      for (int u = 0; u < PASS; ++u) rk[u].u = row16(bk, ko[u]);
    }
  };
  auto fetch_v = [&](int c) {
    const __amdgpu_buffer_rsrc_t bv = chunk_rows(v + (long long)c * C * a.ldv, a.ldv * 2, min(C, s1 - s0 - c * C), P * 2);
#pragma unroll
    for (int i = 0; i < 8; ++i) vn[i] = row2(bv, vo + (pin ? (16 * (i >> 2) + (i & 3)) * ldv : 0));
  };
  // Mode 1: a chunk's step sizes and the running sum of its log decays, by one wave; the waves do those of the NWV chunks ahead
  // together (one wave a chunk, the others waited for it: 64 x 128 x 64, 8 runs of 1012 tokens, 190 -> 186 us).  The sum is a pair of floats: with step sizes that forget in a few tokens
  // it grows to hundreds, and the differences of neighbours, which are what counts, would keep few of its digits.
  const float rate2 = MODE == 1 ? expf(a.rate[h]) * LOG2E : 0.f, dbias = MODE == 1 ? a.dbias[h] : 0.f;
  float rdt = 0.f;
  auto fetch_step = [&](int c) { rdt = lane < s1 - s0 - c * C && lane < C ? (float)dt[(long long)(c * C + lane) * a.ldd] + dbias : 0.f; };
  auto sum_steps = [&](int c) {
    if (c >= chunks) return;
    const int nt = min(C, s1 - s0 - c * C);
    const float b = lane < nt ? softplus_exact(rdt) : 0.f;
    double s = lane < nt ? log_decay(-(double)rate2 * b) : 0.0;
    s = prefix32(s, lane);
    float* fs = sums + (c & (2 * NWV - 1)) * 3 * C;
    if (lane < C) {
      fs[lane] = (float)s;
      fs[C + lane] = (float)(s - (double)(float)s);
      fs[2 * C + lane] = b;
    }
  };
  auto stash = [&](int c) {
    if constexpr (MODE == 0) {
      wait_direct_loads();
    } else {
      bf16* st = reinterpret_cast<bf16*>(smem + (c & 1) * STAGE);
#pragma unroll
      for (int u = 0; u < PASS; ++u) {
        const int tt = tt0 + TSTEP * u;
        if (tt >= C) break;
        if (WALK != STATES) *reinterpret_cast<uint4*>(st + tt * LQ + c8) = rq[u].u;
        *reinterpret_cast<uint4*>(st + oK + tt * LQ + c8) = rk[u].u;
      }
    }
  };
  // mode 0's places in the block, bytes: of q's 8-byte pieces, of k's for the transpose reads, of A's quads
  int qx[NBW][2], kx[2 * NBW], ax[2];
  if constexpr (MODE == 0) {
    const int kr = 4 * g + (col >> 2);
#pragma unroll
    for (int t = 0; t < NBW; ++t)
#pragma unroll
      for (int i = 0; i < 2; ++i) qx[t][i] = col * NP * 2 + 16 * ((ch0 / 8 + 4 * t + 2 * i + (g >> 1)) ^ row_turn<NP>(col)) + 8 * (g & 1);
#pragma unroll
    for (int t = 0; t < 2 * NBW; ++t) kx[t] = kr * NP * 2 + 16 * ((ch0 / 8 + 2 * t + ((col & 3) >> 1)) ^ row_turn<NP>(kr)) + 8 * (col & 1);
#pragma unroll
    for (int j = 0; j < 2; ++j) ax[j] = col * C * 4 + 16 * ((4 * j + g) ^ score_turn(col));
  }

  fetch(0);
  fetch_v(0);
  f32x4 S[2 * NBW];
  // a segment's states (and a split run's own, in the place of its last segment, which hands on none: a run's state may be saved
  // where it came from) in the order of the accumulators, and behind them all their decays
  const int slabs = (P + 63) / 64;
  auto state_of = [&](int item) {
    return reinterpret_cast<f32x4*>(a.seg) + ((((long long)item * a.H + h) * slabs + slab) * 8 * NB + wave * 2 * NBW) * 64 + lane;
  };
  float* const decays = a.seg + (long long)a.segments * a.H * slabs * 64 * NP + (long long)h * NP;      // + item H NP
  const bool own = WALK == WHOLE || (WALK == STATES ? seg.place == 0 : seg.of == 1);
  const bool old = own && pr <= -2 && pin;
  const float* st0 = a.state + (old ? (long long)(-(pr + 2)) * a.state_stride + (long long)h * N * P + p : 0);
#pragma unroll
  for (int t = 0; t < 2 * NBW; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int n = ch0 + 16 * t + 4 * g + r;
      S[t][r] = old && n < N ? st0[(long long)n * P] : 0.f;
    }
  if constexpr (WALK == STATES) {
    if (own)
#pragma unroll
      for (int t = 0; t < 2 * NBW; ++t) state_of(seg.item0 + seg.of - 1)[64 * t] = S[t];
  }
  if constexpr (WALK == SEGMENTS) {
    if (!own) {
      // four segments' at once: one wait for each four
      constexpr int AT = 4;
      const int parts = max(seg.place, 1), first = seg.place ? seg.item0 : seg.item0 + seg.of - 1;
      for (int i0 = 0; i0 < parts; i0 += AT) {
        f32x4 u[AT][2 * NBW], d[AT][MODE == 0 ? 2 * NBW : 1];
#pragma unroll
        for (int i = 0; i < AT; ++i) {
          const int item = first + min(i0 + i, parts - 1);
#pragma unroll
          for (int t = 0; t < 2 * NBW; ++t) {
            u[i][t] = state_of(item)[64 * t];
            if (MODE == 0) d[i][MODE == 0 ? t : 0] = lds4(decays + (long long)item * a.H * NP + ch0 + 16 * t + 4 * g);
          }
          if (MODE == 1) d[i][0][0] = decays[(long long)item * a.H * NP];
        }
#pragma unroll
        for (int i = 0; i < AT; ++i)
          if (i0 + i < parts) {
#pragma unroll
            for (int t = 0; t < 2 * NBW; ++t)
              S[t] = i0 + i == 0 ? u[i][t] : (MODE == 0 ? S[t] * d[i][MODE == 0 ? t : 0] : S[t] * d[i][0][0]) + u[i][t];
          }
      }
    }
  }
  f32x4 gone[MODE == 0 ? 2 * NBW : 1];      // STATES: the segment's decays
#pragma unroll
  for (int t = 0; t < (MODE == 0 ? 2 * NBW : 1); ++t) gone[t] = f32x4{1.f, 1.f, 1.f, 1.f};
  const float skip = a.skip ? a.skip[h] : 0.f;
  if constexpr (MODE == 1) {
    fetch_step(wave);
    sum_steps(wave);
  }
  stash(0);
  __syncthreads();
  f32x4 mine = {0.f, 0.f, 0.f, 0.f};                    // HV 2: the wave's row tile of the chunk before, without the other's part
  auto store_tile = [&](int c, int i, f32x4 y) {        // row tile i past the wave's first
    const __amdgpu_buffer_rsrc_t bo = chunk_rows(out + (long long)c * C * orow, orow * 4, min(C, s1 - s0 - c * C), P * 4);
#pragma unroll
    for (int r = 0; r < 4; ++r)
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(y[r]), bo, oo + (pin ? (16 * i + r) * ldo : 0), 0, 0);
  };
  for (int c = 0; c < chunks; ++c) {
    Pack8 V;
#pragma unroll
    for (int i = 0; i < 8; ++i) V.h[i] = vn[i];
    const bool more = c + 1 < chunks;
    if (more) {
      fetch(c + 1);
      fetch_v(c + 1);
    }
    if constexpr (MODE == 1)
      if (c % NWV == 0 && c + NWV < chunks) fetch_step(c + NWV + wave);
    __builtin_amdgcn_sched_barrier(0);                  // the next chunk's loads in flight ahead of this one's products
    if constexpr (HV == 2 && WALK != STATES)
      if (c) store_tile(c - 1, 0, mine + a.q_scale * given[(((c - 1) & 1) * NWV + wave) * 64 + lane]);
    const bf16* st = reinterpret_cast<const bf16*>(smem + (c & 1) * STAGE);
    const float* fs = MODE == 0 ? reinterpret_cast<const float*>(st + oF) : sums + (c & (2 * NWV - 1)) * 3 * C;
    const bf16* Qr = st + col * LQ + 4 * g + ch0;
    f32x4 O[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    f32x4 A[TI][2];                                     // scores of row tile i, columns 4 g + r and 16 + 4 g + r
    f32x4 gj[2], lj[2], bj[2];
    // A wave or two a SIMD: LDS reads stand a step ahead of the products that take them, and the parts of the next state tiles
    // are formed between products (left to the compiler, every read was waited for: half of the walk).
    bf16x8 qf[2][PL][2];
    auto load_q = [&](int t) {
#pragma unroll
      for (int part = 0; part < PL; ++part)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          if constexpr (MODE == 0) {
            const char* from = reinterpret_cast<const char*>(st) + (part * C + 16 * i) * NP * 2;
            Pack8 f;
            const uint2 x = *reinterpret_cast<const uint2*>(from + qx[t][0]), y = *reinterpret_cast<const uint2*>(from + qx[t][1]);
            f.u = make_uint4(x.x, x.y, y.x, y.y);
            qf[t & 1][part][i] = f.v;
          } else {
            qf[t & 1][part][i] = pair4(Qr + (part * C + 16 * i) * LQ + 32 * t);
          }
        }
    };
    if constexpr (WALK != STATES) {
      load_q(0);
      if (NBW > 1) load_q(1);
    }
    if constexpr (MODE == 0 && WALK != STATES) {
#pragma unroll
      for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) A[i][j] = *reinterpret_cast<const f32x4*>(reinterpret_cast<const char*>(fs + 16 * (i + hf) * C) + ax[j]);
    }
    if constexpr (MODE == 1) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        gj[j] = lds4(fs + 16 * j + 4 * g);
        lj[j] = lds4(fs + C + 16 * j + 4 * g);
        bj[j] = lds4(fs + 2 * C + 16 * j + 4 * g);
      }
    }
    if constexpr (WALK != STATES) {
      Parts s = split<true>(S[0], S[1]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < NBW; ++t) {
        Parts next = s;
        if (t + 1 < NBW) next = split<true>(S[2 * t + 2], S[2 * t + 3]);
#pragma unroll
        for (int term = 0; term < (MODE == 0 ? 6 : 3); ++term)
#pragma unroll
          for (int i = 0; i < 2; ++i) {                   // the smallest terms first
            const auto& f = qf[t & 1];
            if constexpr (MODE == 0) {
              constexpr int qp[6] = {0, 2, 1, 1, 0, 0};
              const bf16x8 sp = term == 0 ? s.l : term == 2 || term == 4 ? s.m : s.h;
              O[i] = mfma16(f[qp[term]][i], sp, O[i]);
            } else {
              O[i] = mfma16(f[0][i], term == 0 ? s.l : term == 1 ? s.m : s.h, O[i]);
            }
          }
        if (t + 2 < NBW) load_q(t + 2);
        s = next;
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    // The product of scores and values runs over the scores' masked half as well, where 0 x inf would reach the rows in front
    // of a value that is not finite: it is left out of the product, and its column is NaN from its token on.
    Pack8 W = V;
    int bad = C;
    const uint4 e = V.u;
    const auto ones = [](unsigned x) { return (x & 0x7f807f80u) + 0x00800080u; };     // bits 15, 31: an exponent of all ones
    if (WALK != STATES && __any(((ones(e.x) | ones(e.y) | ones(e.z) | ones(e.w)) & 0x80008000u) != 0)) {
#pragma unroll
      for (int i = 7; i >= 0; --i)
        if (!__builtin_isfinite((float)V.h[i])) {
          W.h[i] = (bf16)0.f;
          bad = 16 * (i >> 2) + 4 * g + (i & 3);
        }
      bad = min(bad, __shfl_xor(bad, 16, 64));
      bad = min(bad, __shfl_xor(bad, 32, 64));
    }
    if constexpr (MODE == 1 && WALK != STATES) {
      bf16x8 kf[2][NB], qn[TI][NB];
      float gi[TI], li[TI];
#pragma unroll
      for (int i = 0; i < TI; ++i) {
        gi[i] = fs[16 * (i + hf) + col], li[i] = fs[C + 16 * (i + hf) + col];
#pragma unroll
        for (int t = 0; t < NB; ++t)
          qn[i][t] = *reinterpret_cast<const bf16x8*>(st + (16 * (i + hf) + col) * LQ + 8 * g + 32 * t);
      }
      const bool second = HV == 1 || hf;                // (the first row tile sees the first columns only)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int t = 0; t < NB; ++t)
          if (i == 0 || second) kf[i][t] = *reinterpret_cast<const bf16x8*>(st + oK + (16 * i + col) * LQ + 8 * g + 32 * t);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) O[j][r] *= pow2(gj[j][r]);      // (rows 4 g + r of O too)
#pragma unroll
      for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) A[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int t = 0; t < NB; ++t) {
#pragma unroll
        for (int i = 0; i < TI; ++i) A[i][0] = mfma16(kf[0][t], qn[i][t], A[i][0]);
        if (second) A[TI - 1][1] = mfma16(kf[1][t], qn[TI - 1][t], A[TI - 1][1]);
      }
#pragma unroll
      for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < (HV == 1 ? i + 1 : 2); ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float w = pow2((gi[i] - gj[j][r]) + (li[i] - lj[j][r])) * bj[j][r];
            float y = A[i][j][r] * w;
            asm volatile("" : "+v"(y));                 // (a select, no branch around the exponential)
            A[i][j][r] = j < i + hf || (j == i + hf && 4 * g + r <= col) ? y : 0.f;
          }
    }
    // k^T as an A operand in the accumulators' order: 16 channels of 4 tokens at 4 g, 4 at 16 + 4 g (LDS transpose reads)
    const char* Kt = reinterpret_cast<const char*>(st + oK + (4 * g + (col >> 2)) * LQ + ch0) + 8 * (col & 3);
    auto turned = [&](int part, int t) {
      Pack8 f;
      const char* from = MODE == 0 ? reinterpret_cast<const char*>(st + oK) + kx[t] : Kt + 32 * t;
      const uint2 x = read_tr(from + part * C * LQ * 2), y = read_tr(from + (part * C + 16) * LQ * 2);
      f.u = make_uint4(x.x, x.y, y.x, y.y);
      return f.v;
    };
    bf16x8 kt[2 * NBW];                                 // of the part at hand
#pragma unroll
    for (int t = 0; t < 2 * NBW; ++t) kt[t] = turned(PL - 1, t);
    f32x4 dec[MODE == 0 ? 2 * NBW : 1];
    if constexpr (MODE == 0) {
#pragma unroll
      for (int t = 0; t < 2 * NBW; ++t) dec[t] = lds4(fs + C * C + ch0 + 16 * t + 4 * g);
    }
    if constexpr (HV == 2 && WALK != STATES) {
      given[((c & 1) * NWV + (wave ^ 4)) * 64 + lane] = hf ? O[0] : O[1];
      if (hf) O[0] = O[1];
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (WALK != STATES) {
#pragma unroll
      for (int i = 0; i < TI; ++i) {
        const Parts u = split(A[i][0], A[i][1]);
        O[i] = mfma16(u.l, W.v, O[i]);
        O[i] = mfma16(u.m, W.v, O[i]);
        O[i] = mfma16(u.h, W.v, O[i]);
      }
      if (bad < C) {
#pragma unroll
        for (int i = 0; i < TI; ++i)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (16 * (i + hf) + 4 * g + r >= bad) O[i][r] = __builtin_nanf("");
      }
#pragma unroll
      for (int i = 0; i < TI; ++i) {
        f32x4 y;
#pragma unroll
        for (int r = 0; r < 4; ++r) y[r] = a.q_scale * O[i][r] + skip * (float)(HV == 2 && hf ? V.h[4 + r] : V.h[4 * i + r]);
        if constexpr (HV == 2) mine = y;
        else store_tile(c, i, y);
      }
    }
    if constexpr (MODE == 0) {
#pragma unroll
      for (int t = 0; t < 2 * NBW; ++t) {
        S[t] *= dec[t];
        if (WALK == STATES) gone[t] *= dec[t];
      }
#pragma unroll
      for (int part = 2; part >= 0; --part) {
        bf16x8 nk[2 * NBW];
#pragma unroll
        for (int t = 0; t < 2 * NBW; ++t)
          if (part) nk[t] = turned(part - 1, t);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < 2 * NBW; ++t) S[t] = mfma16(kt[t], V.v, S[t]);
#pragma unroll
        for (int t = 0; t < 2 * NBW; ++t)
          if (part) kt[t] = nk[t];
      }
    } else {
      const float gc = fs[C - 1], lc = fs[2 * C - 1], d = pow2(gc);     // (G stands still past the run's end)
      if (WALK == STATES) gone[0] *= d;
      f32x4 w[2];
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) w[j][r] = pow2((gc - gj[j][r]) + (lc - lj[j][r])) * bj[j][r] * (float)V.h[4 * j + r];
      const Parts u = split(w[0], w[1]);
#pragma unroll
      for (int t = 0; t < 2 * NBW; ++t) S[t] = mfma16(kt[t], u.l, S[t] * d);
#pragma unroll
      for (int t = 0; t < 2 * NBW; ++t) S[t] = mfma16(kt[t], u.m, S[t]);
#pragma unroll
      for (int t = 0; t < 2 * NBW; ++t) S[t] = mfma16(kt[t], u.h, S[t]);
      if (c % NWV == NWV / 2 && c + NWV / 2 < chunks) sum_steps(c + NWV / 2 + wave);
    }
    if (more) stash(c + 1);
    __syncthreads();                                    // chunk c + 1 is staged, chunk c has been read
  }
  if constexpr (WALK == STATES) {
    const int item = seg.item0 + seg.place;
#pragma unroll
    for (int t = 0; t < 2 * NBW; ++t) state_of(item)[64 * t] = S[t];
    if (slab == 0 && (wave & 3) == 0 && col == 0) {
      float* to = decays + (long long)item * a.H * NP;
#pragma unroll
      for (int t = 0; t < (MODE == 0 ? 2 * NBW : 1); ++t)
        if (MODE == 0) *reinterpret_cast<f32x4*>(to + ch0 + 16 * t + 4 * g) = gone[t];
        else if (lane == 0 && hf == 0) to[0] = gone[0][0];
    }
    return;
  }
  if constexpr (HV == 2) store_tile(chunks - 1, 0, mine + a.q_scale * given[(((chunks - 1) & 1) * NWV + wave) * 64 + lane]);
  if (sv >= 0 && pin && (WALK == WHOLE || seg.place + 1 == seg.of)) {
    float* so = a.state + (long long)sv * a.state_stride + (long long)h * N * P + p;
#pragma unroll
    for (int t = 0; t < 2 * NBW; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int n = ch0 + 16 * t + 4 * g + r;
        if (n < N) so[(long long)n * P] = S[t][r];
      }
  }
}

template <int MODE, int NB, int HV, int WALK>
void launch_walk(const DecayScanArgs& a, hipStream_t s) {
  constexpr int lds = scan_lds(MODE, NB, HV);
  static const bool raised = [] {
    if (lds > 64 * 1024)
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&decay_chunk_scan_kernel<MODE, NB, HV, WALK>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    return true;
  }();
  (void)raised;
  const int slabs = (a.P + 63) / 64, z = WALK == WHOLE ? a.runs : a.segments;
  decay_chunk_scan_kernel<MODE, NB, HV, WALK><<<dim3(slabs, a.H, z), NT * HV, lds, s>>>(a, walk_unit((long long)slabs * a.H * z, slabs));
}

template <int MODE, int NB, int HV>
void launch_scan(const DecayScanArgs& a, hipStream_t s) {
  if (a.segments > a.runs) {
    launch_walk<MODE, NB, HV, STATES>(a, s);
    launch_walk<MODE, NB, HV, SEGMENTS>(a, s);
  } else {
    launch_walk<MODE, NB, HV, WHOLE>(a, s);
  }
}

template <int MODE, int NB>
void launch_chunks(const DecayScanArgs& a, hipStream_t s) {
  if constexpr (MODE == 0) {
    constexpr int prep = 4 * C * (32 * NB + 4) * 4;
    static const bool raised = [] {
      if (prep > 64 * 1024)
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&decay_chunk_prep_kernel<2 * NB>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, prep);
      return true;
    }();
    (void)raised;
    decay_chunk_prep_kernel<2 * NB><<<dim3(2 * a.ntiles, a.H), NT, prep, s>>>(a);
  }
  if constexpr (NB > 1) {
    // eight waves a workgroup where LDS (mode 0) or their number (at most one a CU) leaves one of them on a CU
    if (MODE == 0 || (long long)((a.P + 63) / 64) * a.H * std::max(a.runs, a.segments) <= 256) return launch_scan<MODE, NB, 2>(a, s);
  }
  if constexpr (MODE == 1 || NB == 1) launch_scan<MODE, NB, 1>(a, s);
}

template <int MODE>
void launch_mode(const DecayScanArgs& a, hipStream_t s) {
  if (a.N <= 32) launch_chunks<MODE, 1>(a, s);
  else if (a.N <= 64) launch_chunks<MODE, 2>(a, s);
  else launch_chunks<MODE, 4>(a, s);
}

}  // namespace

// Is the call one the chunked form takes?  bf16 prompt steps of at least 8 tokens a run, 48 in mode 0 with its second launch
// (below, a chunk's fixed cost is more than the walk: 3 runs of 28 tokens, mode 0 35 us against 34, mode 1 15 against 28), up
// to 128 key channels, 16-byte aligned rows; mode 0 needs the 64-row tiles and the scratch.
bool decay_chunk_takes(const DecayScanArgs& a) {
  auto aligned = [](const void* p, long long ld) { return (uintptr_t)p % 16 == 0 && ld % 8 == 0; };
  if (a.mode > 1 || !a.cu_q || a.T < (a.mode == 0 ? 48LL : 8LL) * a.runs || a.N % 8 || a.N > 128) return false;
  if (!aligned(a.q, a.ldq) || !aligned(a.k, a.ldk)) return false;
  // rows that overlap go token by token: what lies behind a chunk's last row is told by its place
  auto apart = [](long long ld, long long width) { return ld == 0 || ld >= width; };
  if (!apart(a.ldq, a.N) || !apart(a.ldk, a.N) || !apart(a.ldv, a.P)) return false;
  constexpr long long top = 1 << 24;      // (a chunk of 32 rows is addressed by 32-bit offsets)
  if (std::max({a.ldq, a.ldk, a.ldv, a.ldd, (long long)a.H * a.P, (long long)a.H * ws_cols(a.N)}) > top) return false;
  return a.mode == 1 || (a.tiles && a.ntiles > 0 && a.ws && (uintptr_t)a.ws % 16 == 0);
}

// floats of the chunked form's scratch: mode 0's blocks, then the segments' states and decays
static long long block_floats(int mode, long long T, long long runs, long long H, int N) {
  return mode == 0 ? (T / C + runs + 1) * H * (chunk_block(padded(N)) / 4) : 0;
}
long long decay_chunk_scratch(int mode, long long T, long long runs, long long H, int N, long long P) {
  if (mode > 1 || N > 128) return 0;
  return block_floats(mode, T, runs, H, N) + walk_segments(mode, T, runs, H, P) * H * ((P + 63) / 64 * 64 + 1) * padded(N);
}
void decay_chunk_segments(DecayScanArgs& a) {
  a.segments = (uintptr_t)a.ws % 16 == 0 ? walk_segments(a.mode, a.T, a.runs, a.H, a.P) : 0;
  a.seg = a.ws + block_floats(a.mode, a.T, a.runs, a.H, a.N);
}

void launch_decay_chunks(const DecayScanArgs& a, hipStream_t s) {
  if (a.mode == 0) launch_mode<0>(a, s);
  else launch_mode<1>(a, s);
}
