// K4 / K5: paged attention on CDNA4 MFMA (v_mfma_f32_16x16x32_bf16), D = 128.
//
// Cache layout (written by rope_cache.hip):
//   k_cache [NB][Hkv][BS][D]   token-major
//   v_cache [NB][Hkv][D][BS]   dim-major
// Both kernels use the "swapped" products so that no operand needs an LDS
// transpose and every operand fragment is a contiguous 16-byte load:
//   S^T[tok][q] = K[tok][:] . Q[q][:]      A = K rows,   B = Q^T
//   O^T[d][q]  += V^T[d][tok] . P^T[tok][q] A = V^T rows, B = P^T
// The accumulator of S^T (lane: column q = lane&15, rows 4*(lane>>4)+r) is
// turned into the P^T B-operand in registers: a 32-token group is computed as
// two 16-token S^T tiles whose token lists interleave in 4s
// (tile a holds tokens 8*(row>>2) + 4a + (row&3)), so lane group h owns tokens
// 8h..8h+7 of the group = exactly the k-slice its B fragment needs.
// MFMA i of the contraction over D takes dims 32 i + 8 h from lane group h: one
// load instruction of the decode kernels reads 64 contiguous bytes of each of 16
// K rows (a 64-byte run per lane, as the LDS-staged prompt kernel reads its tile,
// touches twice the lines per instruction: 64 x 900 tokens 67 -> 63 us).  Softmax is online (running max / sum per query column),
// in base 2 with the 1/sqrt(D)*log2(e) scale folded into one multiply.
//
// Decode (K5): grid (seq, kv_head, partition), 8 waves, 256 tokens (32 per wave) a step; the
// G = Hq/Hkv query heads of a kv head are the MFMA columns (K/V are read once per kv head).
// Multi-partition sequences write fp32 partials that the last-arriving partition combines
// (split-KV, flash-decoding, one launch).  The grid comes from the number of (sequence, kv head)
// units and the tables' width alone, so the launch is hipGraph-capturable; the kernel cuts every
// context into that many equal parts, one far above the others into more, and workgroups past the
// last one exit at once.
//
// Prefill (K4): causal + varlen + chunked prefill (queries are the LAST qlen
// positions of a context of length ctx), reading K/V from the paged cache.
// Default: attn_prefill_m32p_kernel (32x32x16 MFMA, GQA heads share K/V tiles,
// see its comment) or, for steps of few query rows, attn_prefill_rows_kernel (one head,
// keys shared out over the waves); the 16x16 kernels remain for GQA groups of 1/2 heads.
#include <stdlib.h>
#include <string.h>

#include "attn_decode.h"
#include "common.h"
#include "direct_lds.h"
#include "launchers.h"

namespace {

// ---------------------------------------------------------------------------------------------
// Decode (body: attn_decode.h)
// ---------------------------------------------------------------------------------------------
// Whole contexts on more units (sequence, kv head) than CUs: workgroup i gets the i-th longest, and those of the second round (of
// two at most), from the last CU to the first, the rest, so that a CU's two share out evenly; of more rounds the short ones come
// last.  Up to 64 sequences, whose lengths the lanes of a wave hold; more keep the batch's order, an even
// number of them turned.
// All of a round is resident: what a CU has to read is what it takes (64 contexts of 450 .. 1350 tokens, 8 heads: in the
// order of the batch 60.3 us, rows of it turned 59.4, so 56.1; the longest first 59.0; pairs on neighbouring CUs 61.3; 236 MB that are
// read and not used 40.6).  A group's K loaded under the softmax before it took as long.
constexpr int DECODE_CUS = 256;

// The lengths are below 2^bits, and that of the rank is found bit by bit: the largest that more contexts than the rank reach.  (Each
// lane's rank counted over all sequences instead: 64 of 450 .. 1350 tokens, 8 heads, 41.6 us, so 39.4, in the batch's order 46.3.)
SYM_DEV void by_length(const int* __restrict__ ctx_lens, int num_seqs, int Hkv, int bits, int& seq, int& kvh) {
  const int units = num_seqs * Hkv, id = kvh * num_seqs + seq, lane = threadIdx.x & 63;
  const int k = id < DECODE_CUS || units > 2 * DECODE_CUS ? id : units - 1 - (id - DECODE_CUS);
  const int mine = (unsigned)k / (unsigned)Hkv;
  kvh = k - mine * Hkv;
  const int len = lane < num_seqs ? min(max(ctx_lens[lane], 0), (1 << bits) - 1) : -1;
  int t = 0;
  for (int b = bits - 1; b >= 0; --b) {
    const int up = t | 1 << b;
    if (__popcll(__ballot(len >= up)) > mine) t = up;
  }
  // (every ballot by all lanes: behind a && it would be one of those that are left)
  const unsigned long long same = __ballot(len == t);
  const int among = mine - (int)__popcll(__ballot(len > t));      // of like contexts the first first
  const int before = __builtin_amdgcn_mbcnt_hi((unsigned)(same >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)same, 0));
  seq = __builtin_ctzll(same & __ballot(before == among));
}

// GMAX >= G query heads per kv head: the cross-wave merge stages GMAX columns in LDS (GMAX = 4 for
// Llama-3 GQA: 17 KB instead of 68 KB, so LDS no longer caps the resident workgroups per CU)
// ORDER: the launcher's `order` is not 0 (a kernel of its own: the others' loads stood 0.3 us later with it inside)
template <int GMAX, bool UNEVEN, bool ORDER>
__global__ __launch_bounds__(DWAVES * 64, 4) void attn_decode_kernel(
    const bf16* __restrict__ q, const bf16* __restrict__ k_cache, const bf16* __restrict__ v_cache,
    const int* __restrict__ block_tables, const int* __restrict__ ctx_lens, bf16* __restrict__ out,
    float* __restrict__ tmp_o, float* __restrict__ tmp_ml, int* __restrict__ counters, int num_seqs, int Hq, int Hkv,
    int G, int BS, int max_blocks, int max_parts, int parts, int slots_log2, int further, float scale_log2, unsigned inv,
    unsigned inv_heads) {
  // UNEVEN: grid y = part * Hkv + kvh, and past Hkv * parts the further partitions, `further` items for each head (items in
  // the grid's last rows, so that they start behind the others: between them, a batch of like contexts that fills the chip
  // found its workgroups spread unevenly over the CUs, 64 x 900 tokens 61 instead of 55 us).
  int seq = blockIdx.x, kvh = blockIdx.y, part = blockIdx.z;
  if constexpr (UNEVEN) {
    part = min((int)__umulhi(2 * blockIdx.y, inv_heads), parts);  // blockIdx.y / Hkv
    kvh = blockIdx.y - part * Hkv;
    if (part == parts) {
      const int w = kvh * num_seqs + seq;
      seq = (unsigned)w / (unsigned)Hkv;
      kvh = w - seq * Hkv;
      if (seq >= further) return;
    }
  }
  if constexpr (ORDER) {
    const int order = slots_log2 >> 8;      // (in the argument's upper bytes)
    slots_log2 &= 255;
    if (order > 0) {
      if (part == 0) by_length(ctx_lens, num_seqs, Hkv, order, seq, kvh);
    } else if (part < parts) {
      // Workgroups go round the eight XCDs: of 8 n sequences an XCD would get every eighth with all its heads, and a CU several
      // heads of one.  Each row of the grid starts a sequence further on.
      seq += (blockIdx.y + gridDim.y * blockIdx.z) & 7;
      if (seq >= num_seqs) seq -= num_seqs;
    }
  }
  attn_decode_unit<GMAX, UNEVEN>(q, k_cache, v_cache, block_tables, ctx_lens, out, tmp_o, tmp_ml, counters, num_seqs,
                                 Hq, Hkv, G, BS, max_blocks, max_parts, scale_log2, inv, seq, kvh, part, parts,
                                 slots_log2);
}

// ---------------------------------------------------------------------------------------------
// Prefill (varlen, causal, paged, chunked)
// ---------------------------------------------------------------------------------------------
// tiles[i] = {seq, first query row within the seq's new tokens}; a tile is 64 query rows
// (4 waves x 16 rows) of one query head.
__global__ __launch_bounds__(256) void attn_prefill_kernel(
    const bf16* __restrict__ q, const bf16* __restrict__ k_cache, const bf16* __restrict__ v_cache,
    const int* __restrict__ block_tables, const int* __restrict__ ctx_lens, const int* __restrict__ cu_q,
    const int* __restrict__ tiles, bf16* __restrict__ out, int Hq, int Hkv, int BS, int max_blocks,
    float scale_log2) {
  const int tile = blockIdx.x, head = blockIdx.y;
  const int seq = tiles[2 * tile], qrow0 = tiles[2 * tile + 1];
  const int G = Hq / Hkv, kvh = head / G;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int c = lane & 15, h = lane >> 4;
  const int qstart = cu_q[seq], qlen = cu_q[seq + 1] - qstart;
  const int ctx = ctx_lens[seq];
  const int pos0 = ctx - qlen;  // absolute position of query row 0
  const int row0 = qrow0 + 16 * wid;
  if (row0 >= qlen) return;
  const int myrow = row0 + c;
  const bool row_ok = myrow < qlen;
  const int mypos = pos0 + myrow;

  bf16x8 qf[4];
  if (row_ok) {
    const bf16* qp = q + ((long long)(qstart + myrow) * Hq + head) * D + 8 * h;
#pragma unroll
    for (int i = 0; i < 4; ++i) qf[i] = ld16(qp + 32 * i);
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) qf[i] = zero8();
  }
  f32x4 o[8];
#pragma unroll
  for (int dt = 0; dt < 8; ++dt) o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, lsum = 0.f;
  const int* bt = block_tables + (long long)seq * max_blocks;
  // last key any row of this wave may see
  const int kend = min(ctx, pos0 + min(row0 + 16, qlen));
  // software pipeline: group g+1's K/V loads are in flight while group g is computed
  auto kv_ptrs = [&](int tbase, const bf16*& kb, const bf16*& vb) {
    const long long blk = bt[tbase / BS];
    const int boff = tbase % BS;
    kb = k_cache + ((blk * Hkv + kvh) * BS + boff) * D;
    vb = v_cache + (blk * Hkv + kvh) * (long long)D * BS + boff;
  };
  KVFrag cur, nxt;
  if (kend > 0) {
    const bf16 *kb, *vb;
    kv_ptrs(0, kb, vb);
    load_group(kb, vb, BS, cur);
  }
  for (int tbase = 0; tbase < kend; tbase += 32) {
    if (tbase + 32 < kend) {
      const bf16 *kb, *vb;
      kv_ptrs(tbase + 32, kb, vb);
      load_group(kb, vb, BS, nxt);
    }
    compute_group(cur, qf, scale_log2,
                  [&](int a, int r) {
                    const int t = tbase + 8 * h + 4 * a + r;
                    return row_ok && t <= mypos && t < ctx;
                  },
                  o, m, lsum);
    cur = nxt;
  }
  lsum += __shfl_xor(lsum, 16, 64);
  lsum += __shfl_xor(lsum, 32, 64);
  if (!row_ok) return;
  const float inv = lsum > 0.f ? 1.f / lsum : 0.f;
  bf16* op = out + ((long long)(qstart + myrow) * Hq + head) * D;
#pragma unroll
  for (int dt = 0; dt < 8; ++dt) {
    bf16x4 v;
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = (bf16)(o[dt][r] * inv);
    *reinterpret_cast<bf16x4*>(op + 16 * dt + 4 * h) = v;
  }
}

// ---------------------------------------------------------------------------------------------
// Prefill, LDS-staged (K4): one workgroup per (64-query-row tile, kv head, head slice).
// The HPW query heads that share the kv head (GQA) are processed by the same workgroup, so every
// 64-token K/V tile is read from the paged cache ONCE per workgroup (cooperative 16-byte loads,
// double-buffered through LDS: the next tile's global loads are in flight while the current one is
// computed) and each wave reuses every K/V fragment it reads from LDS for its 2 query-column blocks
// (32 query rows).  Wave w: head = slice * HPW + w % HPW, rows 32 * (w / HPW) .. +31 of the tile.
// Math per 32-token group is compute_group (swapped products, in-register P^T).
// ---------------------------------------------------------------------------------------------
constexpr int KST = D + 8;   // LDS row stride of the K tile (elements): 272 B, 16-B aligned, skewed banks
constexpr int VST = 64 + 8;  // LDS row stride of the V^T tile (elements): 144 B

SYM_DEV void lds_group(const bf16* sk, const bf16* sv, int g, KVFrag& f) {
  const int lane = threadIdx.x & 63;
  const int r16 = lane & 15, h = lane >> 4;
#pragma unroll
  for (int a = 0; a < 2; ++a) {
    const int trow = 32 * g + (r16 >> 2) * 8 + 4 * a + (r16 & 3);
#pragma unroll
    for (int i = 0; i < 4; ++i) f.k[a][i] = *reinterpret_cast<const bf16x8*>(sk + trow * KST + 32 * h + 8 * i);
  }
#pragma unroll
  for (int dt = 0; dt < 8; ++dt)
    f.v[dt] = *reinterpret_cast<const bf16x8*>(sv + (16 * dt + r16) * VST + 32 * g + 8 * h);
}

template <int HPW>
__global__ __launch_bounds__(128 * HPW) void attn_prefill_lds_kernel(
    const bf16* __restrict__ q, const bf16* __restrict__ k_cache, const bf16* __restrict__ v_cache,
    const int* __restrict__ block_tables, const int* __restrict__ ctx_lens, const int* __restrict__ cu_q,
    const int* __restrict__ tiles, bf16* __restrict__ out, int Hq, int Hkv, int BS, int max_blocks,
    float scale_log2) {
  constexpr int NT = 128 * HPW;
  constexpr int CH = 1024 / NT;  // 16-byte chunks per thread, per K and per V tile
  __shared__ bf16 sK[2][64 * KST];
  __shared__ bf16 sV[2][D * VST];
  const int tile = blockIdx.x, kvh = blockIdx.y;
  const int G = Hq / Hkv;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int c = lane & 15, h = lane >> 4;
  const int head = kvh * G + blockIdx.z * HPW + wid % HPW;
  const int half = wid / HPW;
  const int seq = tiles[2 * tile], qrow0 = tiles[2 * tile + 1];
  const int qstart = cu_q[seq], qlen = cu_q[seq + 1] - qstart;
  const int ctx = ctx_lens[seq];
  const int pos0 = ctx - qlen;
  if (qrow0 >= qlen) return;  // padding tile (graph-captured prefill buckets): workgroup-uniform, before any barrier
  const int* bt = block_tables + (long long)seq * max_blocks;
  // keys visible to any row of the workgroup / of this wave
  const int kend_wg = min(ctx, pos0 + min(qrow0 + 64, qlen));
  const int row0 = qrow0 + 32 * half;
  const int kend_w = min(ctx, pos0 + min(row0 + 32, qlen));

  bf16x8 qf[2][4];
  int mypos[2];
  bool row_ok[2];
#pragma unroll
  for (int cb = 0; cb < 2; ++cb) {
    const int myrow = row0 + 16 * cb + c;
    row_ok[cb] = myrow < qlen;
    mypos[cb] = pos0 + myrow;
    if (row_ok[cb]) {
      const bf16* qp = q + ((long long)(qstart + myrow) * Hq + head) * D + 32 * h;
#pragma unroll
      for (int i = 0; i < 4; ++i) qf[cb][i] = ld16(qp + 8 * i);
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) qf[cb][i] = zero8();
    }
  }
  f32x4 o[2][8];
  float m[2] = {-INFINITY, -INFINITY}, lsum[2] = {0.f, 0.f};
#pragma unroll
  for (int cb = 0; cb < 2; ++cb)
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) o[cb][dt] = f32x4{0.f, 0.f, 0.f, 0.f};

  // cooperative tile loads: chunk ci -> K (token ci >> 4, 16-B piece ci & 15), V (dim ci >> 3, tokens 8 (ci & 7)..)
  uint4 rk[CH], rv[CH];
  auto gload = [&](int t0) {
#pragma unroll
    for (int j = 0; j < CH; ++j) {
      const int ci = threadIdx.x + j * NT;
      const int tk = t0 + (ci >> 4);
      const long long bk = tk < ctx ? bt[tk / BS] : 0;  // past the context: reserved block 0 (finite)
      rk[j] = *reinterpret_cast<const uint4*>(k_cache + ((bk * Hkv + kvh) * BS + tk % BS) * D + (ci & 15) * 8);
      const int tv = t0 + 8 * (ci & 7);
      const long long bv = tv < ctx ? bt[tv / BS] : 0;
      rv[j] = *reinterpret_cast<const uint4*>(v_cache + ((bv * Hkv + kvh) * D + (ci >> 3)) * (long long)BS + tv % BS);
    }
  };
  auto lstore = [&](int buf) {
#pragma unroll
    for (int j = 0; j < CH; ++j) {
      const int ci = threadIdx.x + j * NT;
      *reinterpret_cast<uint4*>(&sK[buf][(ci >> 4) * KST + (ci & 15) * 8]) = rk[j];
      *reinterpret_cast<uint4*>(&sV[buf][(ci >> 3) * VST + 8 * (ci & 7)]) = rv[j];
    }
  };

  const int ntiles = (kend_wg + 63) / 64;
  if (ntiles > 0) {
    gload(0);
    lstore(0);
  }
  __syncthreads();
  for (int it = 0; it < ntiles; ++it) {
    const int t0 = it * 64;
    if (it + 1 < ntiles) gload(t0 + 64);
    const bf16* sk = sK[it & 1];
    const bf16* sv = sV[it & 1];
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      const int tbase = t0 + 32 * g;
      if (tbase < kend_w) {
        KVFrag f;
        lds_group(sk, sv, g, f);
#pragma unroll
        for (int cb = 0; cb < 2; ++cb)
          compute_group(f, qf[cb], scale_log2,
                        [&](int a, int r) {
                          const int t = tbase + 8 * h + 4 * a + r;
                          return row_ok[cb] && t <= mypos[cb] && t < ctx;
                        },
                        o[cb], m[cb], lsum[cb]);
      }
    }
    if (it + 1 < ntiles) lstore((it + 1) & 1);
    __syncthreads();
  }
#pragma unroll
  for (int cb = 0; cb < 2; ++cb) {
    float l = lsum[cb];
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    if (!row_ok[cb]) continue;
    const float inv = l > 0.f ? 1.f / l : 0.f;
    bf16* op = out + ((long long)(qstart + row0 + 16 * cb + c) * Hq + head) * D;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) {
      bf16x4 v;
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = (bf16)(o[cb][dt][r] * inv);
      *reinterpret_cast<bf16x4*>(op + 16 * dt + 4 * h) = v;
    }
  }
}

// ---------------------------------------------------------------------------------------------
// Prefill, 32x32x16 MFMA (K4, default for GQA groups of 4k heads): same workgroup shape as the
// LDS-staged kernel above (4 query heads of one kv head x 64 query rows, 8 waves, every K/V tile read
// from the paged cache once per workgroup and double-buffered through LDS), with the per-wave math
// re-tiled for v_mfma_f32_32x32x16_bf16:
//   * a wave owns 32 query rows of one head; per 64-key tile it issues 16 S^T MFMAs and 16 P.V MFMAs
//     (32 cycles each); the online softmax runs per 32-key subtile over 16 scores per lane;
//   * S^T = K . Q^T with the K rows permuted (row r loads key r with bits 2 and 3 swapped) so that
//     accumulator registers 8s..8s+7 of a lane hold 8 CONSECUTIVE keys: the bf16-packed accumulator
//     is directly the B operand of O^T += V^T . P^T, and the matching V^T fragment is one contiguous
//     16-byte LDS read (no transpose, no permute);
//   * the contraction over D is permuted the same way for Q/K: lane half hh covers dims 64hh..64hh+63,
//     so a lane's K fragment reads are 128 contiguous bytes of one key row;
//   * the row max crosses lane halves with one v_permlane32_swap; exp2 is the raw v_exp_f32 with the
//     1/sqrt(D)*log2(e) scale folded into one fma; masks are evaluated only on tiles that touch the
//     causal diagonal or the context end;
//   * deferred rescale (T13): the running max moves only when a tile's max exceeds it by > 8 (log2
//     units), so O and l are rescaled on a few tiles instead of every tile (P <= 2^8 before the bf16
//     cast: relative precision unchanged);
//   * the block-table reads of a tile are issued one tile ahead of its K/V loads (a dependent
//     table -> K/V load pair per tile exposed ~2 memory latencies per iteration: 2.5x slower);
//   * heavier tiles first: the engine orders the tiles by visible keys, descending, and the grid has the
//     kv head fastest, so the long causal rows of a sequence start in the first wave of workgroups
//     instead of forming the tail (1x4096: 241 -> 162 us).
// ---------------------------------------------------------------------------------------------
SYM_DEV f32x16 mfma32(bf16x8 a, bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

typedef __attribute__((address_space(3))) bf16x8 lds_bf16x8;

SYM_DEV float xhalf_max(float v) {  // max with the lane 32 apart (same query column, other key half)
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

SYM_DEV float xhalf_sum(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

constexpr float kRescaleThr = 8.f;  // T13 threshold, log2 units


// ---------------------------------------------------------------------------------------------
// Prefill, 32x32x16 MFMA, software-pipelined per 32-key subtile (K4 default).
// Same workgroup / wave decomposition and operand tricks as described above, restructured so
// that a wave's VALU work hides under its own MFMAs: the online-softmax update is per 32-key subtile
// and the loop body for subtile j is
//     [rescale decision for j]  ->  S(j+1) = K . Q^T MFMAs  ||  second half of P(j): exp2, bf16, sum
//                               ->  P(j) . V MFMAs          ||  row max of S(j+1), first half of P(j+1)
// Masks apply only to the <= 2 subtiles of a wave that touch the causal diagonal / context end (a
// uniform branch).  Three K/V tiles in LDS (96 KB, one workgroup per CU at this register budget anyway),
// filled by direct loads: tile t+1 is resident while tile t is consumed, so S(j+1) can cross a tile
// boundary, and tile t+2 loads for a whole iteration.  16-byte chunk i of a K row r is stored at i ^ (r & 15),
// of a V^T row at i ^ ((r >> 1) & 7): operand reads meet no bank twice.
// What bounds it is power: matrix cores busy 0.51 of the cycles, at 1.8 GHz (a large product: 0.82 at 1.7).  So what counts is
// work beside the products; with the tiles through registers (addresses, waits, LDS stores: a fifth of the time) -> so, us: 32 heads,
// one prompt of 7900 tokens 577 -> 542, 8 of 1012 131 -> 128, 16 heads, 3 of 1000 behind 1000 82 -> 76.
// ---------------------------------------------------------------------------------------------
SYM_DEV void mask_subtile(f32x16& s, int kbase, int mypos) {
  const int hh = (threadIdx.x & 63) >> 5;
  const int lim = mypos - kbase - 8 * hh;  // register i holds key kbase + 16 (i >> 3) + 8 hh + (i & 7)
#pragma unroll
  for (int i = 0; i < 16; ++i)
    if (16 * (i >> 3) + (i & 7) > lim) s[i] = -INFINITY;
}

SYM_DEV float subtile_max(const f32x16& s, float scale_log2) {
  float t = fmaxf(fmaxf(s[0], s[1]), s[2]);
#pragma unroll
  for (int i = 3; i < 15; i += 2) t = fmaxf(fmaxf(t, s[i]), s[i + 1]);
  t = fmaxf(t, s[15]);
  return xhalf_max(t) * scale_log2;
}

__global__ __launch_bounds__(512, 2) void attn_prefill_m32p_kernel(
    const bf16* __restrict__ q, const bf16* __restrict__ k_cache, const bf16* __restrict__ v_cache,
    const int* __restrict__ block_tables, const int* __restrict__ ctx_lens, const int* __restrict__ cu_q,
    const int* __restrict__ tiles, bf16* __restrict__ out, int Hq, int Hkv, int bs_shift, int max_blocks,
    float scale_log2) {
  const int BS = 1 << bs_shift, bs_mask = BS - 1;  // power-of-two blocks: no integer division per tile
  constexpr int HPW = 4, KB = 64 * 256, TB = KB + 128 * 128;  // bytes of a K tile, of a K and a V^T tile
  __shared__ __attribute__((aligned(1024))) char smem[3 * TB];
  const int tile = blockIdx.y, kvh = blockIdx.x;  // tiles arrive heaviest first (engine order)
  const int G = Hq / Hkv;
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform to the compiler
  const int c = lane & 31, hh = lane >> 5;
  const int head = kvh * G + blockIdx.z * HPW + wid % HPW;
  const int half = wid / HPW;
  const int seq = tiles[2 * tile], qrow0 = tiles[2 * tile + 1];
  const int qstart = cu_q[seq], qlen = cu_q[seq + 1] - qstart;
  const int ctx = ctx_lens[seq];
  const int pos0 = ctx - qlen;
  if (qrow0 >= qlen) return;  // padding tile (graph-captured prefill buckets): workgroup-uniform, before any barrier
  const int* bt = block_tables + (long long)seq * max_blocks;
  const int row0 = qrow0 + 32 * half;
  const int kend_wg = min(ctx, pos0 + min(qrow0 + 64, qlen));
  const bool wave_live = row0 < qlen;
  const int kend_w = min(ctx, pos0 + min(row0 + 32, qlen));  // keys [0, kend_w) visible to some row
  const int minpos_w = pos0 + row0;                           // the wave's first query position
  const int nsub = wave_live ? (kend_w + 31) >> 5 : 0;        // 32-key subtiles this wave processes
  const int myrow = row0 + c;
  const bool row_ok = myrow < qlen;
  const int mypos = row_ok ? pos0 + myrow : ctx - 1;  // rows past the prompt attend like the last one
  const int last = ctx - 1;
  const int ntiles = (kend_wg + 63) / 64;

  // A wave's four direct loads of a tile: K rows 8 wid .. + 7 (two of 4 rows), V^T rows 16 wid .. + 15 (two of 8); the chunk that a lane
  // takes from its row stands at its own place.  A group of 8 keys is in one block.  Its block's id, a K and a V one a lane, is
  // fetched a tile ahead.  K rows past the context are whatever the block holds (their scores are masked), V's chunks there are the
  // context's last (finite: the cache is zero-initialised and only ever written with finite K/V).
  const int krow = 8 * wid + (lane >> 4), vrow = 16 * wid + (lane >> 3);
  const char* const kbase = reinterpret_cast<const char*>(k_cache + (long long)kvh * BS * D);
  const char* const vbase = reinterpret_cast<const char*>(v_cache + (long long)kvh * BS * D + (long long)vrow * BS);
  const unsigned bbytes = (unsigned)(Hkv * BS * D) * 2;
  const int kch0 = 16 * ((lane & 15) ^ (krow & 15)), kch1 = 16 * ((lane & 15) ^ ((krow + 4) & 15));
  const int vch0 = (lane & 7) ^ ((vrow >> 1) & 7), vch1 = (lane & 7) ^ (((vrow + 8) >> 1) & 7);
  const unsigned lds0 = lds_address(smem) + wid * 2048;
  struct Ids { int k, v0, v1; };
  auto fetch_ids = [&](int t) {
    const int t0 = 64 * t;
    return Ids{bt[min(t0 + 8 * wid, last) >> bs_shift], bt[min(t0 + 8 * vch0, last) >> bs_shift], bt[min(t0 + 8 * vch1, last) >> bs_shift]};
  };
  auto issue = [&](int t, int buf, const Ids& id) {
    const int t0 = 64 * t, at = lds0 + buf * TB;
    const char* kb = kbase + (size_t)(unsigned)id.k * bbytes + (((t0 + krow) & bs_mask) << 8);
    direct_load16(kb + kch0, at);
    direct_load16(kb + 1024 + kch1, at + 1024);
    const int v0 = min(t0 + 8 * vch0, last & ~7), v1 = min(t0 + 8 * vch1, last & ~7);
    direct_load16(vbase + (size_t)(unsigned)id.v0 * bbytes + 2 * (v0 & bs_mask), at + KB);
    direct_load16(vbase + (size_t)(unsigned)id.v1 * bbytes + 2 * (v1 & bs_mask) + 16 * BS, at + KB + 1024);
  };

  // prologue: tiles 0 and 1 (one memory round trip), the queries behind them
  Ids ids{};
  if (ntiles > 0) {
    const Ids i0 = fetch_ids(0), i1 = fetch_ids(ntiles > 1 ? 1 : 0);
    if (ntiles > 2) ids = fetch_ids(2);
    issue(0, 0, i0);
    if (ntiles > 1) issue(1, 1, i1);
  }
  bf16x8 qf[8];
  if (row_ok) {
    const bf16* qp = q + ((long long)(qstart + myrow) * Hq + head) * D + 64 * hh;
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) qf[kk] = ld16(qp + 8 * kk);
  } else {
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) qf[kk] = zero8();
  }
  f32x16 o[4];
#pragma unroll
  for (int dt = 0; dt < 4; ++dt) o[dt] = f32x16{};
  float m = -INFINITY, lsum = 0.f;
  // (the queries have arrived as well: unsaid, every S product of the loop waits for them anew, which by then is for the tiles in flight)
  wait_direct_loads();
  __syncthreads();

  // LDS operand addresses: K row pr + 32 i (i: subtile of the tile), chunk 8 hh + kk; V^T row c + 32 dt, chunk hh + 2 x
  const int pr = (c & 3) | ((c & 4) << 1) | ((c & 8) >> 1) | (c & 16);  // bits 2 <-> 3
  int kx[8], vx[4];
  const unsigned base = lds_address(smem);
#pragma unroll
  for (int kk = 0; kk < 8; ++kk) kx[kk] = base + pr * 256 + 16 * ((8 * hh + kk) ^ (pr & 15));
#pragma unroll
  for (int x = 0; x < 4; ++x) vx[x] = base + KB + c * 128 + 16 * ((hh + 2 * x) ^ ((c >> 1) & 7));
  auto operand = [&](int at) { return *reinterpret_cast<const lds_bf16x8*>((unsigned)at); };

  // The 16 products of a step, 8 of S(j + 1) and 8 of P(j) . V, take their LDS operands from a ring that is read RING products ahead,
  // over the ends of steps (the next K subtile is resident).  The vector work stands between them, about as much at each: the second
  // half of P(j), the row max of S(j + 1), and with the running maximum as it is the first half of P(j + 1), which is formed anew
  // where the next step masks or rescales.
  constexpr int RING = 4;
  bf16x8 f[RING];
  f32x16 sa, sb;  // scores of the current / next subtile (named: static register allocation)
  Pack8 first;      // P(j)'s first half
  first.u = make_uint4(0, 0, 0, 0);
  float tmax = -INFINITY, fsum = 0.f;
  sa = f32x16{};
  if (nsub > 0) {
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) sa = mfma32(operand(kx[kk]), qf[kk], sa);
    tmax = subtile_max(sa, scale_log2);
#pragma unroll
    for (int n = 0; n < RING; ++n) f[n] = operand(kx[n] + 8192);
  }
  auto prob = [&](float s) { return __builtin_amdgcn_exp2f(fmaf(s, scale_log2, -m)); };
  // step j = 2 it + ST: scores of subtile j in sc, of the next one into sn; to_next: from this tile's buffer to the next one's
  auto step = [&](auto st, int j, f32x16& sc, f32x16& sn, int to_next) __attribute__((always_inline)) {
    constexpr int ST = decltype(st)::value;
    if (j >= nsub) return;
    const bool mask = 32 * j + 31 > minpos_w;  // diagonal / context-end subtile: mask, then its true max
    if (mask) {
      mask_subtile(sc, 32 * j, mypos);
      tmax = subtile_max(sc, scale_log2);
    }
    const bool rescale = !__all(tmax <= m + kRescaleThr);
    if (rescale) {
      const float mn = fmaxf(m, tmax);
      const float alpha = __builtin_amdgcn_exp2f(m - mn);  // first subtile: m = -inf, alpha = 0
      m = mn;
      lsum *= alpha;
#pragma unroll
      for (int dt = 0; dt < 4; ++dt) o[dt] *= alpha;
    }
    if (mask || rescale) {
      fsum = 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float p = prob(sc[i]);
        fsum += p;
        first.h[i] = (bf16)p;
      }
    }
    // branch-free from here: S(j + 1) unconditionally (past the wave's last subtile it is an unused stale-LDS product); its row max
    // is an upper bound until a masked subtile recomputes it above
    Pack8 pf[2];
    pf[0] = first;
    float psum = fsum, top = -INFINITY;
    fsum = 0.f;
    sn = f32x16{};
#pragma unroll
    for (int n = 0; n < 16; ++n) {
      if (n < 8) sn = mfma32(f[n % RING], qf[n & 7], sn);
      else o[n & 3] = mfma32(f[n % RING], pf[(n - 8) >> 2].v, o[n & 3]);
      // k of S(j + 1): the tile's second half (ST 0), the next tile's first; then V; then k of S(j + 2), a half on
      const int to = n + RING;
      if (ST == 0 && to == 8)
#pragma unroll
        for (int kk = 0; kk < 8; ++kk) kx[kk] += to_next;
      if (to < 8) f[n % RING] = operand(kx[to] + (ST ? 0 : 8192));
      else if (to < 16) f[n % RING] = operand(vx[2 * ST + ((to - 8) >> 2)] + 4096 * (to & 3));
      else f[n % RING] = operand(kx[to - 16] + (ST ? 8192 : 0));
      if (n < 8) {
        const float p = prob(sc[8 + n]);
        psum += p;
        pf[1].h[n] = (bf16)p;
      } else if (n >= 9 && n < 12) {
#pragma unroll
        for (int i = 6 * (n - 9); i < (n == 11 ? 16 : 6 * (n - 8)); i += 2) top = fmaxf(fmaxf(top, sn[i]), sn[i + 1]);
      } else if (n >= 12) {
#pragma unroll
        for (int i = 2 * (n - 12); i < 2 * (n - 11); ++i) {
          const float p = prob(sn[i]);
          fsum += p;
          first.h[i] = (bf16)p;
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    lsum += psum;
    tmax = xhalf_max(top) * scale_log2;
  };

  int buf = 0;
  for (int it = 0; it < ntiles; ++it) {
    const int next = buf == 2 ? 0 : buf + 1, to_next = (next - buf) * TB;
    if (it + 2 < ntiles) {
      issue(it + 2, next == 2 ? 0 : next + 1, ids);  // (into the buffer of the tile before this one)
      if (it + 3 < ntiles) ids = fetch_ids(it + 3);
    }
    step(IntC<0>{}, 2 * it, sa, sb, to_next);
    step(IntC<1>{}, 2 * it + 1, sb, sa, to_next);
#pragma unroll
    for (int x = 0; x < 4; ++x) vx[x] += to_next;
    buf = next;
    wait_direct_loads();
    __syncthreads();
  }
  const float l = xhalf_sum(lsum);
  if (!row_ok) return;
  const float inv = l > 0.f ? 1.f / l : 0.f;
  bf16* op = out + ((long long)(qstart + myrow) * Hq + head) * D + 4 * hh;
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      bf16x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = (bf16)(o[dt][4 * g + e] * inv);
      *reinterpret_cast<bf16x4*>(op + 32 * dt + 8 * g) = v;
    }
}

// ---------------------------------------------------------------------------------------------
// Prefill of few query rows: a workgroup is 32 query rows of ONE head, its 8 waves share out the keys and meet in LDS, so a
// short prompt behind a long context fills the chip without a workspace (the kernel above has a workgroup per 64 rows and 4
// heads).  Every wave streams its own 32-key subtiles through 16 KB of LDS by direct loads: K of the next subtile is in flight
// during the softmax and P.V, its V during the S product (counted waits, no barrier), its block id one subtile before that.
// A load instruction covers 4 K rows of 256 B or 16 V rows of 64 B (operands read straight from memory touch 32 lines an
// instruction: 26 us for the case below); the 16-byte chunks of a row are stored permuted so that operand reads do not conflict.  K/V are read
// once per head and 32 rows, from the L2 of the XCD that the kv head's workgroups share (grid x = kv head).
// 137 rows behind 1063 cached tokens, 32 heads: 42 -> 13.6 us, of which ~5 the start (lengths, block ids, first K) and the
// merge, the rest each CU's own pull of K/V (64 bytes a cycle).
// ---------------------------------------------------------------------------------------------
constexpr float kNoMax = -3.0e38f;   // running max before any visible key (finite: a wave may see only masked keys)
constexpr int OST = D + 4;           // floats of a partial row in LDS

__global__ __launch_bounds__(512, 2) void attn_prefill_rows_kernel(
    const bf16* __restrict__ q, const bf16* __restrict__ k_cache, const bf16* __restrict__ v_cache,
    const int* __restrict__ block_tables, const int* __restrict__ ctx_lens, const int* __restrict__ cu_q,
    const int* __restrict__ tiles, bf16* __restrict__ out, int Hq, int Hkv, int bs_shift, int max_blocks,
    float scale_log2) {
  const int BS = 1 << bs_shift, bs_mask = BS - 1;
  __shared__ __attribute__((aligned(16))) char smem[8 * 32 * (OST + 2) * 4];   // >= 8 x 16 KB
  float (*po)[32][OST] = reinterpret_cast<float (*)[32][OST]>(smem);
  float (*pm)[32] = reinterpret_cast<float (*)[32]>(smem + 8 * 32 * OST * 4), (*pl)[32] = pm + 8;
  const int kvh = blockIdx.x, tile = blockIdx.y >> 1;
  const int head = kvh * (Hq / Hkv) + blockIdx.z;
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 31, hh = lane >> 5;
  const int seq = tiles[2 * tile], row0 = tiles[2 * tile + 1] + 32 * (blockIdx.y & 1);
  const int qstart = cu_q[seq], qlen = cu_q[seq + 1] - qstart;
  if (row0 >= qlen) return;  // workgroup-uniform, before any barrier
  const int ctx = ctx_lens[seq], pos0 = ctx - qlen, last = ctx - 1;
  const int* bt = block_tables + (long long)seq * max_blocks;
  const int kend = min(ctx, pos0 + min(row0 + 32, qlen));     // keys [0, kend) visible to some row
  const int minpos = pos0 + row0;
  const int nsub = max(0, (kend + 31) >> 5);                  // 32-key subtiles, shared out in runs
  const int j0 = nsub * wid >> 3, j1 = nsub * (wid + 1) >> 3;
  const int myrow = row0 + c;
  const bool row_ok = myrow < qlen;
  const int mypos = row_ok ? pos0 + myrow : last;

  f32x16 o[4];
#pragma unroll
  for (int dt = 0; dt < 4; ++dt) o[dt] = f32x16{};
  float m = kNoMax, lsum = 0.f;
  if (j0 < j1) {
    const bf16* qp = q + ((long long)(qstart + min(myrow, qlen - 1)) * Hq + head) * D + 8 * hh;
    bf16x8 qf[8];
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) qf[kk] = ld16(qp + 16 * kk);
    const unsigned bstride = (unsigned)(Hkv * BS * D);         // elements of a block
    const bf16* kb = k_cache + (long long)kvh * BS * D;
    const bf16* vb = v_cache + (long long)kvh * BS * D;
    const unsigned lds_k = lds_address(smem) + wid * 16384, lds_v = lds_k + 8192;
    const char* sk = smem + wid * 16384;
    const char* sv = sk + 8192;
    // the block of a subtile (32 keys lie in one; past the context: the last key's)
    auto id_of = [&](int j) {
      return (unsigned)__builtin_amdgcn_readfirstlane(bt[min(32 * j, last) >> bs_shift]);
    };
    // K: instruction n, lane l: row 4 n + (l >> 4), 16-byte slot l & 15 = chunk ^ (row's lane in the S product & 15)
    const int krow = lane >> 4, kslot = (lane & 15) ^ krow;
    auto load_k = [&](int j, unsigned id) {
      const bf16* p = kb + (size_t)id * bstride;
#pragma unroll
      for (int n = 0; n < 8; ++n) {
        const int key = min(32 * j + 4 * n + krow, last), ch = kslot ^ ((n & 1) << 3 | (n & 2) << 1);
        direct_load16(p + (((key & bs_mask) << 7) + 8 * ch), lds_k + 1024 * n);
      }
    };
    // V: instruction n, lane l: dim 16 n + (l >> 2), slot l & 3 = key group ^ ((dim >> 1) & 3)
    const int vg = (lane & 3) ^ ((lane >> 3) & 3), vrow = lane >> 2;
    auto load_v = [&](int j, unsigned id) {
      const int key = min(32 * j + 8 * vg, last & ~7);
      const bf16* p = vb + (size_t)id * bstride + ((vrow << bs_shift) + (key & bs_mask));
#pragma unroll
      for (int n = 0; n < 8; ++n) direct_load16(p + (16 * n << bs_shift), lds_v + 1024 * n);
    };
    const unsigned first = id_of(j0);
    unsigned id = id_of(min(j0 + 1, j1 - 1));
    wait_direct_loads();                    // (q: its waits inside the loop would be waits for the loop's loads)
    load_k(j0, first);
    load_v(j0, first);
    const int pr = (c & 3) | ((c & 4) << 1) | ((c & 8) >> 1) | (c & 16);  // bits 2 <-> 3
    const int koff = pr * 256, ksw = c & 15, voff = c * 64, vsw = (c >> 1) & 3;
    for (int j = j0; j < j1; ++j) {
      const bool more = j + 1 < j1;         // (wave-uniform, as are the branches on it)
      __builtin_amdgcn_s_waitcnt(0x0f78);   // vmcnt(8): K of j has arrived (V of j may be in flight)
      asm volatile("" ::: "memory");
      f32x16 sc = f32x16{};
      {
        Pack8 kf[8];
#pragma unroll
        for (int kk = 0; kk < 8; ++kk) kf[kk].u = *reinterpret_cast<const uint4*>(sk + koff + 16 * ((2 * kk + hh) ^ ksw));
#pragma unroll
        for (int kk = 0; kk < 8; ++kk) sc = mfma32(kf[kk].v, qf[kk], sc);
      }
      __builtin_amdgcn_sched_barrier(0);    // (the operands are in registers before their place is filled again)
      const unsigned cur = id;
      if (more) {
        load_k(j + 1, cur);
        id = id_of(min(j + 2, j1 - 1));
      }
      if (32 * j + 31 > minpos) mask_subtile(sc, 32 * j, mypos);
      const float tmax = subtile_max(sc, scale_log2);
      if (!__all(tmax <= m + kRescaleThr)) {
        const float mn = fmaxf(m, tmax);
        const float alpha = __builtin_amdgcn_exp2f(m - mn);
        m = mn;
        lsum *= alpha;
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) o[dt] *= alpha;
      }
      Pack8 pf[2];
      float psum = 0.f;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float p = __builtin_amdgcn_exp2f(fmaf(sc[i], scale_log2, -m));
        psum += p;
        pf[i >> 3].h[i & 7] = (bf16)p;
      }
      lsum += psum;
      if (more) __builtin_amdgcn_s_waitcnt(0x0f78);   // vmcnt(8): V of j has arrived (K of the next may be in flight)
      else wait_direct_loads();
      asm volatile("" ::: "memory");
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) {
          Pack8 vf;
          vf.u = *reinterpret_cast<const uint4*>(sv + 32 * dt * 64 + voff + 16 * ((2 * ks + hh) ^ vsw));
          o[dt] = mfma32(vf.v, pf[ks].v, o[dt]);
        }
      __builtin_amdgcn_sched_barrier(0);
      if (more) load_v(j + 1, cur);
    }
  }
  __syncthreads();                          // (no load is in flight: the staging becomes the partials' place)
  const float l = xhalf_sum(lsum);
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      f32x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = o[dt][4 * g + e];
      *reinterpret_cast<f32x4*>(&po[wid][c][32 * dt + 8 * g + 4 * hh]) = v;
    }
  if (hh == 0) {
    pm[wid][c] = m;
    pl[wid][c] = l;
  }
  __syncthreads();
  const int r = threadIdx.x >> 4, d0 = 8 * (threadIdx.x & 15);
  if (row0 + r >= qlen) return;
  float mx = pm[0][r], sum = 0.f, acc[8] = {};
#pragma unroll
  for (int w = 1; w < 8; ++w) mx = fmaxf(mx, pm[w][r]);
#pragma unroll
  for (int w = 0; w < 8; ++w) {
    const float f = __builtin_amdgcn_exp2f(pm[w][r] - mx);
    sum = fmaf(pl[w][r], f, sum);
    const f32x4 a = *reinterpret_cast<const f32x4*>(&po[w][r][d0]), b = *reinterpret_cast<const f32x4*>(&po[w][r][d0 + 4]);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      acc[e] = fmaf(a[e], f, acc[e]);
      acc[4 + e] = fmaf(b[e], f, acc[4 + e]);
    }
  }
  const float inv = nsub > 0 ? 1.f / sum : 0.f;   // (every row sees its own key; no sum at all only from infinite scores)
  Pack8 res;
#pragma unroll
  for (int e = 0; e < 8; ++e) res.h[e] = (bf16)(acc[e] * inv);
  *reinterpret_cast<uint4*>(out + ((long long)(qstart + row0 + r) * Hq + head) * D + d0) = res.u;
}

}  // namespace

// Decode: a unit is a (sequence, kv head); contexts are cut so far that the workgroups just fill the chip, two 8-wave
// workgroups on each of the 256 CUs.  Between 256 and 384 units whole contexts would leave some CUs one workgroup and others
// two: cut in three they run as two to three even rounds (304 units of 1514 tokens 64.8 -> 52.3 us, of 300 16.9 -> 14.5; 264
// of 900 32.4 -> 31.6; 384 of 1000 49.8 -> 47.5, of 250 16.3 / 16.6); past that cutting costs more (480 of 600 34.4 -> 38.9).
// The kernel replaced a one-wave-per-partition LDS-DMA streaming kernel and a one-wave-per-unit kernel; us for the
// streaming / per-unit / this kernel, contexts spread by half around the mean and other weights read in between:
//   1 sequence x 700 tokens, 8 kv heads   17.3 /  46 /  8.5      64 x 900      66 /  88 /  52  (236 MB: 4.6 TB/s)
//   8 x 1100, 4 kv heads                  17.8 /  92 /  9.7      32 x 4000    148 /   - / 111
//   5 x 5400, 4 kv heads                  28.7 /   - / 22.8      160 x 600    112 / 126 /  84
//   48 x 60                                8.8 / 9.3 /  6.5      256 x 2000   428 / 370 / 335
// Bound by the K/V stream from ~100 MB on, by four dependent round trips (context, K/V, publish, combine) below ~20 MB.
// A context far above the others' would leave its few workgroups walking alone, so where the block tables hold more than
// LONG_STEPS steps a partition, contexts above 3 / 2 of their share of the batch are cut further (attn_decode_unit; us, the
// streaming kernel / every context cut alike / now, 8 kv heads):
//   60 x 300 + 1 x 8000     51 / 126 / 39      100 x 200 + 2 x 30000   148 /  472 /  80      56 x 1000 + 8 x 7000  201 / 216 / 107
//   60 x 200 + 1 x 2000     33 /  38 / 24       60 x 200 + 1 x 120000  329 / 1816 / 112      100 x 100 .. 8000     194 / 258 / 172
// A batch of like contexts pays for the rule: 64 x 900 54.9 -> 55.2, 32 x 4000 118 -> 119.5, 160 x 600 86.9 -> 87.8.  Shares of
// half the size (twice the workgroups) were up to 15 % faster on uneven batches and lost as much on even ones (32 x 4000: 135).
constexpr int DECODE_UNITS = 512, DECODE_THIRDS = 384;

void launch_attn_decode(const bf16* q, const bf16* k_cache, const bf16* v_cache, const int* block_tables,
                        const int* ctx_lens, bf16* out, float* tmp_o, float* tmp_ml, int* counters, int num_seqs,
                        int Hq, int Hkv, int BS, int max_blocks, int max_parts, float scale, hipStream_t s) {
  if (num_seqs == 0 || max_blocks == 0) return;  // (an empty table: no context has a token)
  const float scale_log2 = scale * 1.4426950408889634f;
  const int G = Hq / Hkv;
  const int units = num_seqs * Hkv;  // (parts <= 512: attn_decode_unit's exact division)
  const int cut = units <= DECODE_UNITS / 2 ? DECODE_UNITS / units : units <= DECODE_THIRDS ? 3 : 1;
  const int parts = min(max_parts, cut);
  // (max_parts is the steps of the longest context that the tables hold)
  const bool uneven = num_seqs > 1 && max_parts > LONG_STEPS * parts;
  // a context has no more further partitions than its steps / quota, the batch no more than 2^slots_log2 per kv head
  const int slots_log2 = 31 - __builtin_clz(max(1, DECODE_UNITS / Hkv));
  const int further = (int)min(1ll << slots_log2, (long long)num_seqs * (max_parts - parts));
  const dim3 grid = uneven ? dim3(num_seqs, Hkv * parts + (further * Hkv + num_seqs - 1) / num_seqs)
                           : dim3(num_seqs, Hkv, parts);
  const unsigned inv = (unsigned)((1ull << 32) / parts) + 1;  // (not used for one partition)
  const unsigned inv_heads = (unsigned)((1ull << 31) / Hkv) + 1;
  // Contexts by length (> 0: the bits of a length), the batch's order turned (-1), or as it is.  By length, us, as it is / so, 8 heads:
  // 64 of 225 .. 675 25.3 / 22.7, of 450 .. 1350 46.3 / 39.4, of 120 with one of 1200 36.8 / 23.2, of 900 39.2 / 39.1 (one batch over
  // and over, its K/V partly in the last-level cache); not behind tables of 512 tokens, where all contexts are a step or two (64 of 60
  // 5.7, ranks counted 8.9).  Turned: 96 of 120 with one of 1200, 8 heads 37.2 / 26.5, 128 of 60 with one of 600, 4 heads 19.8 /
  // 13.1; an odd number is spread as it is (65 of 120 with one of 1200: turned 36.7, not 22.5), and contexts in parts are too (48 of
  // 225 .. 675, 4 heads 16.1 / 16.5).
  const long long room = (long long)max_blocks * BS;      // (no context is longer)
  int order = 0;
  if (parts == 1 && units > DECODE_CUS && room > 512 && room < 1 << 30)
    order = num_seqs <= 64 ? 32 - __builtin_clz((unsigned)room) : num_seqs % 2 == 0 ? -1 : 0;
  auto run = [&](auto kern) {
    kern<<<grid, DWAVES * 64, 0, s>>>(q, k_cache, v_cache, block_tables, ctx_lens, out, tmp_o, tmp_ml, counters, num_seqs,
                                      Hq, Hkv, G, BS, max_blocks, max_parts, parts, slots_log2 | order * 256, further, scale_log2, inv,
                                      inv_heads);
  };
  auto pick = [&](auto u, auto o) {
    constexpr bool U = decltype(u)::value != 0, O = decltype(o)::value != 0;
    if (G <= 4) run(attn_decode_kernel<4, U, O>);
    else if (G <= 8) run(attn_decode_kernel<8, U, O>);
    else run(attn_decode_kernel<16, U, O>);
  };
  if (uneven) order ? pick(IntC<1>{}, IntC<1>{}) : pick(IntC<1>{}, IntC<0>{});
  else order ? pick(IntC<0>{}, IntC<1>{}) : pick(IntC<0>{}, IntC<0>{});
}

// Workgroups of the 64-row x 4-head kernel up to which the row kernel takes a prompt step: below, most CUs would idle; above,
// K/V read once per head costs more than it fills, first for batches of short contexts.  us, 64-row kernel / row kernel (query
// rows behind a context):
//   24: 137 of 1200   42 / 13.6      48: 384 of 2000  65 / 34       64: 4 x 128 of 128  12.6 / 11.3    96: 768 of 4000   133 / 106
//   32: 256 of 8000  233 / 69        48: 6 x 40 of 300  16.5 / 15.6   64: 8 x 60 of 600   27 / 21        96: 6 x 128 of 128  12.8 / 15.9
//   48: 3 x 128 of 128  12.2 / 10.8  64: 512 of 512   23 / 16       64: 8 x 100, 4 kv heads  10.7 / 10.6   96: 12 x 60 of 600  29 / 31
constexpr int ROWS_WGS = 64;

void launch_attn_prefill(const bf16* q, const bf16* k_cache, const bf16* v_cache, const int* block_tables,
                         const int* ctx_lens, const int* cu_q, const int* tiles, int num_tiles, bf16* out, int Hq,
                         int Hkv, int BS, int max_blocks, float scale, hipStream_t s) {
  if (num_tiles == 0) return;
  const float scale_log2 = scale * 1.4426950408889634f;
  const int G = Hq / Hkv;
  // A/B knob SYMMETRY_ATTN_PREFILL=lds: the previous 16x16x32 LDS kernel (profiles/attn_prefill_r1.jsonl)
  static const char* knob = getenv("SYMMETRY_ATTN_PREFILL");
  static const bool use_lds = knob && strstr(knob, "lds");
  if (!use_lds && BS >= 8 && (BS & (BS - 1)) == 0 && G % 4 == 0) {
    if (BS >= 32 && Hkv * num_tiles * (G / 4) <= ROWS_WGS) {
      attn_prefill_rows_kernel<<<dim3(Hkv, 2 * num_tiles, G), 512, 0, s>>>(
          q, k_cache, v_cache, block_tables, ctx_lens, cu_q, tiles, out, Hq, Hkv, __builtin_ctz(BS), max_blocks, scale_log2);
      return;
    }
    attn_prefill_m32p_kernel<<<dim3(Hkv, num_tiles, G / 4), 512, 0, s>>>(
        q, k_cache, v_cache, block_tables, ctx_lens, cu_q, tiles, out, Hq, Hkv, __builtin_ctz(BS), max_blocks,
        scale_log2);
    return;
  }
  if (BS % 8 == 0 && (G == 1 || G == 2 || G % 4 == 0)) {
    // LDS-staged kernel: the kv head's query heads share every K/V tile (slices of <= 4 heads)
    const int hpw = G >= 4 ? 4 : G;
    const dim3 grid(num_tiles, Hkv, G / hpw);
    if (hpw == 4)
      attn_prefill_lds_kernel<4><<<grid, 512, 0, s>>>(q, k_cache, v_cache, block_tables, ctx_lens, cu_q, tiles, out,
                                                      Hq, Hkv, BS, max_blocks, scale_log2);
    else if (hpw == 2)
      attn_prefill_lds_kernel<2><<<grid, 256, 0, s>>>(q, k_cache, v_cache, block_tables, ctx_lens, cu_q, tiles, out,
                                                      Hq, Hkv, BS, max_blocks, scale_log2);
    else
      attn_prefill_lds_kernel<1><<<grid, 128, 0, s>>>(q, k_cache, v_cache, block_tables, ctx_lens, cu_q, tiles, out,
                                                      Hq, Hkv, BS, max_blocks, scale_log2);
    return;
  }
  attn_prefill_kernel<<<dim3(num_tiles, Hq), 256, 0, s>>>(q, k_cache, v_cache, block_tables, ctx_lens, cu_q, tiles,
                                                          out, Hq, Hkv, BS, max_blocks, scale_log2);
}
