// Decode attention building blocks of the split-KV kernel (attention.hip).
// Math, layouts and the MFMA operand tricks are described at the top of attention.hip.
#pragma once
#include "common.h"

namespace {

constexpr int D = 128;
constexpr int DWAVES = 8;            // waves per decode workgroup
constexpr int PART = DWAVES * 32;    // tokens a workgroup covers per step (one 32-token group per wave), the
                                     // shortest partition; ~120 VGPRs -> two workgroups per CU, so one unit's
                                     // loads overlap another's finish (bench_attn_decode.py)

SYM_DEV bf16x8 ld16(const bf16* p) {
  Pack8 pk;
  pk.u = *reinterpret_cast<const uint4*>(p);
  return pk.v;
}

SYM_DEV bf16x8 zero8() {
  Pack8 pk;
  pk.u = make_uint4(0, 0, 0, 0);
  return pk.v;
}

// One 32-token group: S^T for two 16-token tiles, online softmax update, P.V.
// Split into a load phase (K and V fragments of the group to registers) and a compute phase so that
// callers can have the next group's loads in flight while computing the current one.
struct KVFrag {
  bf16x8 k[2][4];  // two 16-token S^T tiles x 4 D-slices
  bf16x8 v[8];     // 8 dim tiles of V^T
};

SYM_DEV void load_group(const bf16* __restrict__ kb, const bf16* __restrict__ vb, int BS, KVFrag& f) {
  // kb and vb are uniform over the wave: scalar bases and one 32-bit lane offset each, so that the 16 loads hold no
  // address registers of their own
  const int lane = threadIdx.x & 63;
  const int r16 = lane & 15, h = lane >> 4;
  const unsigned ko = (unsigned)(((r16 >> 2) * 8 + (r16 & 3)) * D + 8 * h) * 2;
  const unsigned vo = (unsigned)(r16 * BS + 8 * h) * 2;
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      f.k[a][i] = ld16(reinterpret_cast<const bf16*>(reinterpret_cast<const char*>(kb + 4 * a * D + 32 * i) + ko));
#pragma unroll
  for (int dt = 0; dt < 8; ++dt)
    f.v[dt] = ld16(reinterpret_cast<const bf16*>(reinterpret_cast<const char*>(vb + 16 * dt * BS) + vo));
}

// `valid(a, r)` tells whether token (8h + 4a + r) of the group is visible to this lane's query column.
template <typename ValidFn>
SYM_DEV void compute_group(const KVFrag& f, const bf16x8 (&qf)[4], float scale_log2, ValidFn valid, f32x4 (&o)[8],
                           float& m, float& lsum) {
  f32x4 s[2];
#pragma unroll
  for (int a = 0; a < 2; ++a) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 4; ++i) acc = mfma16(f.k[a][i], qf[i], acc);
    s[a] = acc;
  }
  float x[8];
  float gmax = -INFINITY;
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float v = valid(a, r) ? s[a][r] * scale_log2 : -INFINITY;
      x[4 * a + r] = v;
      gmax = fmaxf(gmax, v);
    }
  gmax = fmaxf(gmax, __shfl_xor(gmax, 16, 64));
  gmax = fmaxf(gmax, __shfl_xor(gmax, 32, 64));
  const float m_new = fmaxf(m, gmax);
  // m_new == -inf only if this column saw no visible token yet (causal prefill rows); keep zeros.
  // raw v_exp_f32 (the ocml exp2f adds a denormal range reduction softmax does not need)
  const float alpha = (m_new == -INFINITY) ? 1.f : __builtin_amdgcn_exp2f(m - m_new);
  Pack8 pf;
  float psum = 0.f;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float p = (m_new == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(x[j] - m_new);
    psum += p;
    pf.h[j] = (bf16)p;
  }
  lsum = lsum * alpha + psum;
  m = m_new;
#pragma unroll
  for (int dt = 0; dt < 8; ++dt) {
    o[dt] *= alpha;
    o[dt] = mfma16(f.v[dt], pf.v, o[dt]);
  }
}

// Cross-wave finish of one (seq, kv head, partition) unit: the 8 waves' online-softmax states are merged
// through LDS; a single-partition context writes its output rows, a multi-partition one publishes fp32
// partials and the last-arriving partition combines them (split-KV, flash-decoding, one launch).
// GMAX >= G query columns are staged.
//
// Both phases are latency, and every thread takes part in both.  In the merges a thread has DIMS dims of a column, so that the 8
// states are 8 DIMS multiply-adds for it (8 dims of a thread in the first 16 GMAX threads took 64 multiply-adds, in scalar
// instructions: 5 contexts of 5400 tokens, 4 heads, 17.5 -> 16.8 us; 516 batches 0.98 of the time, 3 over 1.03).  In the combine the
// 512 threads are 512 / (16 GMAX) sets that walk the partitions strided and merge through LDS, so the partials of up to 8
// partitions of a 4-head group are one round trip past the L2.
template <int N>
struct IntC {
  static constexpr int value = N;
};

union F2 {
  unsigned long long u;
  float f[2];
};

template <int GMAX>
SYM_DEV void attn_finish(const f32x4 (&o)[8], float m, float lsum, int nparts, int seq, int kvh, int part, int Hq,
                         int Hkv, int G, int max_parts, bf16* __restrict__ out, float* __restrict__ tmp_o,
                         float* __restrict__ tmp_ml, int* __restrict__ counters) {
  constexpr int SETS = DWAVES * 4 / GMAX;  // thread sets of 16 GMAX threads
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int c = lane & 15, h = lane >> 4;
  lsum += __shfl_xor(lsum, 16, 64);
  lsum += __shfl_xor(lsum, 32, 64);

  __shared__ F2 sm_ml[DWAVES][GMAX];
  __shared__ __attribute__((aligned(16))) float sm_o[DWAVES][GMAX][D + 4];
  if (c < GMAX) {
    if (h == 0) {
      F2 ml;
      ml.f[0] = m;
      ml.f[1] = lsum;
      sm_ml[wid][c].u = ml.u;
    }
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) *reinterpret_cast<f32x4*>(&sm_o[wid][c][16 * dt + 4 * h]) = o[dt];
  }
  __syncthreads();

  // merging, thread (mq, md) owns DIMS dims of query column mq; combining, thread (set, qq, d0) reads 8 dims of column qq
  constexpr int DIMS = GMAX / 4, COL = DWAVES * 64 / GMAX;
  static_assert(COL * DIMS == D, "all threads share the columns' dims");
  const int mq = threadIdx.x / COL, md = threadIdx.x % COL * DIMS;
  const int set = threadIdx.x / (16 * GMAX);
  const int qq = (threadIdx.x >> 4) % GMAX;
  const int d0 = (threadIdx.x & 15) * 8;
  const bool owner = mq < G;
  float M, L, sum[DIMS];
  // all of a column's states at once: their LDS reads are independent (one after the other the merge was 2 us longer)
  auto merge = [&](auto count) {
    constexpr int N = decltype(count)::value;
    F2 ml[N];
    M = -INFINITY;
    L = 0.f;
#pragma unroll
    for (int j = 0; j < DIMS; ++j) sum[j] = 0.f;
#pragma unroll
    for (int w = 0; w < N; ++w) {
      ml[w].u = sm_ml[w][mq].u;
      M = fmaxf(M, ml[w].f[0]);
    }
#pragma unroll
    for (int w = 0; w < N; ++w) {
      const float f = ml[w].f[0] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ml[w].f[0] - M);
      L += ml[w].f[1] * f;
#pragma unroll
      for (int j = 0; j < DIMS; ++j) sum[j] += sm_o[w][mq][md + j] * f;
    }
  };
  if (owner) merge(IntC<DWAVES>{});
  bool last = true;
  if (nparts > 1) {  // uniform over the workgroup
    // Split-KV combine in the same launch (no reduce kernel): every partition publishes its partial
    // state with write-through (sc1) stores, drains them (vmcnt(0)), then bumps the (seq, kv head)
    // arrival counter; the workgroup whose add returns nparts - 1 reads all partials back with sc1
    // loads and writes the output, then re-arms the counter to 0 (graph-replay safe, no memset).
    F2 t;
    if (owner) {
      const long long row = ((long long)seq * Hq + kvh * G + mq) * max_parts + part;
      float* po = tmp_o + row * D + md;
      if constexpr (DIMS == 1) {
        __hip_atomic_store(po, sum[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      } else {
#pragma unroll
        for (int j = 0; j < DIMS; j += 2) {
          t.f[0] = sum[j];
          t.f[1] = sum[j + 1];
          __hip_atomic_store(reinterpret_cast<unsigned long long*>(po + j), t.u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
      }
      if (md == 0) {
        t.f[0] = M;
        t.f[1] = L;
        __hip_atomic_store(reinterpret_cast<unsigned long long*>(tmp_ml + row * 2), t.u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __shared__ int s_last;
    __syncthreads();  // (also: the merge's LDS reads are done before the combine rewrites the arrays)
    int* cnt = counters + (long long)seq * Hkv + kvh;
    if (threadIdx.x == 0)
      s_last = __hip_atomic_fetch_add(cnt, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == nparts - 1;
    __syncthreads();
    last = s_last;
    if (!last) return;
    if (threadIdx.x == 0) __hip_atomic_store(cnt, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (qq < G) {
      const long long base = ((long long)seq * Hq + kvh * G + qq) * max_parts;
      const unsigned long long* po = reinterpret_cast<const unsigned long long*>(tmp_o + base * D + d0);
      const unsigned long long* pm = reinterpret_cast<const unsigned long long*>(tmp_ml + base * 2);
      float Mc = -INFINITY, Lc = 0.f;
      f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll 2
      for (int p = set; p < nparts; p += SETS) {
        F2 v[4];
        t.u = __hip_atomic_load(pm + p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int j = 0; j < 4; ++j)
          v[j].u = __hip_atomic_load(po + p * (D / 2) + j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        // online merge of one state: an empty one has m = -inf, l = 0 and finite sums
        const float mn = fmaxf(Mc, t.f[0]);
        const float fo = mn == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(Mc - mn);
        const float fw = mn == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(t.f[0] - mn);
        Lc = Lc * fo + t.f[1] * fw;
        acc[0] = acc[0] * fo + f32x4{v[0].f[0], v[0].f[1], v[1].f[0], v[1].f[1]} * fw;
        acc[1] = acc[1] * fo + f32x4{v[2].f[0], v[2].f[1], v[3].f[0], v[3].f[1]} * fw;
        Mc = mn;
      }
      if (d0 == 0) {
        t.f[0] = Mc;
        t.f[1] = Lc;
        sm_ml[set][qq].u = t.u;
      }
      f32x4* w = reinterpret_cast<f32x4*>(&sm_o[set][qq][d0]);
      w[0] = acc[0];
      w[1] = acc[1];
    }
    __syncthreads();
    if (owner) merge(IntC<SETS>{});
  }
  if (owner) {
    const float inv = 1.f / L;
    bf16* to = out + ((long long)seq * Hq + kvh * G + mq) * D + md;
#pragma unroll
    for (int j = 0; j < DIMS; ++j) to[j] = (bf16)(sum[j] * inv);
  }
}

SYM_DEV void load_q(const bf16* __restrict__ q, int seq, int Hq, int kvh, int G, bf16x8 (&qf)[4]) {
  const int lane = threadIdx.x & 63;
  const int c = lane & 15, h = lane >> 4;
  if (c < G) {
    const bf16* qp = q + ((long long)seq * Hq + kvh * G + c) * D + 8 * h;
#pragma unroll
    for (int i = 0; i < 4; ++i) qf[i] = ld16(qp + 32 * i);
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) qf[i] = zero8();
  }
}

SYM_DEV int steps_of(int ctx) { return (int)((unsigned)max(0, ctx + PART - 1) / PART); }

// Sum over the wave, in a scalar register (DPP inside each row of 16 lanes, then the four rows).
SYM_DEV int wave_total(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xf, 0xf, true);   // lanes 1 apart
  v += __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xf, 0xf, true);   // 2
  v += __builtin_amdgcn_update_dpp(0, v, 0x141, 0xf, 0xf, true);  // the other four of eight
  v += __builtin_amdgcn_update_dpp(0, v, 0x140, 0xf, 0xf, true);  // the other eight of sixteen
  return __builtin_amdgcn_readlane(v, 0) + __builtin_amdgcn_readlane(v, 16) + __builtin_amdgcn_readlane(v, 32) +
         __builtin_amdgcn_readlane(v, 48);
}

// Steps a partition of a long context has: the batch's steps shared out over 2^slots_log2 workgroups per kv head.  Every wave
// that asks computes the same from the same lengths.
SYM_DEV int batch_quota(const int* __restrict__ ctx_lens, int num_seqs, int slots_log2) {
  int total = 0;
#pragma unroll 4
  for (int i = threadIdx.x & 63; i < num_seqs; i += 64) total += steps_of(ctx_lens[i]);
  return max(1, (wave_total(total) + (1 << slots_log2) - 1) >> slots_log2);
}

// Partitions of a context: `parts` (none shorter than a step), or for one of more than 3 / 2 of its share of the batch as many
// as make partitions of that share (half above the mean is left alone).  Contexts up to LONG_STEPS steps a partition are not asked about the batch: the sum over
// the lengths is a round trip in front of their K/V (contexts of ~900 tokens, 64 of them: 0.6 us of 55 when all above four
// steps asked).
constexpr int LONG_STEPS = 6;

SYM_DEV bool may_be_long(int steps, int parts) { return steps > LONG_STEPS * parts; }

SYM_DEV int partitions_of(int steps, int parts, int quota, int max_parts) {
  if (!may_be_long(steps, parts) || 2 * steps <= 3 * parts * quota) return min(steps, parts);
  return min((int)((unsigned)(steps + quota - 1) / (unsigned)quota), max_parts);
}

// Item e of the further partitions (those past a context's first `parts`, in the order of the sequences) -> (seq, part);
// false: there are fewer.
SYM_DEV bool further_partition(const int* __restrict__ ctx_lens, int num_seqs, int parts, int quota, int max_parts, int e,
                               int& seq, int& part) {
  const int lane = threadIdx.x & 63;
  for (int i0 = 0; i0 < num_seqs; i0 += 64) {
    const int steps = i0 + lane < num_seqs ? steps_of(ctx_lens[i0 + lane]) : 0;
    const int more = max(0, partitions_of(steps, parts, quota, max_parts) - parts);
    int upto = more;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(upto, o, 64);
      if (lane >= o) upto += v;
    }
    const unsigned long long past = __ballot(upto > e);
    if (past) {
      const int l = __builtin_ctzll(past);
      seq = i0 + l;
      part = parts + e - __builtin_amdgcn_readlane(upto - more, l);
      return true;
    }
    e -= __builtin_amdgcn_readlane(upto, 63);
  }
  return false;
}

// Split-KV decode attention unit (seq, kv head, partition) on an 8-wave workgroup; the G = Hq/Hkv query heads
// of the kv head are the MFMA columns.  A context of n 256-token steps (8 waves x one 32-token group) is cut
// into min(parts, n) partitions of whole steps, as equal as they allow: the launcher picks `parts` from the
// number of units, the kernel the partition from the context, so that a batch of like contexts gives the chip
// about the same number of workgroups and one that fills it alone is not split at all.
// UNEVEN (block tables wide enough for contexts far above the others'): a context of more than 3 / 2 of its
// share of the batch is cut into partitions of that share; part == parts then stands for the further partitions, and
// seq is the item's number among them.
template <int GMAX, bool UNEVEN>
SYM_DEV void attn_decode_unit(const bf16* __restrict__ q, const bf16* __restrict__ k_cache,
                              const bf16* __restrict__ v_cache, const int* __restrict__ block_tables,
                              const int* __restrict__ ctx_lens, bf16* __restrict__ out, float* __restrict__ tmp_o,
                              float* __restrict__ tmp_ml, int* __restrict__ counters, int num_seqs, int Hq, int Hkv,
                              int G, int BS, int max_blocks, int max_parts, float scale_log2, unsigned inv, int seq,
                              int kvh, int part, int parts, int slots_log2) {
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h = lane >> 4;
  if (UNEVEN && __builtin_expect(part >= parts, 0)) {
    const int quota = batch_quota(ctx_lens, num_seqs, slots_log2);
    if (!further_partition(ctx_lens, num_seqs, parts, quota, max_parts, seq, seq, part)) return;
  }
  const int* bt = block_tables + (long long)seq * max_blocks;
  const int bsh = __builtin_ctz(BS);  // block sizes are powers of two (launchers check)
  // The context length, the block of this wave's first group in a context of at most `parts` steps and the query are
  // independent loads: one memory round trip before the K/V stream instead of three (ctx -> table -> K/V).
  // Entries past the context are fetched from within the row but never dereferenced.
  int blk = bt[min((part * PART + wid * 32) >> bsh, max_blocks - 1)];
  bf16x8 qf[4];
  load_q(q, seq, Hq, kvh, G, qf);
  const int ctx = ctx_lens[seq];
  const int steps = steps_of(ctx);
  int nparts = min(parts, steps);
  // first step of partition i: floor(i * steps / parts); `inv` = floor(2^32 / parts) + 1 is exact for i * steps
  // below 2^32 / parts (the launcher keeps parts <= 512).  Fewer steps than partitions: one step each.
  auto first = [&](int i) { return steps <= parts ? i : i == parts ? steps : (int)__umulhi((unsigned)(i * steps), inv); };
  int from = first(part), to = first(part + 1);
  if (UNEVEN && __builtin_expect(may_be_long(steps, parts), 0)) {
    nparts = partitions_of(steps, parts, batch_quota(ctx_lens, num_seqs, slots_log2), max_parts);
    if (nparts > parts) {
      from = (unsigned)(part * steps) / (unsigned)nparts;
      to = (unsigned)(part * steps + steps) / (unsigned)nparts;
    }
  }
  if (part >= nparts) return;  // (an empty context has no partition)
  const int end = min(ctx, to * PART);
  int tok0 = from * PART + wid * 32;
  if (steps > parts) blk = bt[min(tok0 >> bsh, max_blocks - 1)];
  f32x4 o[8];
#pragma unroll
  for (int dt = 0; dt < 8; ++dt) o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, lsum = 0.f;
  while (tok0 < end) {  // uniform over the wave
    const int boff = tok0 & (BS - 1);
    KVFrag f;
    load_group(k_cache + (((long long)blk * Hkv + kvh) * BS + boff) * D,
               v_cache + ((long long)blk * Hkv + kvh) * (long long)D * BS + boff, BS, f);
    blk = bt[min((tok0 + PART) >> bsh, max_blocks - 1)];  // the next group's, beside this one's loads
    // all 16 loads in flight before the first use (left alone, the scheduler saves registers by waiting for every
    // V fragment in turn: 16 round trips a group, 12.3 instead of 8 us for 10 sequences of ~300 tokens)
    __builtin_amdgcn_sched_barrier(0);
    compute_group(f, qf, scale_log2, [&](int a, int r) { return tok0 + 8 * h + 4 * a + r < end; }, o, m, lsum);
    tok0 += PART;
  }
  attn_finish<GMAX>(o, m, lsum, nparts, seq, kvh, part, Hq, Hkv, G, max_parts, out, tmp_o, tmp_ml, counters);
}


}  // namespace
