// One token of the decaying recurrences of decay_scan.hip for one (sequence, head) by one workgroup of 256 threads, and what follows
// the scan in the model: the head's norm, weight and gate, in bf16.
//
// What bounds it is the state, read and written once (128 KB at 128 x 256).  The whole head is in one workgroup, so that its norm is
// too: a wave owns a quarter of the key channels, a lane four neighbouring value columns of NPAD / 4 / (64 / PQ) of them, in 16-byte
// pieces that are all in flight before the first is used.  The waves' sums meet in LDS.
#pragma once
#include "common.h"
#include "hybrid_launchers.h"

constexpr int DECAY_NT = 256;
constexpr int decay_token_lds(int P) { return (3 * 128 + 4 * P + 8) * 4; }

SYM_DEV float decay_softplus(float v) { return fmaxf(v, 0.f) + log1pf(expf(-fabsf(v))); }

// MODE 0 (channel gate), 1 (step size); PQ: P / 4; NPAD: N
template <int MODE, int PQ, int NPAD>
SYM_DEV void decay_token_block(const DecayTokenArgs& d, int h, int run, float* lds) {
  constexpr int P = 4 * PQ, RL = NPAD / 4 / (64 / PQ);
  const DecayScanArgs& a = d.s;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int cq = lane & (PQ - 1), n0 = wave * (NPAD / 4) + lane / PQ * RL;
  const int pr = a.prev_row[run], sv = a.save_slot[run];
  f32x4 S[RL];
  if (pr <= -2) {
    const float* st = a.state + (long long)(-(pr + 2)) * a.state_stride + ((long long)h * NPAD + n0) * P + 4 * cq;
#pragma unroll
    for (int i = 0; i < RL; ++i) S[i] = *reinterpret_cast<const f32x4*>(st + i * P);
  } else {
#pragma unroll
    for (int i = 0; i < RL; ++i) S[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  float *qS = lds, *kS = lds + NPAD, *aS = lds + 2 * NPAD, *red = lds + 3 * NPAD, *scratch = red + 4 * P;
  const bf16* vr = reinterpret_cast<const bf16*>(a.v) + run * a.ldv + (long long)h * P;
  const bf16x4 vb = *reinterpret_cast<const bf16x4*>(vr + 4 * cq);
  float gate = 0.f, w = 0.f, own = 0.f;      // of column tid
  if (tid < P) {
    gate = (float)reinterpret_cast<const bf16*>(d.gate)[run * d.ldg + (long long)h * P + tid];
    w = d.w[(h * P + tid) % d.wlen];
    own = (float)vr[tid];
  }
  const int grp = h / a.hpg;
  if (tid < NPAD) {
    qS[tid] = (float)reinterpret_cast<const bf16*>(a.q)[run * a.ldq + (long long)grp * NPAD + tid] * a.q_scale;
    kS[tid] = (float)reinterpret_cast<const bf16*>(a.k)[run * a.ldk + (long long)grp * NPAD + tid];
    if constexpr (MODE == 0) {
      const long long n = (long long)h * NPAD + tid;
      float z = 0.f;
      if (d.low) {      // a low-rank projection's second factor, rounded as its own launch leaves it
        const bf16 *x = reinterpret_cast<const bf16*>(d.low) + run * d.ldl, *f = reinterpret_cast<const bf16*>(a.dz) + n * d.rank;
#pragma unroll 2
        for (int r = 0; r < d.rank; r += 8) {
          float xv[8], fv[8];
          load8(x + r, xv);
          load8(f + r, fv);
#pragma unroll
          for (int j = 0; j < 8; ++j) z += xv[j] * fv[j];
        }
        z = (float)(bf16)z;
      } else {
        z = (float)reinterpret_cast<const bf16*>(a.dz)[run * a.ldd + n];
      }
      aS[tid] = expf(-decay_softplus(-(z + a.dbias[n])) * (1.f / a.tau));
    }
  }
  float at = 0.f, bt = 1.f;
  if constexpr (MODE == 1) {
    bt = decay_softplus((float)reinterpret_cast<const bf16*>(a.dz)[run * a.ldd + h] + a.dbias[h]);
    at = expf(-expf(a.rate[h]) * bt);
  }
  __syncthreads();
  f32x4 u, o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int c = 0; c < 4; ++c) u[c] = (float)vb[c] * bt;
#pragma unroll
  for (int i = 0; i < RL; i += 4) {
    const f32x4 k4 = *reinterpret_cast<const f32x4*>(kS + n0 + i), q4 = *reinterpret_cast<const f32x4*>(qS + n0 + i);
    const f32x4 a4 = MODE == 0 ? *reinterpret_cast<const f32x4*>(aS + n0 + i) : f32x4{at, at, at, at};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      S[i + j] = a4[j] * S[i + j] + k4[j] * u;
      o += S[i + j] * q4[j];
    }
  }
  if (sv >= 0) {
    float* st = a.state + (long long)sv * a.state_stride + ((long long)h * NPAD + n0) * P + 4 * cq;
#pragma unroll
    for (int i = 0; i < RL; ++i) *reinterpret_cast<f32x4*>(st + i * P) = S[i];
  }
#pragma unroll
  for (int sh = PQ; sh < 64; sh <<= 1)
#pragma unroll
    for (int c = 0; c < 4; ++c) o[c] += __shfl_xor(o[c], sh, 64);
  if (lane < PQ) *reinterpret_cast<f32x4*>(red + wave * P + 4 * cq) = o;
  __syncthreads();
  float y = 0.f;
  if (tid < P) {
    y = (red[tid] + red[P + tid]) + (red[2 * P + tid] + red[3 * P + tid]) + (a.skip ? a.skip[h] * own : 0.f);
    gate *= 1.f / (1.f + expf(-gate));
    if (d.ss) y *= gate;
  }
  const float sq = block_sum<DECAY_NT>(y * y, scratch);
  if (tid < P) {
    const float r = d.ss ? 1.f : 1.f / sqrtf(sq / (float)P + d.eps);
    y = d.ss ? y * w : y * r * w * gate;
    reinterpret_cast<bf16*>(d.out)[((long long)run * a.H + h) * P + tid] = (bf16)y;
    if (d.ss && tid == 0) d.ss[(long long)run * a.H + h] = sq;
  }
}
