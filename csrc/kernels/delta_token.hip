// One token of the gated delta rule (delta_rule.hip) for one (sequence, head) by one workgroup, from the projections to the head's
// normed and gated output: what a decode step did in four to six launches (convolution, low-rank factors, recurrence, norm).
//
//     q, k, v = silu(conv(z)),  q and k to unit length,  beta = sigmoid(b),  S <- g S;  u = beta (v - S^T k);  S <- S + k u^T;  y = S^T q
//     out = y / rms(y) * w * gate
//
// What bounds it is the state, 128 KB read and written at 128 x 256: its loads, 16 bytes a lane, are all in flight first, and the
// convolution, the step size's dot products and the low-rank factors (matrix products of 16 channels whose 16 columns are the same
// row) are formed while they arrive.  A wave owns 16 of the 128 key channels, a lane four neighbouring value columns of PQ / 4 of
// them (four waves of 32 with the factors a tile at a time: 16 rows of 8 heads x 128 x 256 11.3 us, with factors of rank 128 18.1); S^T k and S^T q meet in LDS.  A head's query, key and value channels belong to its workgroup alone, so the carried taps and
// the state may move on in place.
#include "common.h"
#include "hybrid_launchers.h"

namespace {

constexpr int NT = 512, NW = NT / 64, N = 128, TAPS = 4;

SYM_DEV float softplus_exact(float v) { return fmaxf(v, 0.f) + log1pf(expf(-fabsf(v))); }
SYM_DEV float sigmoidf(float v) { return 1.f / (1.f + expf(-v)); }
SYM_DEV float low16(unsigned int v) { return __uint_as_float(v << 16); }
SYM_DEV float high16(unsigned int v) { return __uint_as_float(v & 0xffff0000u); }

// lane (lane & 15) < 4 of each 16: its output of a product whose 16 columns are the same, 4 (lane / 16) + (lane & 15)
SYM_DEV float own_of(f32x4 v, int lane) {
  const int r = lane & 3;
  return r == 0 ? v[0] : r == 1 ? v[1] : r == 2 ? v[2] : v[3];
}

// CHANNEL: 0, or the low-rank factors' rank in 32s where that is at most 4 for both (their loads are then in flight at once), or -1
template <int CHANNEL, int PQ>
__global__ __launch_bounds__(NT) void delta_token_kernel(DeltaTokenArgs a) {
  constexpr int P = 4 * PQ, RL = PQ / 4;
  __shared__ __attribute__((aligned(16))) float qS[N], kS[N], gS[N], vS[P], gateS[P], redk[NW][P], redq[NW][P], dots[NW], scratch[NW];
  const int h = blockIdx.x, row = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int cq = lane & (PQ - 1), n0 = N / NW * wave + lane / PQ * RL;
  // What does not wait for the row's slot is loaded first.
  // Waves 0, 1: the head's query and key channels, two a lane; 2, 3: its values; 4 to 7: the step size's and, a decay a head, the
  // decay's pre-activations
  const int kind = wave < 2 ? wave : 2, e = 2 * (kind < 2 ? lane : tid - 128);
  const bool on = kind < 2 || (wave < 4 && e < P);
  const int c = (kind < 2 ? (kind * a.H + h) * N : 2 * a.H * N + h * P) + e;
  const int C = 2 * a.H * N + a.H * P;
  unsigned int x[TAPS] = {0, 0, 0, 0};      // x[b]: the inputs b places back
  uint4 w = {0, 0, 0, 0};                   // [channel][tap]
  float d0 = 0.f, d1 = 0.f;
  if (on) {
    x[0] = *reinterpret_cast<const unsigned int*>(reinterpret_cast<const bf16*>(a.z) + row * a.ldz + c);
    w = *reinterpret_cast<const uint4*>(reinterpret_cast<const bf16*>(a.cw) + (long long)c * TAPS);
  } else if (wave >= 4) {
    const bf16 *g = reinterpret_cast<const bf16*>(a.gx) + row * a.ldgx, *w0 = reinterpret_cast<const bf16*>(a.gw) + (long long)h * a.gd,
               *w1 = w0 + (long long)a.H * a.gd;
    for (int i = 8 * (tid - 256); i < a.gd; i += 8 * 256) {
      float gv[8], wv[8], uv[8];
      load8(g + i, gv);
      load8(w0 + i, wv);
      if constexpr (!CHANNEL) load8(w1 + i, uv);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        d0 += gv[j] * wv[j];
        if constexpr (!CHANNEL) d1 += gv[j] * uv[j];
      }
    }
  }
  const float rate = expf(a.A_log[h]);
  float nw = 0.f, gate = 0.f;
  if (tid < P) {
    nw = a.w[tid];
    if constexpr (!CHANNEL) gate = (float)reinterpret_cast<const bf16*>(a.gate)[row * a.ldg + (long long)h * P + tid];
  }
  // low-rank factors: tiles of 16 channels, a wave one of the decays' and PQ / 32 of the gate's (of 64 columns half the waves)
  constexpr int FK = CHANNEL > 0 ? CHANNEL : 1, GT = CHANNEL ? (PQ + 31) / 32 : 1;
  Pack8 fa[FK], fg[GT][FK], xa[FK], xg[FK];
  f32x4 za = {0.f, 0.f, 0.f, 0.f}, zg[GT];
  const bool gated = GT * 32 <= PQ || wave < 4;
  if constexpr (CHANNEL != 0) {
    const int r16 = lane & 15, k8 = 8 * (lane >> 4);
    const bf16 *a1 = reinterpret_cast<const bf16*>(a.a1) + row * a.lda1 + k8, *g1 = reinterpret_cast<const bf16*>(a.gate) + row * a.ldg + k8;
    const bf16* a2 = reinterpret_cast<const bf16*>(a.a2) + ((long long)h * N + 16 * wave + r16) * a.rank + k8;
    const bf16* g2[GT];
#pragma unroll
    for (int t = 0; t < GT; ++t)
      g2[t] = reinterpret_cast<const bf16*>(a.g2) + ((long long)h * P + 16 * (gated ? NW * t + wave : 0) + r16) * a.grank + k8;
    auto at = [](const bf16* p) {
      Pack8 v;
      v.u = *reinterpret_cast<const uint4*>(p);
      return v;
    };
#pragma unroll
    for (int t = 0; t < GT; ++t) zg[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    if constexpr (CHANNEL > 0) {
      const Pack8 none = {.u = {0, 0, 0, 0}};
#pragma unroll
      for (int k = 0; k < FK; ++k) {
        const bool ina = 32 * k < a.rank, ing = 32 * k < a.grank;
        xa[k] = ina ? at(a1 + 32 * k) : none;
        fa[k] = ina ? at(a2 + 32 * k) : none;
        xg[k] = ing ? at(g1 + 32 * k) : none;
#pragma unroll
        for (int t = 0; t < GT; ++t) fg[t][k] = ing ? at(g2[t] + 32 * k) : none;
      }
    } else {
      for (int k = 0; k < a.rank; k += 32) za = mfma16(at(a2 + k).v, at(a1 + k).v, za);
      for (int k = 0; k < a.grank; k += 32)
#pragma unroll
        for (int t = 0; t < GT; ++t) zg[t] = mfma16(at(g2[t] + k).v, at(g1 + k).v, zg[t]);
    }
  }
  const int pr = a.prev_row[row], sv = a.save_slot[row];
  if (on && pr <= -2) {
    const bf16* st = reinterpret_cast<const bf16*>(a.conv) + (long long)(-(pr + 2)) * a.conv_stride + c;
#pragma unroll
    for (int b = 1; b < TAPS; ++b) x[b] = *reinterpret_cast<const unsigned int*>(st + (TAPS - 1 - b) * C);
  }
  const long long head = ((long long)h * N + n0) * P + 4 * cq;
  f32x4 S[RL];
  if (pr <= -2) {
    const float* st = a.state + (long long)(-(pr + 2)) * a.state_stride + head;
#pragma unroll
    for (int i = 0; i < RL; ++i) S[i] = *reinterpret_cast<const f32x4*>(st + i * P);
  } else {
#pragma unroll
    for (int i = 0; i < RL; ++i) S[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  __builtin_amdgcn_sched_barrier(0);      // all loads are in flight ahead of what takes them
  if constexpr (CHANNEL != 0) {
    if constexpr (CHANNEL > 0) {
#pragma unroll
      for (int k = 0; k < FK; ++k) {
        za = mfma16(fa[k].v, xa[k].v, za);
#pragma unroll
        for (int t = 0; t < GT; ++t) zg[t] = mfma16(fg[t][k].v, xg[k].v, zg[t]);
      }
    }
    const int m = 4 * (lane >> 4) + (lane & 3);
    if ((lane & 15) < 4) {
      const int n = 16 * wave + m;
      gS[n] = expf(-rate * softplus_exact(own_of(za, lane) + a.dt_bias[h * N + n]));
#pragma unroll
      for (int t = 0; t < GT; ++t)
        if (gated) gateS[16 * (NW * t + wave) + m] = (float)(bf16)own_of(zg[t], lane);
    }
  }
  if (on) {
    const unsigned int wr[2][2] = {{w.x, w.y}, {w.z, w.w}};      // a channel's taps, the oldest input's first
    float y[2] = {0.f, 0.f};
#pragma unroll
    for (int b = 0; b < TAPS; ++b)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int t = TAPS - 1 - b;
        y[i] += (t & 1 ? high16(wr[i][t >> 1]) : low16(wr[i][t >> 1])) * (i ? high16(x[b]) : low16(x[b]));
      }
#pragma unroll
    for (int i = 0; i < 2; ++i) y[i] *= sigmoidf(y[i]);
    if (kind < 2) {
      const float r = 1.f / sqrtf(wave_sum(y[0] * y[0] + y[1] * y[1]) + a.unit_eps) * (kind == 0 ? a.q_scale : 1.f);
      float* to = kind == 0 ? qS : kS;
      to[e] = y[0] * r, to[e + 1] = y[1] * r;
    } else {
      vS[e] = (float)(bf16)y[0], vS[e + 1] = (float)(bf16)y[1];
    }
    if (sv >= 0) {
      bf16* st = reinterpret_cast<bf16*>(a.conv) + (long long)sv * a.conv_stride + c;
#pragma unroll
      for (int b = 0; b < TAPS - 1; ++b) *reinterpret_cast<unsigned int*>(st + (TAPS - 2 - b) * C) = x[b];
    }
  } else if (wave >= 4) {
    d0 = wave_sum(d0);
    if constexpr (!CHANNEL) d1 = wave_sum(d1);
    if (lane == 0) dots[wave - 4] = d0, dots[wave] = d1;
  }
  __syncthreads();
  const float beta = sigmoidf((dots[0] + dots[1]) + (dots[2] + dots[3]));
  float at = 0.f;
  if constexpr (!CHANNEL) at = expf(-rate * softplus_exact((dots[4] + dots[5]) + (dots[6] + dots[7]) + a.dt_bias[h]));
  f32x4 d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < RL; i += 4) {
    const f32x4 k4 = *reinterpret_cast<const f32x4*>(kS + n0 + i);
    const f32x4 g4 = CHANNEL ? *reinterpret_cast<const f32x4*>(gS + n0 + i) : f32x4{at, at, at, at};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      S[i + j] *= g4[j];
      d += S[i + j] * k4[j];
    }
  }
  auto meet = [&](f32x4 v, float (&red)[NW][P]) {
#pragma unroll
    for (int sh = PQ; sh < 64; sh <<= 1)
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] += __shfl_xor(v[i], sh, 64);
    if (lane < PQ) *reinterpret_cast<f32x4*>(red[wave] + 4 * cq) = v;
    __syncthreads();
  };
  meet(d, redk);
  f32x4 u, o = {0.f, 0.f, 0.f, 0.f};
  {
    const auto two = [&](int i) {
      return *reinterpret_cast<const f32x4*>(redk[i] + 4 * cq) + *reinterpret_cast<const f32x4*>(redk[i + 1] + 4 * cq);
    };
    u = beta * (*reinterpret_cast<const f32x4*>(vS + 4 * cq) - ((two(0) + two(2)) + (two(4) + two(6))));
  }
#pragma unroll
  for (int i = 0; i < RL; i += 4) {
    const f32x4 k4 = *reinterpret_cast<const f32x4*>(kS + n0 + i), q4 = *reinterpret_cast<const f32x4*>(qS + n0 + i);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      S[i + j] += k4[j] * u;
      o += S[i + j] * q4[j];
    }
  }
  if (sv >= 0) {
    float* st = a.state + (long long)sv * a.state_stride + head;
#pragma unroll
    for (int i = 0; i < RL; ++i) *reinterpret_cast<f32x4*>(st + i * P) = S[i];
  }
  meet(o, redq);
  float y = 0.f;
  if (tid < P) {
    const auto two = [&](int i) { return redq[i][tid] + redq[i + 1][tid]; };
    y = (two(0) + two(2)) + (two(4) + two(6));
  }
  const float r = 1.f / sqrtf(block_sum<NT>(y * y, scratch) / (float)P + a.eps);
  if (tid >= P) return;
  if constexpr (CHANNEL) gate = sigmoidf(gateS[tid]);
  else gate *= sigmoidf(gate);
  reinterpret_cast<bf16*>(a.out)[((long long)row * a.H + h) * P + tid] = (bf16)(y * r * nw * gate);
}

template <int CHANNEL>
bool by_width(const DeltaTokenArgs& a, hipStream_t s) {
  const dim3 grid(a.H, a.T);
  switch (a.P) {
    case 64: delta_token_kernel<CHANNEL, 16><<<grid, NT, 0, s>>>(a); return true;
    case 128: delta_token_kernel<CHANNEL, 32><<<grid, NT, 0, s>>>(a); return true;
    case 256: delta_token_kernel<CHANNEL, 64><<<grid, NT, 0, s>>>(a); return true;
    default: return false;
  }
}

}  // namespace

bool launch_delta_token(const DeltaTokenArgs& a, hipStream_t s) {
  const auto al = [](const void* p, int to) { return reinterpret_cast<uintptr_t>(p) % to == 0; };
  if (a.N != N || a.taps != TAPS || a.T < 1 || a.T > 65535 || a.H > (1 << 20) / (2 * N + a.P)) return false;
  if (!al(a.z, 4) || a.ldz % 2 || !al(a.cw, 16) || !al(a.conv, 4) || a.conv_stride % 2 || !al(a.state, 16) || a.state_stride % 4 ||
      !al(a.gx, 16) || a.ldgx % 8 || !al(a.gw, 16) || a.gd % 8)
    return false;
  if (!a.a1) return by_width<0>(a, s);
  if (a.rank < 32 || a.rank % 32 || a.rank > 1024 || a.grank < 32 || a.grank % 32 || a.grank > 1024 || !al(a.a1, 16) || a.lda1 % 8 ||
      !al(a.a2, 16) || !al(a.gate, 16) || a.ldg % 8 || !al(a.g2, 16))
    return false;
  return a.rank <= 128 && a.grank <= 128 ? by_width<4>(a, s) : by_width<-1>(a, s);
}
