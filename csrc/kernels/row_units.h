// Row work of a decode step that more than one launch does: as a launch of its own (hybrid_rows.hip) and beside a weight stream
// that does not read it (row_linear.hip).
#pragma once
#include "common.h"
#include "hybrid_launchers.h"

constexpr int MAX_TAPS = 16;

// qkv_rope_cache of one row by threads first, first + step, ..
template <typename T>
SYM_DEV void qkv_rope_row(const QkvRopeArgs& a, int row, int first, int step) {
  const T* z = reinterpret_cast<const T*>(a.z) + (long long)row * a.ldz;
  const int nq = a.H * a.dk, nk = a.G * a.dk, nv = a.G * a.dv;
  const int rot = 2 * a.pairs;
  const float* cs = a.rope ? a.rope + (long long)a.positions[row] * rot : nullptr;   // [pairs][2]
  const int slot = a.slots[row];
  T* qo = reinterpret_cast<T*>(a.q_out) + (long long)row * nq;
  T* kc = slot >= 0 ? reinterpret_cast<T*>(a.k_cache) + (long long)slot * nk : nullptr;
  T* vc = slot >= 0 ? reinterpret_cast<T*>(a.v_cache) + (long long)slot * nv : nullptr;
  for (int i = first; i < nq + nk; i += step) {
    const int e = i < nq ? i % a.dk : (i - nq) % a.dk;   // entry within its head
    float v = (float)z[i] + (a.bias ? a.bias[i] : 0.f);
    if (e < rot) {
      if (a.half) {                                      // entry e with entry e +- pairs, table pair e mod pairs
        const bool lo = e < a.pairs;
        const int j = lo ? i + a.pairs : i - a.pairs, pi = lo ? e : e - a.pairs;
        const float u = (float)z[j] + (a.bias ? a.bias[j] : 0.f);
        const float c = cs[2 * pi], s = cs[2 * pi + 1];
        v = lo ? v * c - u * s : v * c + u * s;
      } else {
        const int j = i - e + (e ^ 1);                   // the pair's other entry
        const float u = (float)z[j] + (a.bias ? a.bias[j] : 0.f);
        const float c = cs[e & ~1], s = cs[(e & ~1) + 1];
        v = (e & 1) ? v * c + u * s : v * c - u * s;
      }
    }
    if (i < nq) qo[i] = (T)v;
    else if (kc) kc[i - nq] = (T)v;
  }
  if (vc)
    for (int i = first; i < nv; i += step)
      vc[i] = (T)((float)z[nq + nk + i] + (a.bias ? a.bias[nq + nk + i] : 0.f));
}

// causal_conv_silu of channel c of a row that is a run of its own, whose newest inputs move on
template <typename T>
SYM_DEV void conv_silu_save(const ConvArgs& a, int row, int c) {
  const int taps = a.taps, pr = a.prev_row[row];
  const T* st = pr <= -2 ? reinterpret_cast<const T*>(a.state) + (long long)(-(pr + 2)) * a.state_stride : nullptr;
  const T* w = reinterpret_cast<const T*>(a.w) + (long long)c * taps;
  float acc = a.b[c];
  const int sv = a.save_slot[row];
  T old[MAX_TAPS];                     // old[m]: m + 1 positions back
#pragma unroll
  for (int m = 0; m < MAX_TAPS - 1; ++m)
    if (m < taps - 1) old[m] = st ? st[(long long)(taps - 2 - m) * a.C + c] : (T)0.f;
  const T now = reinterpret_cast<const T*>(a.xin)[(long long)row * a.ldx + c];
  acc += (float)w[taps - 1] * (float)now;
#pragma unroll
  for (int m = 0; m < MAX_TAPS - 1; ++m)
    if (m < taps - 1) acc += (float)w[taps - 2 - m] * (float)old[m];
  reinterpret_cast<T*>(a.out)[(long long)row * a.C + c] = (T)(acc * (1.f / (1.f + expf(-acc))));
  if (sv < 0) return;
  T* dst = reinterpret_cast<T*>(a.state) + (long long)sv * a.state_stride + c;
#pragma unroll
  for (int m = 0; m < MAX_TAPS - 1; ++m)
    if (m < taps - 1) dst[(long long)(taps - 2 - m) * a.C] = m == 0 ? now : old[m - 1];
}
