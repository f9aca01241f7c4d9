// K2 + K3: rotary embedding on Q/K fused with the paged KV-cache write.
//
// Input is the QKV projection output (LinOut: bf16 [T][(Hq+2Hkv)*D] or fp32
// split-K slabs), so the split-K reduce of the decode QKV GEMM happens here.
// Outputs:
//   q_out   bf16 [T][Hq][D]            rotated queries
//   k_cache bf16 [NB][Hkv][BS][D]      token-major K blocks (rotated)
//   v_cache bf16 [NB][Hkv][D][BS]      dim-major ("transposed") V blocks
// The V layout makes the P.V MFMA B-operand (8 consecutive tokens of one
// dim) a single 16-byte load in the attention kernels.
// rotate_half (NeoX/Llama) convention; cos/sin come from a host-built fp32
// table [max_pos][D] = [cos(0..D/2) | sin(0..D/2)] (no device trig).
#include "common.h"
#include "launchers.h"

namespace {

constexpr int NT = 256;

__global__ __launch_bounds__(NT) void rope_cache_kernel(LinOut qkv, const int* __restrict__ positions,
                                                        const int* __restrict__ slots,
                                                        const float* __restrict__ cos_sin,
                                                        bf16* __restrict__ q_out, bf16* __restrict__ k_cache,
                                                        bf16* __restrict__ v_cache, int Hq, int Hkv, int D,
                                                        int BS, int perm) {
  const int t = blockIdx.x;
  const int N = (Hq + 2 * Hkv) * D;
  const long long row = (long long)t * N;
  const int pos = positions[t];
  const int slot = slots ? slots[t] : -1;
  const int half = D / 2;
  const int gpr = half / 8;  // 8-pair groups per head
  const float* cs = cos_sin + (long long)pos * D;
  const int rot_items = (Hq + Hkv) * gpr;
  const int v_items = Hkv * (D / 8);
  // gridDim.y workgroups per row: one item (8 dims of a head) per thread, one load round trip per row
  for (int it = blockIdx.y * NT + threadIdx.x; it < rot_items + v_items; it += gridDim.y * NT) {
    if (it < rot_items) {
      const int h = it / gpr;          // 0..Hq+Hkv-1 (q heads then k heads)
      const int i0 = (it % gpr) * 8;   // pair index within the half
      float x1[8], x2[8], c[8], s[8];
      // perm: rows of a q/k head are stored tile-interleaved (decode layout, decode_gemm.hip):
      // dims i0..i0+7 at 2*i0, dims half+i0.. at 2*i0 + 8
      const int p1 = perm ? 2 * i0 : i0, p2 = perm ? 2 * i0 + 8 : half + i0;
      linout_load8(qkv, row + (long long)h * D + p1, x1);
      linout_load8(qkv, row + (long long)h * D + p2, x2);
      load8f(cs + i0, c);
      load8f(cs + half + i0, s);
      float o1[8], o2[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        o1[j] = x1[j] * c[j] - x2[j] * s[j];
        o2[j] = x2[j] * c[j] + x1[j] * s[j];
      }
      if (h < Hq) {
        bf16* q = q_out + ((long long)t * Hq + h) * D;
        store8(q + i0, o1);
        store8(q + half + i0, o2);
      } else if (slot >= 0) {
        const int kh = h - Hq;
        const long long blk = slot / BS, off = slot % BS;
        bf16* k = k_cache + ((blk * Hkv + kh) * BS + off) * D;
        store8(k + i0, o1);
        store8(k + half + i0, o2);
      }
    } else if (slot >= 0) {
      const int vi = it - rot_items;
      const int kh = vi / (D / 8);
      const int d0 = (vi % (D / 8)) * 8;
      float x[8];
      linout_load8(qkv, row + (long long)(Hq + Hkv + kh) * D + d0, x);
      const long long blk = slot / BS, off = slot % BS;
      bf16* v = v_cache + ((blk * Hkv + kh) * D + d0) * BS + off;
#pragma unroll
      for (int j = 0; j < 8; ++j) v[(long long)j * BS] = (bf16)x[j];
    }
  }
}

// Prefill form, two kinds of workgroups in one launch.
// V (the first nv): 64 tokens x 64 columns through LDS, so that the dim-major cache is written as 16-byte runs of 8 slots, the
// runs of a dim by neighbouring lanes (64 tokens of a block: whole 128-byte lines, by one XCD).  Runs are cut where the SLOTS
// are multiples of 8, so a prompt behind a cached context of any length has them too; tokens outside such a run (ends,
// sequence changes, padding) are written one by one.
// Rotation: one item (8 dim pairs of a head) per thread over all rows.
// Bound by the bytes at long prompts (8100 tokens of 32 + 2 x 8 heads: 60 -> 39 us, from a place that is no multiple of 8
// 101 -> 43) and by one chain of dependent loads at short ones (137 tokens behind 1063, fp32 slabs: 14.9 -> 7.1 us).  Before, a
// workgroup took a row's rotation and then its share of V, and runs only where a group of 8 rows began at a multiple of 8.
constexpr int VT = 64, VC = 64, VST = VC + 2;
typedef bf16 bf16x2 __attribute__((ext_vector_type(2)));

__global__ __launch_bounds__(NT) void rope_cache_prompt_kernel(LinOut qkv, const int* __restrict__ positions,
                                                               const int* __restrict__ slots,
                                                               const float* __restrict__ cos_sin,
                                                               bf16* __restrict__ q_out, bf16* __restrict__ k_cache,
                                                               bf16* __restrict__ v_cache, int T, int Hq, int Hkv,
                                                               int D, int BS, int perm, int nv) {
  const int N = (Hq + 2 * Hkv) * D;
  if ((int)blockIdx.x >= nv) {
    const int half = D / 2, gpr = half / 8, items = (Hq + Hkv) * gpr;
    const unsigned idx = (blockIdx.x - nv) * NT + threadIdx.x;
    const int t = idx / (unsigned)items, it = idx - (unsigned)t * items;
    if (t >= T) return;
    const int h = it / gpr, i0 = (it - h * gpr) * 8;
    const int pos = positions[t], slot = slots ? slots[t] : -1;
    const long long row = (long long)t * N + (long long)h * D;
    float x1[8], x2[8], c[8], sn[8];
    linout_load8(qkv, row + (perm ? 2 * i0 : i0), x1);
    linout_load8(qkv, row + (perm ? 2 * i0 + 8 : half + i0), x2);
    const float* cs = cos_sin + (long long)pos * D + i0;
    load8f(cs, c);
    load8f(cs + half, sn);
    float o1[8], o2[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      o1[j] = x1[j] * c[j] - x2[j] * sn[j];
      o2[j] = x2[j] * c[j] + x1[j] * sn[j];
    }
    bf16* o = q_out + ((long long)t * Hq + h) * D;
    if (h >= Hq) {
      if (slot < 0) return;
      const long long blk = slot / BS, off = slot % BS;
      o = k_cache + ((blk * Hkv + h - Hq) * BS + off) * D;
    }
    store8(o + i0, o1);
    store8(o + half + i0, o2);
    return;
  }
  __shared__ bf16 tile[VT * VST];
  __shared__ int sl[VT], run[VT / 8 + 1];
  const int cols = Hkv * D, nc = (cols + VC - 1) / VC;
  const int t0 = (blockIdx.x / nc) * VT, c0 = (blockIdx.x % nc) * VC, nt = min(VT, T - t0);
  if (threadIdx.x < VT) sl[threadIdx.x] = (int)threadIdx.x < nt ? slots[t0 + threadIdx.x] : -1;
  {
    const int tok = threadIdx.x >> 2, cc = (threadIdx.x & 3) * 16;
    if (tok < nt && c0 + cc < cols) {                      // (columns come in sixteens)
      const long long at = (long long)(t0 + tok) * N + (long long)(Hq + Hkv) * D + c0 + cc;
      float x[16];
      linout_load8(qkv, at, x);
      linout_load8(qkv, at + 8, x + 8);
      bf16* d = tile + tok * VST + cc;
#pragma unroll
      for (int j = 0; j < 16; j += 2) {
        bf16x2 v;
        v[0] = (bf16)x[j], v[1] = (bf16)x[j + 1];
        *reinterpret_cast<bf16x2*>(d + j) = v;
      }
    }
  }
  __syncthreads();
  const int phase = max(sl[0], 0) & 7;                     // run j: tokens 8 j - phase .. + 7
  if (threadIdx.x <= VT / 8) {
    const int s = 8 * threadIdx.x - phase;
    bool r = BS % 8 == 0 && s >= 0 && s + 8 <= nt;
    if (r) {
      const int first = sl[s];
      r = first >= 0 && first % 8 == 0;
      for (int j = 1; j < 8; ++j) r = r && sl[s + j] == first + j;
    }
    run[threadIdx.x] = r;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < (VT / 8 + 1) * VC; i += NT) {
    const int j = i < VT / 8 * VC ? i % (VT / 8) : VT / 8, c = i < VT / 8 * VC ? i / (VT / 8) : i - VT / 8 * VC;
    if (c0 + c >= cols) continue;
    const int kh = (c0 + c) / D, d = (c0 + c) - kh * D, s = 8 * j - phase;
    if (run[j]) {
      const int first = sl[s];
      const long long blk = first / BS, off = first % BS;
      Pack8 v;
#pragma unroll
      for (int e = 0; e < 8; ++e) v.h[e] = tile[(s + e) * VST + c];
      *reinterpret_cast<uint4*>(v_cache + ((blk * Hkv + kh) * D + d) * BS + off) = v.u;
    } else {
      for (int e = max(s, 0); e < min(s + 8, nt); ++e) {
        const int slot = sl[e];
        if (slot < 0) continue;
        const long long blk = slot / BS, off = slot % BS;
        v_cache[((blk * Hkv + kh) * D + d) * BS + off] = tile[e * VST + c];
      }
    }
  }
}

}  // namespace

void launch_rope_cache(LinOut qkv, const int* positions, const int* slots, const float* cos_sin, bf16* q_out,
                       bf16* k_cache, bf16* v_cache, int T, int Hq, int Hkv, int D, int BS, hipStream_t s, int perm,
                       int decode) {
  if (T == 0) return;
  // decode rows belong to different sequences (no V token runs to gain): the per-row kernel with enough
  // workgroups per row that every thread handles one 8-dim item
  const long long rot = (long long)T * (Hq + Hkv) * (D / 16);
  if (!decode && T >= 32 && rot < (1ll << 31)) {
    const int nv = slots ? (T + VT - 1) / VT * ((Hkv * D + VC - 1) / VC) : 0;
    rope_cache_prompt_kernel<<<nv + (unsigned)((rot + NT - 1) / NT), NT, 0, s>>>(
        qkv, positions, slots, cos_sin, q_out, k_cache, v_cache, T, Hq, Hkv, D, BS, perm, nv);
    return;
  }
  const int items = (Hq + Hkv) * (D / 16) + Hkv * (D / 8);
  rope_cache_kernel<<<dim3(T, (items + NT - 1) / NT), NT, 0, s>>>(qkv, positions, slots, cos_sin, q_out, k_cache,
                                                                   v_cache, Hq, Hkv, D, BS, perm);
}
