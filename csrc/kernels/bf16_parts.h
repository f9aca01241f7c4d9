// fp32 operands of v_mfma_f32_16x16x32_bf16 as sums of three bf16 parts: hi = bf16(x), mid = bf16(x - hi), lo = bf16(x - hi - mid)
// hold all of x's 24 bits (of an infinity the parts make NaN); of a product of two such operands the six terms down to 2^-16 of
// the largest are taken: what is left is 2^-24 of it, an fp32 rounding.  3 / 8 of the matrix cycles of v_mfma_f32_16x16x4_f32.
#pragma once
#include "common.h"

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

constexpr float BF16_MAX = 3.3895313892515355e38f;

struct Parts {
  bf16x8 h, m, l;
};

// (two at a time: v_cvt_pk_bf16_f32 rounds a pair, and a bf16 is a float's upper half; 5.5 instructions a number, 9.7 one by one)
// WIDE: numbers past bf16's largest, which would round to an infinity, too (the rest is in the other parts); the chunk walks' states,
// where it costs 1 % of a walk, of all operands 4
template <bool WIDE = false>
SYM_DEV Parts split(f32x4 a, f32x4 b) {
  union {
    unsigned int u[4];
    bf16x8 v;
  } h, m, l;
  auto fit = [](float x) { return WIDE ? __builtin_amdgcn_fmed3f(x, -BF16_MAX, BF16_MAX) : x; };
  auto round2 = [](float x, float y) {
    const bf16x2 p = __builtin_convertvector((f32x2){x, y}, bf16x2);
    return __builtin_bit_cast(unsigned int, p);
  };
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float x = i < 2 ? a[2 * i] : b[2 * i - 4], y = i < 2 ? a[2 * i + 1] : b[2 * i - 3];
    h.u[i] = round2(fit(x), fit(y));
    const float rx = x - __uint_as_float(h.u[i] << 16), ry = y - __uint_as_float(h.u[i] & 0xffff0000u);
    m.u[i] = round2(rx, ry);
    l.u[i] = round2(rx - __uint_as_float(m.u[i] << 16), ry - __uint_as_float(m.u[i] & 0xffff0000u));
  }
  return Parts{h.v, m.v, l.v};
}

// an A operand in the accumulators' contraction order: 4 elements at p, 4 at p + 16
SYM_DEV bf16x8 pair4(const bf16* p) {
  union {
    bf16x8 v;
    uint2 u[2];
  } r;
  r.u[0] = *reinterpret_cast<const uint2*>(p);
  r.u[1] = *reinterpret_cast<const uint2*>(p + 16);
  return r.v;
}

// (chunk_rows: 64-bit products per load and a check each were a third of the walk's vector time)
SYM_DEV uint4 row16(__amdgpu_buffer_rsrc_t r, int off) {
  const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0);
  return make_uint4(v[0], v[1], v[2], v[3]);
}
SYM_DEV f32x4 row16f(__amdgpu_buffer_rsrc_t r, int off) {
  return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}
