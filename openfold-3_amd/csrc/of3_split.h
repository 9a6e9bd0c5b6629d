// fp32 values split into three bf16 terms, for fp32-grade products on the bf16 matrix instructions:
// x = xh + xm + xl with xh = bf16(x), xm = bf16(x - xh), xl = bf16(x - xh - xm): both differences are
// exact in fp32, so the three terms carry 24 significant bits of x.  A product then is
//     x w = xh wh + xh wm + xm wh + xh wl + xl wh + xm wm + (three terms below 2^-24 |x w|),
// six bf16 MFMA products (exact, summed in fp32) at a sixteenth of the cost of an fp32 MFMA product each:
// 2.7 times less matrix time for the accuracy of an fp32 product.
#pragma once

#include "of3_device.h"

namespace of3 {

struct Split3 {
  bf16_t h, m, l;
};
__device__ __forceinline__ Split3 split3(float v) {
  Split3 s;
  s.h = to_bf16(v);
  const float r1 = v - bf16_to_f32(s.h);
  s.m = to_bf16(r1);
  s.l = to_bf16(r1 - bf16_to_f32(s.m));
  return s;
}

// eight values at once, as three MFMA operands of 8 bf16
__device__ __forceinline__ void split8(const float (&x)[8], u32x4_t& h, u32x4_t& m, u32x4_t& l) {
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    const float a = x[2 * w], b = x[2 * w + 1];
    const uint32_t ph = pack_bf16(a, b);
    const float ra = a - __uint_as_float(ph << 16), rb = b - __uint_as_float(ph & 0xffff0000u);
    const uint32_t pm = pack_bf16(ra, rb);
    const float sa = ra - __uint_as_float(pm << 16), sb = rb - __uint_as_float(pm & 0xffff0000u);
    h[w] = ph;
    m[w] = pm;
    l[w] = pack_bf16(sa, sb);
  }
}

// A mask bias as the matrix instructions can add logits to it: with an even mantissa.  What is negative and far below half of the
// accumulator's last bit is rounded as that half, to the even neighbour: an odd bias of -1e10 lost a last bit, 1024, to every negative logit
// and to no other, and a row of masked keys averaged those that had lost none.
__device__ __forceinline__ float even_bias(float v) { return __uint_as_float(__float_as_uint(v) & ~1u); }

// ---- two fp16 terms -----------------------------------------------------------------------------
// x s = h + l with h = fp16(x s), l = fp16(x s - h) and s a power of two: 22 to 23 significant bits, and three products
//     x w = (l wh + h wl + h wh) / (sx sw)        (l wl is below 2^-22 |x w| and left out)
// instead of six, four bytes per value instead of six.  A rounded operand adds about 2^-24.6 of its value; what fp32
// accumulation adds grows with the number of products summed and is the larger part of either form's error.  Measured
// against float64 on normal operands, relative 2-norm in 1e-8, three bf16 terms | two fp16 terms | plain fp32 fused
// multiply-adds: 32 values summed 6.8 | 9.3 | 10.4, 64 10.9 | 11.3 | 14.3, 128 16.3 | 14.2 | 20.5, 256 23.4 | 19.0 | 28.6, 768 42 | 31 | 50.
// fp16 ends at 65504, so every operand is scaled by a power of two (exact) that a bound on its values allows: of3_weight_split.h.
// Below 2^-3 after scaling the second term is one of fp16's subnormal numbers, 2^-24 apart, and has one bit less for every power
// of two: an operand bounded by 2^14 is held to 2^-39 of the bound, 2^17 of them with all bits.
typedef __attribute__((__vector_size__(8 * sizeof(_Float16)))) _Float16 f16x8_t;
typedef __attribute__((__vector_size__(2 * sizeof(_Float16)))) _Float16 f16x2_t;
__device__ __forceinline__ f32x16_t mfma_32x32x16_f16(u32x4_t a, u32x4_t b, f32x16_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
}
// two values (scaled) as the halves of a word of each term, round to nearest even
__device__ __forceinline__ void split2h(float a, float b, uint32_t& h, uint32_t& l) {
  const f32x2_t x = {a, b};
  const f16x2_t hi = __builtin_convertvector(x, f16x2_t);
  h = __builtin_bit_cast(uint32_t, hi);
  f32x2_t r;  // a - hi[0], b - hi[1], exact (the compiler makes a conversion and a subtraction of it, two instructions each)
  float ra, rb;
  __asm__("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(ra) : "v"(h), "v"(a));
  __asm__("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(rb) : "v"(h), "v"(b));
  r[0] = ra, r[1] = rb;
  l = __builtin_bit_cast(uint32_t, __builtin_convertvector(r, f16x2_t));
}
__device__ __forceinline__ void split8h(const float (&x)[8], u32x4_t& h, u32x4_t& l) {
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    uint32_t a, b;
    split2h(x[2 * w], x[2 * w + 1], a, b);
    h[w] = a, l[w] = b;
  }
}

// row of accumulator register v in lane half lh of a 32 x 32 MFMA result (the lane's column is lane & 31)
__device__ __forceinline__ int acc_row(int v, int lh) { return 8 * (v >> 2) + 4 * lh + (v & 3); }

}  // namespace of3
