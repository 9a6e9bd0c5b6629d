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

// row of accumulator register v in lane half lh of a 32 x 32 MFMA result (the lane's column is lane & 31)
__device__ __forceinline__ int acc_row(int v, int lh) { return 8 * (v >> 2) + 4 * lh + (v & 3); }

}  // namespace of3
