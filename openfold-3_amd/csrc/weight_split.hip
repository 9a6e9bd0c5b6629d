// Splits weight matrices into the operand order of the split-operand kernels (of3_weight_split.h).
#include "of3_device.h"
#include "of3_split.h"
#include "of3_weight_split.h"

namespace of3 {

namespace {

constexpr int kThreads = 256;

// the largest power of two s with bound * s <= 2^limit, at most 2^cap (1 where the bound is no finite number)
__device__ __forceinline__ float scale_for(float bound, int limit, int cap) {
  if (!(bound < __builtin_inff())) return 1.f;
  int e = cap;
  if (bound > 0.f) {
    e = limit - __builtin_amdgcn_frexp_expf(bound);
    e = e < cap ? e : cap;
  }
  return __builtin_ldexpf(1.f, e > -110 ? e : -110);
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) v = fmaxf(v, __shfl_xor(v, d, 64));
  return v;
}

// A work-group per tile of 32 rows, a thread per (step, lane) of it: 8 consecutive k-values, one 16-byte store per term.
// fp16 terms: the largest weight first, then the same values again (in L1) scaled and split, with the rows' 2-norms.
// 3 to 5 us whatever it splits, as when it went by single operands.
__global__ __launch_bounds__(kThreads) void split_weights_f32(SplitJobs j) {
  __shared__ float part[4][64];
  __shared__ float tops[4][3];
  const int tile = blockIdx.x, tid = threadIdx.x;
  int q = 0, end = j.n;  // the matrix that holds the tile
  while (end - q > 1) {
    const int mid = (q + end) / 2;
    if (tile >= j.first[mid]) q = mid;
    else end = mid;
  }
  const int rows = j.rows[q], K = j.K[q], steps = K / 16, t = tile - j.first[q];
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int row = 32 * t + (lane & 31);
  row = row < rows ? row : rows - 1;  // rows past the end repeat the last one (their results are dropped)
  const float* src = j.src[q] + (size_t)row * K + 8 * (lane >> 5);
  const bool aligned = (reinterpret_cast<uintptr_t>(j.src[q]) & 15u) == 0;  // K % 16 == 0: every operand is then 16-byte aligned
  auto load = [&](int s, float (&x)[8]) {
    const float* p = src + 16 * s;
    if (aligned) {
      const float4 u = *reinterpret_cast<const float4*>(p), v = *reinterpret_cast<const float4*>(p + 4);
      x[0] = u.x, x[1] = u.y, x[2] = u.z, x[3] = u.w, x[4] = v.x, x[5] = v.y, x[6] = v.z, x[7] = v.w;
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = p[e];
    }
  };
  const long plane = packed_elems(rows, K) / 8;
  u32x4_t* dst = reinterpret_cast<u32x4_t*>(j.dst[q]) + (size_t)t * steps * 64 + lane;
  float x[8];
  if (j.terms[q] == 3) {
    for (int s = wave; s < steps; s += 4) {
      load(s, x);
      u32x4_t h, m, l;
      split8(x, h, m, l);
      dst[64 * s] = h;
      dst[64 * s + plane] = m;
      dst[64 * s + 2 * plane] = l;
    }
    return;
  }
  const int norm = j.norm[q];
  float top = 0.f, top_w = 0.f, top_b = 0.f;
  for (int s = wave; s < steps; s += 4) {
    load(s, x);
#pragma unroll
    for (int e = 0; e < 8; ++e) top = fmaxf(top, __builtin_fabsf(x[e]));
  }
  if (norm != kNoNorm)
    for (int c = tid; c < K; c += kThreads) {
      top_w = fmaxf(top_w, __builtin_fabsf(j.ln_w[norm][c]));
      top_b = fmaxf(top_b, __builtin_fabsf(j.ln_b[norm][c]));
    }
  top = wave_max(top), top_w = wave_max(top_w), top_b = wave_max(top_b);
  if (lane == 0) tops[wave][0] = top, tops[wave][1] = top_w, tops[wave][2] = top_b;
  __syncthreads();
  auto all = [&](int k) { return fmaxf(fmaxf(tops[0][k], tops[1][k]), fmaxf(tops[2][k], tops[3][k])); };
  const float scale = scale_for(all(0), 14, 80);
  float sq = 0.f;
  for (int s = wave; s < steps; s += 4) {
    load(s, x);
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] *= scale, sq += x[e] * x[e];
    u32x4_t h, l;
    split8h(x, h, l);
    dst[64 * s] = h;
    dst[64 * s + plane] = l;
  }
  part[wave][lane] = sq;
  __syncthreads();
  if (wave > 0) return;
  sq = (part[0][lane] + part[1][lane]) + (part[2][lane] + part[3][lane]);
  sq += __shfl_xor(sq, 32, 64);
  const float row_norm = sqrtf(wave_max(sq)) / scale;
  WeightScales sc = {1.f / scale, 1.f, 0.f, 0.f};
  if (norm != kNoNorm) {
    const float root = sqrtf((float)K), input_top = root * all(1) + all(2), input_norm = root * (all(1) + all(2));
    const float bound = row_norm * input_norm;
    sc.input = scale_for(input_top, 14, 40);  // 80 + 40: the inverse of the product is a normal number
    sc.unscale = 1.f / (scale * sc.input);
    sc.output = j.use[q] == kUseProduct ? scale_for(bound, 8, 60) : scale_for(bound, 14, j.use[q] == kUseLogits ? 24 : 60);
    sc.inv_bound = scale_for(bound, 0, 60);
  }
  WeightScales* out = reinterpret_cast<WeightScales*>(j.dst[q] + 2 * packed_elems(rows, K)) + t;
  if (lane == 0) *out = sc;
}

}  // namespace

hipError_t split_weights_launch(const SplitJobs& jobs, hipStream_t stream) {
  hipLaunchKernelGGL(split_weights_f32, dim3((unsigned)jobs.first[jobs.n]), dim3(kThreads), 0, stream, jobs);
  return hipGetLastError();
}

}  // namespace of3
