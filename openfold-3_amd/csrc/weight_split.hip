// Splits weight matrices into the operand order of the split-operand kernels (of3_weight_split.h).
#include "of3_device.h"
#include "of3_split.h"
#include "of3_weight_split.h"

namespace of3 {

namespace {

constexpr int kThreads = 256;

// one thread per (matrix, row tile, step, lane): its 8 consecutive k-values, one 16-byte store per term
__global__ __launch_bounds__(kThreads) void split_weights_f32(SplitJobs j) {
  const int gitem = (int)blockIdx.x * kThreads + (int)threadIdx.x;
  // the 64 items of a wave belong to one matrix (every matrix has a multiple of 64)
  const int wave_item = __builtin_amdgcn_readfirstlane(gitem);
  if (wave_item >= j.first[j.n]) return;
  int q = 0, end = j.n;  // the matrix that holds the item
  while (end - q > 1) {
    const int mid = (q + end) / 2;
    if (wave_item >= j.first[mid]) q = mid;
    else end = mid;
  }
  const int rows = j.rows[q], K = j.K[q], steps = K / 16;
  const int item = gitem - j.first[q];
  const int lane = item & 63, ts = item >> 6;
  const int s = ts % steps, t = ts / steps;
  int row = 32 * t + (lane & 31);
  row = row < rows ? row : rows - 1;  // rows past the end repeat the last one (their results are dropped)
  const float* src = j.src[q] + (size_t)row * K + 16 * s + 8 * (lane >> 5);
  float x[8];
  if ((reinterpret_cast<uintptr_t>(j.src[q]) & 15u) == 0) {  // K % 16 == 0: every operand is then 16-byte aligned
    const float4 u = *reinterpret_cast<const float4*>(src), v = *reinterpret_cast<const float4*>(src + 4);
    x[0] = u.x, x[1] = u.y, x[2] = u.z, x[3] = u.w, x[4] = v.x, x[5] = v.y, x[6] = v.z, x[7] = v.w;
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = src[e];
  }
  u32x4_t h, m, l;
  split8(x, h, m, l);
  u32x4_t* dst = reinterpret_cast<u32x4_t*>(j.dst[q]) + item;
  const long plane = packed_elems(rows, K) / 8;
  dst[0] = h;
  dst[plane] = m;
  dst[2 * plane] = l;
}

}  // namespace

hipError_t split_weights_launch(const SplitJobs& jobs, hipStream_t stream) {
  const int items = jobs.first[jobs.n];
  hipLaunchKernelGGL(split_weights_f32, dim3((unsigned)((items + kThreads - 1) / kThreads)), dim3(kThreads), 0, stream, jobs);
  return hipGetLastError();
}

}  // namespace of3
