// Copies bf16 weight matrices into MFMA operand order (of3_pass_bf16.h), all matrices of a block in one launch.
#include "of3_device.h"
#include "of3_kernels.h"

namespace of3 {

namespace {

constexpr int kThreads = 256;

// one thread per (matrix, row tile, k-step, lane): 16 bytes
__global__ __launch_bounds__(kThreads) void pack_weights(PackJobs j) {
  const int gitem = (int)blockIdx.x * kThreads + (int)threadIdx.x;
  const int wave_item = __builtin_amdgcn_readfirstlane(gitem);  // a matrix is a multiple of 64 items
  if (wave_item >= j.first[j.n]) return;
  int q = 0, end = j.n;  // the matrix that holds the item
  while (end - q > 1) {
    const int mid = (q + end) / 2;
    if (wave_item >= j.first[mid]) q = mid;
    else end = mid;
  }
  const int K = j.K[q], steps = K / 16, item = gitem - j.first[q];
  const int lane = item & 63, ts = item >> 6, s = ts % steps, t = ts / steps;
  reinterpret_cast<u32x4_t*>(j.dst[q])[item] =
      *reinterpret_cast<const u32x4_t*>(j.src[q] + (size_t)(32 * t + (lane & 31)) * K + 16 * s + 8 * (lane >> 5));
}

}  // namespace

hipError_t pack_weights_launch(const PackJobs& jobs, hipStream_t stream) {
  hipLaunchKernelGGL(pack_weights, dim3((unsigned)((jobs.first[jobs.n] + kThreads - 1) / kThreads)), dim3(kThreads), 0, stream, jobs);
  return hipGetLastError();
}

}  // namespace of3
