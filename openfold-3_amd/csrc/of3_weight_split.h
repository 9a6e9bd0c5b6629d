// Weight matrices split into three bf16 terms (of3_split.h) in the order the MFMA operands are read, once per call:
// the 16 bytes lane l needs for k-step s of row tile t of a matrix [rows][K] sit at ((t * K / 16 + s) * 64 + l) * 16
// of each of three planes, rows padded to multiples of 32 (WeightX3).
#pragma once

#include "of3_kernels.h"
#include "of3_pair_f32.h"

namespace of3 {

// Matrices are added one after the other into the workspace, then split by one launch (a launch costs 4 to 5 us
// whatever it splits: a whole block's matrices go together).
struct SplitJobs {
  static constexpr int kBlock = 25, kMax = 4 * kBlock;  // a pair block: 2 x 6 + 2 x 5 + 3
  const float* src[kMax];
  bf16_t* dst[kMax];
  int rows[kMax], K[kMax];
  int first[kMax + 1];  // first item (8 values) of each matrix; first[n] = all items
  int n;
};
hipError_t split_weights_launch(const SplitJobs& jobs, hipStream_t stream);

struct WeightSplitter {
  SplitJobs j;
  bf16_t* w;
  explicit WeightSplitter(void* workspace) : j(), w(static_cast<bf16_t*>(workspace)) {}
  void add(const float* src, int rows, int K, WeightX3& dst) {
    dst.h = w;
    dst.plane = packed_elems(rows, K);
    j.src[j.n] = src;
    j.dst[j.n] = w;
    j.rows[j.n] = rows;
    j.K[j.n] = K;
    j.first[j.n + 1] = j.first[j.n] + (int)(dst.plane / 8);
    ++j.n;
    w += 3 * dst.plane;
  }
  hipError_t launch(hipStream_t stream) const { return split_weights_launch(j, stream); }
};

// which widths run on split operands, and the matrices of each module in the order of its kernels
constexpr int kTrimulMatrices = 6, kTriattnMatrices = 5, kTransitionMatrices = 3;
inline bool trimul_split_widths(long C, long CH) { return C % 16 == 0 && CH % 16 == 0; }
inline bool triattn_split_widths(long C, long H, long D) { return C % 16 == 0 && (H * D) % 16 == 0; }
inline bool transition_split_widths(long C, long HID) { return C % 16 == 0 && HID % 128 == 0; }

inline void trimul_split_jobs(WeightSplitter& s, const TrimulF32Args& a, WeightX3* w) {
  s.add(a.w_ap, a.CH, a.C, w[0]);
  s.add(a.w_ag, a.CH, a.C, w[1]);
  s.add(a.w_bp, a.CH, a.C, w[2]);
  s.add(a.w_bg, a.CH, a.C, w[3]);
  s.add(a.w_g, a.C, a.C, w[4]);
  s.add(a.w_z, a.C, a.CH, w[5]);
}
inline void triattn_split_jobs(WeightSplitter& s, const TriattnF32Args& a, WeightX3* w) {
  const int HD = a.H * a.D;
  s.add(a.w_q, HD, a.C, w[0]);
  s.add(a.w_k, HD, a.C, w[1]);
  s.add(a.w_v, HD, a.C, w[2]);
  s.add(a.w_g, HD, a.C, w[3]);
  s.add(a.w_o, a.C, HD, w[4]);
}
inline void transition_split_jobs(WeightSplitter& s, const TransitionF32Args& a, WeightX3* w) {
  s.add(a.w_a, a.HID, a.C, w[0]);
  s.add(a.w_b, a.HID, a.C, w[1]);
  s.add(a.w_out, a.C, a.HID, w[2]);
}

}  // namespace of3
