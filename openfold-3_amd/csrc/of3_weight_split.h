// Weight matrices split into three bf16 or two fp16 terms (of3_split.h) in the order the MFMA operands are read, once per
// call: the 16 bytes lane l needs for k-step s of row tile t of a matrix [rows][K] sit at ((t * K / 16 + s) * 64 + l) * 16
// of each of the planes, rows padded to multiples of 32 (WeightX3).
//
// fp16 terms: the weights of a tile of 32 rows are scaled by the power of two that brings their largest value to at most
// 2^14.  What a layer's inputs and outputs are scaled by follows from the parameters alone, before any value is known:
// a LayerNorm over K channels gives values of at most sqrt(K) max|w| + max|b| and a vector of 2-norm at most
// sqrt(K) (max|w| + max|b|), so a row's output is at most its 2-norm times that.  No finite input can overflow, and
// a value is 2^-4 to 2^-5 of such a bound as a rule: of the 2^38 between 2^14 and where fp16 ends, 23 bits of precision
// are left over 2^9 below that.
#pragma once

#include "of3_kernels.h"
#include "of3_pair_f32.h"

namespace of3 {

// Matrices are added one after the other into the workspace, then split by one launch (a launch costs 4 to 5 us
// whatever it splits: a whole block's matrices go together).
struct SplitJobs {
  static constexpr int kBlock = 25, kMax = 4 * kBlock;  // a pair block: 2 x 6 + 2 x 5 + 3
  static constexpr int kNorms = 4 * 7;                  // of which 2 x 2, 2 and 1 LayerNorms
  const float* src[kMax];
  bf16_t* dst[kMax];
  const float *ln_w[kNorms], *ln_b[kNorms];
  int first[kMax + 1];  // first tile of 32 rows of each matrix; first[n] = all tiles
  int n, norms;
  uint16_t rows[kMax], K[kMax];
  uint8_t terms[kMax], norm[kMax], use[kMax];  // norm: the LayerNorm that the inputs come from, kNoNorm: none
};
constexpr uint8_t kNoNorm = 255;
// What becomes of a layer's outputs, which decides the scale that they take (fp16 terms only)
enum LayerUse : uint8_t {
  kUsePlain,      // nothing is multiplied with them as terms
  kUseProduct,    // a and b of the triangle multiplication, times the mask: bound at 2^8, which leaves masks up to 255
  kUseLogits,     // q and k: bound at 2^14, scale at most 2^24 (a logit and its biases are scaled by both: 2^48, where a mask bias of
                  // -1e9 and far beyond is finite)
  kUseValues,     // v: bound at 2^14
};
hipError_t split_weights_launch(const SplitJobs& jobs, hipStream_t stream);

struct WeightSplitter {
  SplitJobs j;
  bf16_t* w;
  int terms = 3;  // of the matrices added next
  uint8_t norm = kNoNorm;
  explicit WeightSplitter(void* workspace) : j(), w(static_cast<bf16_t*>(workspace)) {}
  // the inputs of the matrices added next
  void input(const float* ln_w, const float* ln_b) {
    norm = (uint8_t)j.norms++;
    j.ln_w[norm] = ln_w;
    j.ln_b[norm] = ln_b;
  }
  void no_norm() { norm = kNoNorm; }
  void add(const float* src, int rows, int K, WeightX3& dst, LayerUse use = kUsePlain) {
    dst.h = w;
    dst.plane = packed_elems(rows, K);
    dst.terms = terms;
    j.src[j.n] = src;
    j.dst[j.n] = w;
    j.rows[j.n] = (uint16_t)rows;
    j.K[j.n] = (uint16_t)K;
    j.terms[j.n] = (uint8_t)terms;
    j.norm[j.n] = norm;
    j.use[j.n] = use;
    j.first[j.n + 1] = j.first[j.n] + (rows + 31) / 32;
    ++j.n;
    w += 3 * dst.plane;  // room for either form: the scales of two planes lie in the third's
  }
  hipError_t launch(hipStream_t stream) const { return split_weights_launch(j, stream); }
};

// which widths run on split operands, and the matrices of each module in the order of its kernels
constexpr int kTrimulMatrices = 6, kTriattnMatrices = 5, kTransitionMatrices = 3;
inline bool trimul_split_widths(long C, long CH) { return C % 16 == 0 && CH % 16 == 0; }
inline bool triattn_split_widths(long C, long H, long D) { return C % 16 == 0 && (H * D) % 16 == 0; }
inline bool transition_split_widths(long C, long HID) { return C % 16 == 0 && HID % 128 == 0; }

// the shapes whose passes hold fp16 terms (pair_pass_f32.hip, transition_f32.hip); the tensors' rows have to be on 16-byte boundaries too,
// and 32 positions of a row or of a column within the 31 bits of a buffer offset
inline bool near_rows(int64_t stride_r, int64_t stride_k) { return stride_r < (1 << 24) && stride_k < (1 << 24); }
inline bool trimul_half_shapes(long B, long N, long C, long CH) {
  const long Np = (N + 31) / 32 * 32;
  return C == CH && (C == 64 || C == 128) && Np * Np * 2 <= 0x7fffffffL && B * (N + 3) * (Np / 32) <= 0x3fffffffL;
}
inline bool triattn_half_shapes(long B, long N, long C, long H, long D) {
  const long Jp = (N + 31) / 32 * 32;
  return H * D == C && (C == 64 || C == 128) && H <= 8 && (D == 32 || (D == 16 && H % 2 == 0)) && N * Jp * 4 <= 0x7fffffffL &&
         B * N * (Jp / 32) <= 0x3fffffffL;
}
inline bool transition_half_shapes(long B, long N, long C, long HID) {
  return (C == 64 || C == 128) && HID % 128 == 0 && B * N * ((N + 31) / 32) <= 0x3fffffffL;
}

inline void trimul_split_jobs(WeightSplitter& s, const TrimulF32Args& a, bool half, WeightX3* w) {
  s.terms = half ? 2 : 3;
  s.input(a.ln_in_w, a.ln_in_b);
  s.add(a.w_ap, a.CH, a.C, w[0], kUseProduct);
  s.add(a.w_ag, a.CH, a.C, w[1]);
  s.add(a.w_bp, a.CH, a.C, w[2], kUseProduct);
  s.add(a.w_bg, a.CH, a.C, w[3]);
  s.add(a.w_g, a.C, a.C, w[4]);
  s.input(a.ln_out_w, a.ln_out_b);
  s.add(a.w_z, a.C, a.CH, w[5]);
}
inline void triattn_split_jobs(WeightSplitter& s, const TriattnF32Args& a, bool half, WeightX3* w) {
  const int HD = a.H * a.D;
  s.terms = half ? 2 : 3;
  s.input(a.ln_w, a.ln_b);
  s.add(a.w_q, HD, a.C, w[0], kUseLogits);
  s.add(a.w_k, HD, a.C, w[1], kUseLogits);
  s.add(a.w_v, HD, a.C, w[2], kUseValues);
  s.add(a.w_g, HD, a.C, w[3]);
  s.no_norm();
  s.add(a.w_o, a.C, HD, w[4]);
}
inline void transition_split_jobs(WeightSplitter& s, const TransitionF32Args& a, bool half, WeightX3* w) {
  s.terms = half ? 2 : 3;
  s.input(a.ln_w, a.ln_b);
  s.add(a.w_a, a.HID, a.C, w[0]);
  s.add(a.w_b, a.HID, a.C, w[1]);
  s.no_norm();
  s.add(a.w_out, a.C, a.HID, w[2]);
}

}  // namespace of3
