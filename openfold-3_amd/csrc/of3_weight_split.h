// Weight matrices split into three bf16 or two fp16 terms (of3_split.h) in the order the MFMA operands are read, once per
// call: the 16 bytes lane l needs for k-step s of row tile t of a matrix [rows][K] sit at ((t * K / 16 + s) * 64 + l) * 16
// of each of the planes, rows padded to multiples of 32 (WeightX3).
//
// fp16 terms: what weights, inputs and outputs are scaled by are powers of two that follow from the parameters alone, before any
// value is known.  A LayerNorm over K channels gives w n + b with |n|_2 <= sqrt(K), so its values are at most
// sqrt(K) max|w| + max|b| and a row W of the next layer gives at most sqrt(K) |W * w|_2 + |W . b|: no finite input can
// overflow.  Both bounds are brought to at most 2^14, and the largest weight likewise.  A value loses bits of its second term
// below 2^-3 (of3_split.h), 2^17 below the bound.  As a rule a LayerNorm's value is 2^-4 of its bound, q, k and v are 2^-4 of
// theirs, a and b 2^-5 (the gate) and the transition's hidden values, whose bound is the product of their factors' bounds, 2^-9.
// What outputs of one row are multiplied with decides how far rows share a scale:
//   a, b         contracted with their own channel only: a scale for each channel
//   v, hidden    the inputs of a next layer without a LayerNorm: a scale for each channel, whose inverse is in that layer's columns.
//                These have a scale for every 32 of them, so that no part of the split waits for another; the layer's kernel
//                lowers its inputs to the smallest of them (column_scales)
//   q, k         summed over a head's channels: one scale for 32 rows
// Looser bounds (max|w| and whole rows) and one scale for all hidden channels cost what the largest bounds lay above the others'.  Relative
// 2-norm of the error of a transition 128 -> 512 -> 128 in 1e-7, so | now (plain fp32 4.1): even parameters 3.2 | 3.2; one LayerNorm weight 30, 100, 300
// times the others and the columns behind it as much smaller 5.5, 72, 1140 | 3.2; three hidden channels 30, 100, 1000 times larger in both factors
// 18, 71, 18200 | 3.2.
#pragma once

#include <cmath>

#include "of3_kernels.h"
#include "of3_pair_f32.h"

namespace of3 {

// Matrices are added one after the other into the workspace, then split by one launch (whatever it splits: a whole block's
// matrices go together).
struct SplitJobs {
  static constexpr int kBlock = 25, kMax = 4 * kBlock;  // a pair block: 2 x 6 + 2 x 5 + 3
  static constexpr int kNorms = 4 * 7;                  // of which 2 x 2, 2 and 1 LayerNorms
  const float* src[kMax];
  bf16_t* dst[kMax];
  const float *ln_w[kNorms], *ln_b[kNorms];
  int first[kMax + 1];  // first tile of each matrix; first[n] = all tiles
  int n, norms;
  uint16_t rows[kMax], K[kMax];
  // norm: the LayerNorm that the inputs come from; with: kUseHidden: the matrix whose outputs are multiplied with this one's, without a
  // LayerNorm: the matrix whose outputs (times something of at most 1) are the inputs
  uint8_t terms[kMax], norm[kMax], use[kMax], with[kMax];
  // a mask [B][N][N] whose largest value is taken by work-groups behind those of the tiles
  const float* mask;
  PairView mask_view;
  int B, N, mask_parts, masked;
  MaskTop* mask_top[kMax / kBlock * 2];
  int logit_limit;  // largest exponent of the scale of q and of k
};
constexpr uint8_t kNone = 255;
// What becomes of a layer's outputs, which decides the scale that they take (fp16 terms only)
enum LayerUse : uint8_t {
  kUsePlain,      // nothing is multiplied with them as terms
  kUseProduct,    // a and b of the triangle multiplication, times a mask of at most 1 (MaskTop)
  kUseLogits,     // q and k: a logit and its biases are scaled by both, so their scale is at most 2^24, less for mask biases beyond
                  // 1e22 (logit_limit)
  kUseValues,     // v
  kUseHidden,     // times silu of the outputs of `with`
};
hipError_t split_weights_launch(const SplitJobs& jobs, hipStream_t stream);

struct WeightSplitter {
  SplitJobs j;
  bf16_t* w;
  int terms = 3;  // of the matrices added next
  uint8_t norm = kNone;
  explicit WeightSplitter(void* workspace) : j(), w(static_cast<bf16_t*>(workspace)) {}
  // the inputs of the matrices added next
  void input(const float* ln_w, const float* ln_b) {
    norm = (uint8_t)j.norms++;
    j.ln_w[norm] = ln_w;
    j.ln_b[norm] = ln_b;
  }
  void no_norm() { norm = kNone; }
  int add(const float* src, int rows, int K, WeightX3& dst, LayerUse use = kUsePlain, int with = kNone) {
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
    j.with[j.n] = (uint8_t)with;
    j.first[j.n + 1] = j.first[j.n] + (with != kNone && norm == kNone && terms == 2 ? K / 32 : (rows + 31) / 32);
    w += 3 * dst.plane;  // room for either form: the scales of two planes lie in the third's
    return j.n++;
  }
  // of a triangle multiplication; all of a launch have the same mask
  void take_mask(const TrimulF32Args& a, const WeightX3& w_ap) {
    j.mask = a.mask;
    j.mask_view = a.mask_view;
    j.B = a.B;
    j.N = a.N;
    j.mask_parts = MaskTop::count(a.mask, a.B, a.N);
    j.mask_top[j.masked++] = MaskTop::of(w_ap);
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
  return (C == 64 || C == 128) && HID % 128 == 0 && HID <= 1024 && B * N * ((N + 31) / 32) <= 0x3fffffffL;
}

inline void trimul_split_jobs(WeightSplitter& s, const TrimulF32Args& a, bool half, WeightX3* w) {
  s.terms = half ? 2 : 3;
  s.input(a.ln_in_w, a.ln_in_b);
  s.add(a.w_ap, a.CH, a.C, w[0], kUseProduct);
  if (half) s.take_mask(a, w[0]);
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
  // inf (mask - 1) times both scales is finite: for masks up to 16 with an inf near fp32's largest number, 2^50 at 1e9
  s.j.logit_limit = (int)std::fmin(24.f, std::floor((122.f - std::log2(std::fmax(a.inf, 1.f))) / 2.f));
  s.add(a.w_q, HD, a.C, w[0], kUseLogits);
  s.add(a.w_k, HD, a.C, w[1], kUseLogits);
  const int v = s.add(a.w_v, HD, a.C, w[2], kUseValues);
  s.add(a.w_g, HD, a.C, w[3]);
  s.no_norm();
  s.add(a.w_o, a.C, HD, w[4], kUsePlain, v);
}
inline void transition_split_jobs(WeightSplitter& s, const TransitionF32Args& a, bool half, WeightX3* w) {
  s.terms = half ? 2 : 3;
  s.input(a.ln_w, a.ln_b);
  const int gate = s.add(a.w_a, a.HID, a.C, w[0]);
  const int hidden = s.add(a.w_b, a.HID, a.C, w[1], kUseHidden, gate);
  s.no_norm();
  s.add(a.w_out, a.C, a.HID, w[2], kUsePlain, hidden);
}

}  // namespace of3
