// Arguments of the fp32 pair kernels, shared by pair_f32.hip (every shape) and pair_pass_f32.hip (the
// position-wise passes at 64 and 128 channels).
#pragma once

#include "of3_kernels.h"

namespace of3 {

// split, operand-ordered copy of a weight matrix [rows][K]: planes of ceil(rows / 32) * 32 * K values, three of bf16 or
// two of fp16 (of3_split.h); behind the fp16 planes, the scales of each 32 rows
struct WeightScales {
  float unscale;   // from the accumulator to the layer's output, where its rows have one scale (not kUseProduct, kUseValues, kUseHidden);
                   // without a LayerNorm before the layer a tile is 32 columns, and this what its products have to be multiplied with
  float input;     // the scale of the inputs where these come from a LayerNorm (the same for all rows), else 1
  float store;     // from the accumulator to the values that the outputs take as fp16 terms (0: not used as such)
  float output;    // the scale of these, where the rows have one
  float rows[32];  // ... of each row, where they have their own
};
struct WeightX3 {
  const bf16_t* h;
  long plane;
  int terms;
  __device__ __forceinline__ const WeightScales* scales() const { return reinterpret_cast<const WeightScales*>(h + 2 * plane); }
};
// The largest absolute value of a pair mask, as the triangle multiplication's fp16 terms need it: a and b are those of mask 2^-exponent, at
// most 1.  Behind the scales of w_ap: partial maxima from the launch that splits the weights, and the exponent from trimul_proj_pass
// for the contraction.
struct MaskTop {
  static constexpr int kParts = 64;
  int exponent;
  float parts[kParts];
  // work-groups that take them: 1024 values each, four to a thread, until there are 64
  __host__ __device__ static int count(const float* mask, int B, int N) {
    const long n = mask ? ((long)B * N * N + 1023) / 1024 : 0;
    return n < kParts ? (int)n : kParts;
  }
  __host__ __device__ static MaskTop* of(const WeightX3& w_ap) {  // the third plane, of at least 64 x 64 values
    return reinterpret_cast<MaskTop*>(const_cast<bf16_t*>(w_ap.h) + 2 * w_ap.plane + 2048);
  }
};
__host__ __device__ constexpr long packed_elems(long rows, long K) { return (rows + 31) / 32 * 32 * K; }

// Row of a k-panel that holds row r of channel c: the rows of a channel's panels are rotated by 4 c.  A store of the
// projection pass writes 32 channels of one row at once; without the rotation these are Np * Np * 2 bytes apart, at
// the usual lengths a multiple of the memory system's interleave, and all 32 pieces go to one L2 channel
// (N = 768: see trimul_proj_pass).  rot = panel_rotation(c, Np), Np >= 32.
__host__ __device__ inline int panel_rotation(int c, int Np) { return (4 * c) % Np; }
__host__ __device__ inline int panel_row(int r, int rot, int Np) {
  const int s = r + rot;
  return s < Np ? s : s - Np;
}

// ---- triangle multiplication
struct TrimulF32 {
  const float *z, *mask;
  PairView zv, mv;          // view used by the projection pass (swapped for the incoming update)
  PairView zc;              // canonical view (output pass)
  const float *ln_in_w, *ln_in_b, *ln_out_w, *ln_out_b;
  const float *w_ap, *w_ag, *w_bp, *w_bg, *w_g, *w_z;
  WeightX3 s_ap, s_ag, s_bp, s_bg, s_g, s_z;  // split copies (the *_x3 kernels only)
  float *a, *b, *x, *out;
  // a and b as terms (three bf16, or two fp16 of the values times the scales of w_ap's and w_bp's rows) in the k-panel
  // layout (the split-operand contraction only):
  // element (b, c, r, k) of a term sits at ((((b CH + c) Np / 32 + k / 32) Np + panel_row(r, c)) 32 + k % 32,
  // the terms ab_plane elements apart; Np = N rounded up to whole 32-wide panels
  bf16_t *as, *bs;
  long ab_plane;
  int Np;
  int B, N, C, CH, add_residual;
};

// ---- triangle attention
struct TriattnF32 {
  const float *x, *mask;
  PairView xv, mv;
  const float *ln_w, *ln_b, *w_q, *w_k, *w_v, *w_b, *w_g, *w_o;
  WeightX3 s_q, s_k, s_v, s_g, s_o;  // split copies (the *_x3 kernels only)
  float *q, *k, *v, *tb, *o, *out;
  // q, k and v^T as terms (three bf16, or two fp16 of the values times the scale of their weights' outputs) stored as MFMA
  // operands (the split-operand cores only):
  // the 16 bytes of lane l for step s of 32-position tile t of (b, i, h) are slot
  // (((b N + i) H + h) * Jp / 32 + t) * steps + s) * 64 + l of a plane.  q and k have D / 16 steps (16
  // head channels each) and planes of qk_plane elements; v^T always has two steps (16 keys each) of 32
  // rows, the rows from D on being zero, and planes of v_plane elements.  As fp16 terms at D = 16, v^T is one plane: the
  // rows 0 .. 15 of an operand are the first terms, 16 .. 31 the second ones of the same channels.  With fp16 terms tb
  // holds the bias times the scales of q and k, and o is at the scales of v's channels.
  bf16_t *qs, *ks, *vs;
  long qk_plane, v_plane;
  int Jp;  // N rounded up to whole 32-position tiles
  int B, N, C, H, D, add_residual;
  float inf;
};

// position-wise passes with the weights held in registers (pair_pass_f32.hip): which shapes they serve (the
// caller has split the weights and asked for split intermediates), and their launches
bool trimul_pass_serves(const TrimulF32& p);
hipError_t trimul_proj_pass_f32(const TrimulF32& p, hipStream_t stream);
hipError_t trimul_out_pass_f32(const TrimulF32& p, hipStream_t stream);
bool triattn_pass_serves(const TriattnF32& p);
hipError_t triattn_proj_pass_f32(const TriattnF32& p, hipStream_t stream);
hipError_t triattn_core_h2_f32_launch(const TriattnF32& p, hipStream_t stream);  // triattn_core_f32.hip
hipError_t triattn_out_pass_f32(const TriattnF32& p, hipStream_t stream);
// the pair transition likewise (transition_f32.hip)
bool transition_pass_serves(const TransitionF32Args& a);
bool transition_pass_takes(const TransitionF32Args& a);  // a.end, as the beginning of its launch
hipError_t transition_pass_f32(const TransitionF32Args& a, const WeightX3& s_a, const WeightX3& s_b, const WeightX3& s_out,
                               hipStream_t stream);

// projections off a pair tensor (pair_proj_f32.hip)
bool pair_bias_pass_serves(const PairBiasF32Args& a);
hipError_t pair_bias_pass_f32(const PairBiasF32Args& a, hipStream_t stream);
bool template_tail_pass_serves(const TemplateTailF32Args& a);
hipError_t template_tail_pass_f32(const TemplateTailF32Args& a, hipStream_t stream);

}  // namespace of3
