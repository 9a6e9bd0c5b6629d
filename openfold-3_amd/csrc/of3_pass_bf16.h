// Building blocks of the bf16 position-wise passes: weight operands (row-major, or packed in operand order by
// weight_pack.hip), LayerNorm lanes, LDS tiles of one 32-position panel.
#pragma once

#include "of3_device.h"
#include "of3_kernels.h"

namespace of3 {
namespace pass_bf16 {

// The lane number, opaque to the compiler: what is derived from it inside a tile loop is recomputed there (a few
// instructions) instead of being hoisted into registers that the weights occupy.
struct Lane {
  int l32, lh;
};
__device__ __forceinline__ Lane lane_here() {
  int lane = threadIdx.x & 63;
  __asm__ volatile("" : "+v"(lane));
  return {lane & 31, lane >> 5};
}

// MFMA operands of output rows 32 t .. + 31 of a matrix with K inputs: this lane takes row r of the tile, k-half lh.
// packed: the 16 bytes of lane l for k-step s of tile t sit at ((t * K / 16 + s) * 64 + l) * 16, one contiguous
// kilobyte per wave instruction; row-major the same operand touches 32 cache lines, and reading a pass's 64 to 128 KB of
// weights that way takes 2 us longer (8.6 against 11.1 us for trimul_proj at N = 40, 15.8 against 18.1 at N = 200).
struct UnitSource {
  const bf16_t* base;
  int step;  // elements between k-steps
};
template <int K>
__device__ __forceinline__ UnitSource unit_source(const bf16_t* W, int t, int r, int lh, int packed) {
  UnitSource u;
  u.base = packed ? W + ((t * (K / 16)) * 64 + r + 32 * lh) * 8 : W + (32 * t + r) * K + 8 * lh;
  u.step = packed ? 512 : 16;
  return u;
}
template <int K>
__device__ __forceinline__ void load_unit(const bf16_t* W, int t, int r, int lh, int packed, u32x4_t (&w)[K / 16]) {
  const UnitSource u = unit_source<K>(W, t, r, lh, packed);
#pragma unroll
  for (int s = 0; s < K / 16; ++s) w[s] = *reinterpret_cast<const u32x4_t*>(u.base + s * u.step);
}

// A lane's part in the LayerNorm of rows of C channels: 16 bytes of one position, C / 8 lanes per position
template <int C>
struct LnLane {
  static constexpr int NCH = C / 8, PPI = 64 / NCH;  // positions per wave instruction
  u32x4_t w, b;
  // chunk and position (inside the PPI of an instruction) of this lane, recomputed where they are used
  __device__ __forceinline__ static int chunk() { return opaque_lane() % NCH; }
  __device__ __forceinline__ static int pos() { return opaque_lane() / NCH; }
  __device__ __forceinline__ static int opaque_lane() {
    int lane = threadIdx.x & 63;
    __asm__ volatile("" : "+v"(lane));
    return lane;
  }
  // Weight and bias unpacked where they are used (16 to 32 instructions) rather than held as 16 floats.  SCALED: the result
  // feeds a gate only, both carry the factor -log2(e) of its base-2 exponential
  template <bool SCALED>
  __device__ __forceinline__ void unpacked(float (&lw)[8], float (&lb)[8]) const {
    u32x4_t tw = w, tb = b;
    __asm__ volatile("" : "+v"(tw), "+v"(tb));
    unpack8(tw, lw);
    unpack8(tb, lb);
    if (SCALED) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        lw[e] *= -kLog2e, lb[e] *= -kLog2e;
        __asm__("" : "+v"(lb[e]));  // rounded here: the fused multiply-add is the one with the weight, as in the 128-position passes
      }
    }
  }
  template <bool SCALED>
  __device__ __forceinline__ u32x4_t normalised(u32x4_t raw) const {
    float lw[8], lb[8];
    unpacked<SCALED>(lw, lb);
    return layer_norm_chunk<C>(raw, lw, lb);
  }
};
template <int C>
__device__ __forceinline__ LnLane<C> ln_lane(const bf16_t* w, const bf16_t* b, int lane) {
  const int chunk = lane % LnLane<C>::NCH;
  LnLane<C> l;
  l.w = *reinterpret_cast<const u32x4_t*>(w + 8 * chunk);
  l.b = *reinterpret_cast<const u32x4_t*>(b + 8 * chunk);
  return l;
}

// LDS tile of 32 positions x C channels, 16-byte chunks.  PERMUTED: operand readers take the positions in rowperm16
// order ({x .. x+3, x+16 .. x+19} per 8 lanes) as well as in natural order, otherwise in natural order only.
template <int C, bool PERMUTED>
struct PanelTile {
  static constexpr int NCH = C / 8, SLOTS = 32 * NCH;
  u32x4_t* s;
  __device__ __forceinline__ static int slot(int pos, int chunk) {
    // 128 channels: a position is one 256-byte bank window; 64: half of one
    int key;
    if (NCH == 16) key = PERMUTED ? (pos & 7) | ((pos ^ (pos >> 1)) & 8) : pos & 15;
    else key = PERMUTED ? ((pos >> 1) & 3) | (((pos >> 2) ^ (pos >> 1)) & 4) : (pos >> 1) & 7;
    return pos * NCH + (chunk ^ key);
  }
};

// 16 consecutive bf16 values
__device__ __forceinline__ void store16(bf16_t* dst, const float (&x)[16]) {
  u32x4_t o0, o1;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    o0[q] = pack_bf16(x[2 * q], x[2 * q + 1]);
    o1[q] = pack_bf16(x[8 + 2 * q], x[8 + 2 * q + 1]);
  }
  *reinterpret_cast<u32x4_t*>(dst) = o0;
  *reinterpret_cast<u32x4_t*>(dst + 8) = o1;
}
__device__ __forceinline__ void add16(const bf16_t* src, float (&x)[16]) {
  float r[8];
  unpack8(*reinterpret_cast<const u32x4_t*>(src), r);
#pragma unroll
  for (int v = 0; v < 8; ++v) x[v] += r[v];
  unpack8(*reinterpret_cast<const u32x4_t*>(src + 8), r);
#pragma unroll
  for (int v = 0; v < 8; ++v) x[8 + v] += r[v];
}

// ---- triangle attention, projections of one panel: kind 0, 1, 2 a 32-channel tile of q, k or v, 3 the triangle bias (4 rows, the
// others of its tile zero)
template <int C>
__device__ __forceinline__ void load_attention_unit(const TriattnProjArgs& p, int kind, int ot, int lane, u32x4_t (&w)[C / 16]) {
  constexpr int H = 4;
  if (kind == 3) {
#pragma unroll
    for (int s = 0; s < C / 16; ++s) {
      w[s] = u32x4_t{0u, 0u, 0u, 0u};
      if ((lane & 31) < H) w[s] = *reinterpret_cast<const u32x4_t*>(p.w_b + (lane & 31) * C + 16 * s + 8 * (lane >> 5));
    }
  } else {
    load_unit<C>(kind == 0 ? p.w_q : kind == 1 ? p.w_k : p.w_v, ot, kind == 2 ? lane & 31 : rowperm16(lane & 31), lane >> 5, p.packed, w);
  }
}
// products and stores of the wave for the normalised positions j0 .. j0 + 31 of row bi
template <int C, int D>
__device__ __forceinline__ void project_panel(const TriattnProjArgs& p, const u32x4_t (&w)[C / 16], const PanelTile<C, true>& tile, int kind,
                                              int ot, int bi, int j0) {
  typedef PanelTile<C, true> Tile;
  constexpr int H = 4, KS = C / 16;
  const int N = p.N, Jp = p.Jp;
  const float qscale = kLog2e * __builtin_amdgcn_rsqf((float)D);
  const Lane at = lane_here();
  const int l32 = at.l32, lh = at.lh;
  f32x16_t acc = zero16();
  float res[16];
  bf16_t* dst;
  if (kind == 3) {
#pragma unroll
    for (int s = 0; s < KS; ++s) acc = mfma_32x32x16(w[s], tile.s[Tile::slot(l32, 2 * s + lh)], acc);
    if (lh == 0) {  // rows 0..3 of the result: registers 0..3 of lanes 0..31
      const int b = bi / N, i = bi - b * N, j = j0 + l32;
#pragma unroll
      for (int h = 0; h < H; ++h) p.tbias[(((size_t)b * H + h) * N + i) * Jp + j] = j < N ? acc[h] * kLog2e : 0.f;
    }
    return;
  }
  if (kind == 2) {
    // V^T panel: rows = keys (dealt by rowperm16), columns = channels; lane: channel 32 ot + l32, keys 16 lh + v
    const int kpos = rowperm16(l32);
#pragma unroll
    for (int s = 0; s < KS; ++s) acc = mfma_32x32x16(tile.s[Tile::slot(kpos, 2 * s + lh)], w[s], acc);
    const int ch = 32 * ot + l32, head = ch / D, d = ch % D;
#pragma unroll
    for (int v = 0; v < 16; ++v) res[v] = acc[v];
    dst = p.vt + ((size_t)bi * H + head) * D * Jp + (size_t)(j0 >> 5) * (D * 32) + d * 32 + 16 * lh;
  } else {
#pragma unroll
    for (int s = 0; s < KS; ++s) acc = mfma_32x32x16(w[s], tile.s[Tile::slot(l32, 2 * s + lh)], acc);
    const int ch0 = 32 * ot + 16 * lh, head = ch0 / D, d0 = ch0 % D;
    const float sc = kind == 0 ? qscale : 1.f;
#pragma unroll
    for (int v = 0; v < 16; ++v) res[v] = acc[v] * sc;
    dst = (kind == 0 ? p.q : p.k) + (((size_t)bi * H + head) * Jp + j0 + l32) * D + d0;
  }
  store16(dst, res);
}
// log2(e) times the mask bias of position j of row bi
__device__ __forceinline__ void store_mask_bias(const TriattnProjArgs& p, int bi, int j, float mask) {
  p.mbias[(size_t)bi * p.Jp + j] = j < p.N ? kLog2e * (p.inf * (mask - 1.f)) : -__builtin_inff();
}


// n / d for n * d < 2^32 by a multiplication
struct Division {
  int d;
  unsigned inverse;  // 2^32 / d rounded up, 0 for d = 1
  static Division by(int d) { return {d, d == 1 ? 0u : (unsigned)(((1ull << 32) + d - 1) / d)}; }
  __device__ __forceinline__ int quotient(int n) const { return inverse ? (int)__umulhi((unsigned)n, inverse) : n; }
};

// logical number of a work-group: consecutive numbers run on one XCD where the grid deals evenly
__device__ __forceinline__ int grid_slot() {
  return gridDim.x % 8 == 0 ? xcd_logical_block(blockIdx.x, gridDim.x / 8) : blockIdx.x;
}

}  // namespace pass_bf16
}  // namespace of3
