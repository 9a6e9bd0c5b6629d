// Building blocks of the fp32 position-wise passes on split operands (pair_pass_f32.hip, transition_f32.hip,
// pair_proj_f32.hip): LDS tiles of 32 positions in planes of terms, LayerNorm of rows spread over 16 lanes, MFMA steps of
// three (two fp16 terms) or six (three bf16 terms) products.
#pragma once

#include "of3_device.h"
#include "of3_launch.h"
#include "of3_pair_f32.h"
#include "of3_split.h"
#include "of3_weight_split.h"

namespace of3 {
namespace pass_f32 {

constexpr float kEps = 1e-5f;
constexpr float kLog2eF32 = 1.4426950408889634f;
__device__ __forceinline__ float sigmoid_hw_f32(float x) {
  return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-x * kLog2eF32));
}

// of a value still multiplied by 1 / unscale, a power of two
__device__ __forceinline__ float sigmoid_hw_f32(float x, float unscale) {
  return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(x * (-kLog2eF32 * unscale)));
}

// four values as the halves of three MFMA operand chunks
__device__ __forceinline__ void split4(const float4& x, u32x2_t& h, u32x2_t& m, u32x2_t& l) {
  const float v[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
  for (int w = 0; w < 2; ++w) {
    const float a = v[2 * w], b = v[2 * w + 1];
    const uint32_t ph = pack_bf16(a, b);
    const float ra = a - __uint_as_float(ph << 16), rb = b - __uint_as_float(ph & 0xffff0000u);
    const uint32_t pm = pack_bf16(ra, rb);
    h[w] = ph;
    m[w] = pm;
    l[w] = pack_bf16(ra - __uint_as_float(pm << 16), rb - __uint_as_float(pm & 0xffff0000u));
  }
}

// LDS tile of 32 positions x C channels: three planes [position][C / 8 chunks of 8 bf16].  The 16 lanes of a read
// phase hold 16 consecutive positions at one chunk index: the key spreads them over the banks.
template <int C>
struct PassTile {
  static constexpr int NCH = C / 8, PLANE = 32 * NCH, SLOTS = 3 * PLANE;  // in 16-byte slots
  u32x4_t* s;
  __device__ __forceinline__ static int slot(int pos, int chunk) {
    return pos * NCH + (chunk ^ (NCH >= 16 ? (pos & 15) : ((pos >> 1) & 7)));
  }
  // channels 4 c4 .. + 3 of a position
  __device__ __forceinline__ void store4(int pos, int c4, const float4& y) const {
    u32x2_t h, m, l;
    split4(y, h, m, l);
    u32x2_t* d = reinterpret_cast<u32x2_t*>(s) + 2 * slot(pos, c4 >> 1) + (c4 & 1);
    d[0] = h;
    d[2 * PLANE] = m;
    d[4 * PLANE] = l;
  }
  // channels 8 chunk .. + 7
  __device__ __forceinline__ void store8(int pos, int chunk, const float (&y)[8]) const {
    u32x4_t h, m, l;
    split8(y, h, m, l);
    u32x4_t* d = s + slot(pos, chunk);
    d[0] = h;
    d[PLANE] = m;
    d[2 * PLANE] = l;
  }
};

// The same in two planes of fp16 terms, of values already scaled
template <int C>
struct HalfTile {
  static constexpr int NCH = C / 8, PLANE = 32 * NCH, SLOTS = 2 * PLANE;
  u32x4_t* s;
  __device__ __forceinline__ static int slot(int pos, int chunk) { return PassTile<C>::slot(pos, chunk); }
  __device__ __forceinline__ void store4(int pos, int c4, const float4& y) const {
    u32x2_t h, l;
    uint32_t a, b;
    split2h(y.x, y.y, a, b), h[0] = a, l[0] = b;
    split2h(y.z, y.w, a, b), h[1] = a, l[1] = b;
    u32x2_t* d = reinterpret_cast<u32x2_t*>(s) + 2 * slot(pos, c4 >> 1) + (c4 & 1);
    d[0] = h;
    d[2 * PLANE] = l;
  }
  __device__ __forceinline__ void store8(int pos, int chunk, const float (&y)[8]) const {
    u32x4_t h, l;
    split8h(y, h, l);
    u32x4_t* d = s + slot(pos, chunk);
    d[0] = h;
    d[PLANE] = l;
  }
};

// The lane number, opaque to the compiler: what is derived from it inside a tile loop is recomputed there (a few
// instructions) instead of being hoisted into registers that the weights occupy.
struct Lane {
  int l32, lh, li, lg;
};
__device__ __forceinline__ Lane lane_here() {
  int lane = threadIdx.x & 63;
  __asm__ volatile("" : "+v"(lane));
  return {lane & 31, lane >> 5, lane & 15, lane >> 4};
}

// A row of C channels over 16 lanes: lane li holds channels 64 e + 4 li .. + 3 (a wave reads four rows at a time,
// 256 contiguous bytes of each per instruction)
template <int C>
struct RowRegs {
  float4 v[C / 64];
};
template <int C>
__device__ __forceinline__ void load_row(const float* row, int li, RowRegs<C>& r) {
#pragma unroll
  for (int e = 0; e < C / 64; ++e) r.v[e] = *reinterpret_cast<const float4*>(row + 64 * e + 4 * li);
}
// 1 / sqrt(v), v a variance plus eps: the hardware's (1 ulp) and one Newton step, in the place of a correctly rounded root and a correctly rounded
// division, 22 instructions for every row.  Infinity gives 0, NaN NaN.  Error against float64 over 2^-17 ... 2^20,
// rms and largest in 1e-8: 2.8 and 7.4, of the two 3.6 and 8.9.
__device__ __forceinline__ float rsqrt_f32(float v) {
  const float r = __builtin_amdgcn_rsqf(v);
  const float vh = fminf(v, 3.402823466e38f) * (0.5f * r);
  return __builtin_fmaf(r, __builtin_fmaf(-vh, r, 0.5f), r);
}
// LayerNorm of the row (two-pass statistics); ln: LDS, weights [C] then biases [C].  Rows past the end are some real row's or zeros: whoever sums over
// positions leaves them out.
template <int C>
__device__ __forceinline__ void norm_row(const RowRegs<C>& r, const float* ln, int li, float4 (&y)[C / 64]) {
  float s = 0.f;
#pragma unroll
  for (int e = 0; e < C / 64; ++e) s += (r.v[e].x + r.v[e].y) + (r.v[e].z + r.v[e].w);
  const float mean = group_sum<16>(s) * (1.f / C);
  float q = 0.f;
#pragma unroll
  for (int e = 0; e < C / 64; ++e) {
    y[e].x = r.v[e].x - mean, y[e].y = r.v[e].y - mean, y[e].z = r.v[e].z - mean, y[e].w = r.v[e].w - mean;
    q += y[e].x * y[e].x + y[e].y * y[e].y + y[e].z * y[e].z + y[e].w * y[e].w;
  }
  const float rstd = rsqrt_f32(group_sum<16>(q) * (1.f / C) + kEps);
#pragma unroll
  for (int e = 0; e < C / 64; ++e) {
    const float4 w = *reinterpret_cast<const float4*>(ln + 64 * e + 4 * li);
    const float4 b = *reinterpret_cast<const float4*>(ln + C + 64 * e + 4 * li);
    y[e].x = y[e].x * rstd * w.x + b.x;
    y[e].y = y[e].y * rstd * w.y + b.y;
    y[e].z = y[e].z * rstd * w.z + b.z;
    y[e].w = y[e].w * rstd * w.w + b.w;
  }
}

// the split operands of output rows 32 t .. + 31 of a weight matrix with K = C inputs; lane_src: whose packed
// operand this lane takes (its own, or rowperm16's to deal the rows so that a lane ends with 16 consecutive ones)
template <int C, int TERMS>
__device__ __forceinline__ void load_unit(const WeightX3& W, int t, int lane_src, u32x4_t (&w)[C / 16][TERMS]) {
  const u32x4_t* src = reinterpret_cast<const u32x4_t*>(W.h) + (size_t)t * (C / 16) * 64 + lane_src;
#pragma unroll
  for (int s = 0; s < C / 16; ++s)
#pragma unroll
    for (int pl = 0; pl < TERMS; ++pl) w[s][pl] = src[pl * (W.plane / 8) + 64 * s];
}

// the least e with |mask| <= 2^e, of the whole mask: its loads first, what follows from them behind other loads
struct MaskExponent {
  uint32_t part;  // of a non-negative number: ordered as the bits
  int count;
  __device__ __forceinline__ void load(const TrimulF32& p) {
    const int lane = threadIdx.x & 63;
    count = MaskTop::count(p.mask, p.B, p.N);
    part = __float_as_uint(MaskTop::of(p.s_ap)->parts[lane < count ? lane : 0]);
  }
  __device__ __forceinline__ int of_wave() const {
    const int top = count ? wave_max((int)part) : 0;
    return top == 0 ? 0 : __builtin_amdgcn_frexp_expf(__uint_as_float(top - 1));
  }
};

// Layers without a LayerNorm before them (fp16 terms): `total` leads from the accumulator to the output, where the inputs of column
// tile t, at the scales of their channels, are multiplied with at(t) <= 1
struct ColumnScales {
  const WeightScales* s;
  float total;
  // at most 32 tiles; the load first, what follows from it behind other loads
  __device__ __forceinline__ ColumnScales(const WeightX3& W, int tiles) : s(W.scales()) {
    const int l32 = threadIdx.x & 31;
    total = s[l32 < tiles ? l32 : tiles - 1].unscale;
  }
  __device__ __forceinline__ void finish() { total = __int_as_float(wave_max(__float_as_int(total))); }  // positive: ordered as the bits
  __device__ __forceinline__ float of(float unscale) const {  // of a tile, read before any wait: behind one it is a trip to L2 by itself
    return unscale * __uint_as_float(0x7f000000u - __float_as_uint(total));  // 1 / total, a power of two
  }
  __device__ __forceinline__ float at(int t) const { return of(s[t].unscale); }
};

// rows of a fp32 weight matrix as split MFMA operands: k-values 16 s + 8 lh .. + 7 of `row`
__device__ __forceinline__ void split_operand(const float* row, int s, int lh, u32x4_t (&w)[3]) {
  const float4 u = *reinterpret_cast<const float4*>(row + 16 * s + 8 * lh);
  const float4 v = *reinterpret_cast<const float4*>(row + 16 * s + 8 * lh + 4);
  const float x[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
  split8(x, w[0], w[1], w[2]);
}

constexpr int kBiasLd = 36;  // floats per head row of the pair bias's partial tiles

// one k-step: six products, smallest terms first (one chain of dependent MFMAs: two alternating chains were no
// faster, their second accumulator is what some of the kernels spill for).  W_ROWS: the outputs are the MFMA rows,
// otherwise the positions
template <bool W_ROWS>
__device__ __forceinline__ f32x16_t mm(u32x4_t w, u32x4_t x, f32x16_t acc) {
  return W_ROWS ? mfma_32x32x16(w, x, acc) : mfma_32x32x16(x, w, acc);
}
template <bool W_ROWS>
__device__ __forceinline__ f32x16_t step6(const u32x4_t (&w)[3], const u32x4_t (&x)[3], f32x16_t acc) {
  acc = mm<W_ROWS>(w[2], x[0], acc);
  acc = mm<W_ROWS>(w[0], x[2], acc);
  acc = mm<W_ROWS>(w[1], x[1], acc);
  acc = mm<W_ROWS>(w[1], x[0], acc);
  acc = mm<W_ROWS>(w[0], x[1], acc);
  return mm<W_ROWS>(w[0], x[0], acc);
}
// Sum of a product over C channels in fp16 terms, k-step by k-step.  At 64 channels the products with a second term are
// summed apart and added at the end: rounded to the size of their own sum they leave 0.86 of the error (9.8 against 11.3 in
// 1e-8, three bf16 terms 10.9); at 128 channels one sum is below the three terms' error already.
template <bool W_ROWS>
__device__ __forceinline__ f32x16_t mm_f16(u32x4_t w, u32x4_t x, f32x16_t acc) {
  return W_ROWS ? mfma_32x32x16_f16(w, x, acc) : mfma_32x32x16_f16(x, w, acc);
}
template <int C, bool W_ROWS>
struct HalfSum {
  static constexpr bool kApart = C == 64;
  f32x16_t acc = zero16(), low = zero16();
  // one of a k-step's three products, in this order
  __device__ __forceinline__ void term(int i, const u32x4_t (&w)[2], const u32x4_t (&x)[2]) {
    f32x16_t& sum = kApart && i < 2 ? low : acc;
    sum = mm_f16<W_ROWS>(w[i == 0], x[i == 1], sum);
  }
  __device__ __forceinline__ void step(const u32x4_t (&w)[2], const u32x4_t (&x)[2]) {
#pragma unroll
    for (int i = 0; i < 3; ++i) term(i, w, x);
  }
  __device__ __forceinline__ f32x16_t total() const { return kApart ? acc + low : acc; }
};
template <int C, bool W_ROWS>
__device__ __forceinline__ f32x16_t unit_product(const HalfTile<C>& t, const u32x4_t (&w)[C / 16][2]) {
  HalfSum<C, W_ROWS> sum;
  const Lane at = lane_here();
  u32x4_t nxt[2];
  auto read = [&](int s) {
    const u32x4_t* x = t.s + HalfTile<C>::slot(at.l32, 2 * s + at.lh);
    nxt[0] = x[0], nxt[1] = x[HalfTile<C>::PLANE];
  };
  read(0);
#pragma unroll
  for (int s = 0; s < C / 16; ++s) {
    const u32x4_t op[2] = {nxt[0], nxt[1]};
    if (s + 1 < C / 16) read(s + 1);
    __builtin_amdgcn_sched_barrier(0);
    sum.step(w[s], op);
    __builtin_amdgcn_sched_barrier(0);
  }
  return sum.total();
}

template <int C, bool W_ROWS>
__device__ __forceinline__ f32x16_t unit_product(const PassTile<C>& t, const u32x4_t (&w)[C / 16][3]) {
  f32x16_t acc = zero16();
  const Lane at = lane_here();
#pragma unroll
  for (int s = 0; s < C / 16; ++s) {
    const u32x4_t* x = t.s + PassTile<C>::slot(at.l32, 2 * s + at.lh);
    const u32x4_t op[3] = {x[0], x[PassTile<C>::PLANE], x[2 * PassTile<C>::PLANE]};
    acc = step6<W_ROWS>(w[s], op, acc);
  }
  return acc;
}

// Residual and result rows of a tile of 32 positions, 16 channels to a lane, through buffer descriptors: a lane whose position
// lies past the end has an offset past the range, its loads return zeros and its stores are dropped, and without a
// residual so does every load.  No branch lies around them, so the compiler counts what is in flight: a wait for the
// residual leaves the next tile's rows, requested after it, in flight, and a wait for those the stores.
struct Row16 {
  u32x4_t v[4];
};
struct GlobalRows {
  __amdgpu_buffer_rsrc_t z, out;
  __device__ __forceinline__ GlobalRows(const float* zp, float* op, int64_t first, bool add_residual)
      : z(buffer_rsrc(zp + first, add_residual ? 0x7fffffff : 0)), out(buffer_rsrc(op + first, 0x7fffffff)) {}
  // of the lane's position and 16 channels from c0 + 16 (lane half) on; a position's distance to the first one fits 31 bits: rows_aligned
  __device__ __forceinline__ uint32_t offset(int j0, int N, int64_t stride_k, int c0) const {
    const Lane at = lane_here();
    return j0 + at.l32 < N ? (uint32_t)(((uint32_t)at.l32 * (uint32_t)stride_k + c0 + 16 * at.lh) * sizeof(float)) : 0x80000000u;
  }
  __device__ __forceinline__ Row16 load(uint32_t off) const {
    Row16 r;
#pragma unroll
    for (int a = 0; a < 4; ++a) r.v[a] = __builtin_amdgcn_raw_buffer_load_b128(z, off + 16 * a, 0, 0);
    return r;
  }
  __device__ __forceinline__ void store(uint32_t off, const f32x16_t& v, const Row16& res) const {
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      u32x4_t r;
#pragma unroll
      for (int e = 0; e < 4; ++e) r[e] = __float_as_uint(__uint_as_float(res.v[a][e]) + v[4 * a + e]);
      __builtin_amdgcn_raw_buffer_store_b128(r, out, off + 16 * a, 0, 0);
    }
  }
};

// out row (16 channels from op on) = [residual +] v * g
__device__ __forceinline__ void store_row16(const float* zp, float* op, const f32x16_t& v, bool add_residual) {
  float4 z[4];
  if (add_residual) {
#pragma unroll
    for (int a = 0; a < 4; ++a) z[a] = *reinterpret_cast<const float4*>(zp + 4 * a);
  }
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    float4 r = make_float4(v[4 * a], v[4 * a + 1], v[4 * a + 2], v[4 * a + 3]);
    if (add_residual) r.x = z[a].x + r.x, r.y = z[a].y + r.y, r.z = z[a].z + r.z, r.w = z[a].w + r.w;
    *reinterpret_cast<float4*>(op + 4 * a) = r;
  }
}

// 32 fp32 rows in LDS on their way from a tile's residual to its result: put as they were loaded (16 lanes a row), added to by the waves
// that own 32 of their channels each, and stored whole, so that a store instruction writes four rows (256 bytes of each) in
// the place of 16 bytes of 64.  16-byte slots, XOR-swizzled by the position.
template <int C>
struct RowTile {
  static constexpr int ROW = C / 4, SLOTS = 32 * ROW;
  float4* s;
  __device__ __forceinline__ float4& at(int pos, int c4) const { return s[pos * ROW + (c4 ^ (pos & (ROW - 1)))]; }
  __device__ __forceinline__ void put(int pos, int li, const RowRegs<C>& r) const {
#pragma unroll
    for (int e = 0; e < C / 64; ++e) at(pos, 16 * e + li) = r.v[e];
  }
  // the lane's position and 16 channels from 32 ot + 16 (lane half) on
  __device__ __forceinline__ void add(int ot, const f32x16_t& v, bool to_residual) const {
    const Lane here = lane_here();
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      float4& place = at(here.l32, 8 * ot + 4 * here.lh + a);
      float4 r = make_float4(v[4 * a], v[4 * a + 1], v[4 * a + 2], v[4 * a + 3]);
      if (to_residual) {
        const float4 z = place;
        r.x = z.x + r.x, r.y = z.y + r.y, r.z = z.z + r.z, r.w = z.w + r.w;
      }
      place = r;
    }
  }
  __device__ __forceinline__ void store(float* row, int pos, int li) const {
#pragma unroll
    for (int e = 0; e < C / 64; ++e) *reinterpret_cast<float4*>(row + 64 * e + 4 * li) = at(pos, 16 * e + li);
  }
};

// logical number of a work-group: consecutive numbers run on one XCD where the grid deals evenly
__device__ __forceinline__ int grid_slot() {
  return gridDim.x % 8 == 0 ? xcd_logical_block(blockIdx.x, gridDim.x / 8) : blockIdx.x;
}

inline bool rows_aligned(const float* p, const PairView& v) {
  return (reinterpret_cast<uintptr_t>(p) & 15u) == 0 && ((v.stride_b | v.stride_r | v.stride_k) & 3) == 0 && near_rows(v.stride_r, v.stride_k);
}

// persistent grid: what fits the device at once, at most one work-group per tile
template <auto Kern>
hipError_t resident_grid(int threads, size_t lds, long tiles, unsigned* grid) {
  static int cache[kMaxDevices];
  int fit = 0;
  hipError_t e = allow_dynamic_lds<Kern>(lds);
  if (e != hipSuccess) return e;
  e = per_device(
      cache,
      [&](int dev, int* v) {
        int cus = 0, per_cu = 0;
        hipError_t s = cu_count(dev, &cus);
        if (s == hipSuccess) s = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, Kern, threads, lds);
        *v = cus * (per_cu > 0 ? per_cu : 1);
        return s;
      },
      &fit);
  *grid = (unsigned)(tiles < fit ? tiles : fit);
  return e;
}

}  // namespace pass_f32
}  // namespace of3
