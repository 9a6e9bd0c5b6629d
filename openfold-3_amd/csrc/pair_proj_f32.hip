// Two fp32 projections that read a pair tensor once and write little: the pair bias of the attention over s
// (attention_pair_bias.py:151-161) and the tail of the template branch (template_module.py:376, :462-465), at 64 and
// 128 channels; pair_f32.hip has the kernels for every other shape.
//
// Both are bound by their reads (302 MB at N = 768 and C = 128).  Built like the passes of pair_pass_f32.hip: a
// persistent work-group of four waves, tiles of 32 positions, the few weights split in registers once, the next
// tile's rows in flight, several work-groups per CU.
#include "of3_pass_f32.h"

namespace of3 {

namespace {

using namespace pass_f32;

// ---- out[b][h][i][j] = LN(z[b,i,j,:]) . w[h,:], H <= 32: head h is row h of one accumulator tile whose sum over the
// channels is dealt to the four waves and meets in LDS, so that a head's 32 positions leave as one 128-byte store.
// One wave per tile with its LayerNorm in 16 dependent steps (pair_f32.hip): 17 / 62 / 255 us at N = 64 / 384 / 768.
template <int C>
constexpr size_t pair_bias_lds() {
  return (size_t)PassTile<C>::SLOTS * 16 + (4 * 32 * kBiasLd + 2 * C) * sizeof(float);
}
template <int C>
__global__ __launch_bounds__(256, 3) void pair_bias_pass(PairBiasF32Args p, int panels, int total) {
  typedef PassTile<C> Tile;
  constexpr int NW = 4, SPW = C / 16 / NW;  // k-steps per wave
  extern __shared__ u32x4_t lds[];
  const Tile tile = {lds};
  float* part = reinterpret_cast<float*>(lds + Tile::SLOTS);  // [4][32 heads][kBiasLd]
  float* ln = part + 4 * 32 * kBiasLd;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int N = p.N, H = p.H;
  for (int c = tid; c < C; c += 64 * NW) ln[c] = p.ln_w[c], ln[C + c] = p.ln_b ? p.ln_b[c] : 0.f;
  u32x4_t w[SPW][3];
  {
    const int l32 = tid & 31, row = l32 < H ? l32 : H - 1;  // the rows from H on are dropped
#pragma unroll
    for (int s = 0; s < SPW; ++s) split_operand(p.w + (size_t)row * C, SPW * wave + s, (tid >> 5) & 1, w[s]);
  }
  __syncthreads();
  auto row_of = [&](int pn, int& j0) {
    const int bi = pn / panels;
    j0 = 32 * (pn - bi * panels);
    return bi;
  };
  RowRegs<C> raw[2];
  auto load_tile = [&](int pn) {
    const Lane here = lane_here();
    int j0;
    const int bi = row_of(pn, j0), b = bi / N, i = bi - b * N;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      int j = j0 + 4 * (wave + NW * u) + here.lg;
      j = j < N ? j : N - 1;
      load_row<C>(p.z + b * p.z_view.stride_b + i * p.z_view.stride_r + j * p.z_view.stride_k, here.li, raw[u]);
    }
  };
  int pn = grid_slot();
  if (pn < total) load_tile(pn);
  for (; pn < total; pn += gridDim.x) {
    int j0;
    const int bi = row_of(pn, j0), b = bi / N, i = bi - b * N;
    {
      const Lane here = lane_here();
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        float4 y[C / 64];
        norm_row<C>(raw[u], ln, here.li, y);
#pragma unroll
        for (int e = 0; e < C / 64; ++e) tile.store4(4 * (wave + NW * u) + here.lg, here.li + 16 * e, y[e]);
      }
    }
    load_tile(pn + (int)gridDim.x < total ? pn + gridDim.x : pn);
    __syncthreads();  // the tile is complete, and everybody has read the partial tiles before
    {
      const Lane at = lane_here();
      f32x16_t acc = zero16();
#pragma unroll
      for (int s = 0; s < SPW; ++s) {
        const u32x4_t* x = tile.s + Tile::slot(at.l32, 2 * (SPW * wave + s) + at.lh);
        const u32x4_t op[3] = {x[0], x[Tile::PLANE], x[2 * Tile::PLANE]};
        acc = step6<true>(w[s], op, acc);
      }
      // lane (position l32, half lh), register v: head acc_row(v, lh)
      float* mine = part + wave * (32 * kBiasLd) + at.l32;
#pragma unroll
      for (int v = 0; v < 16; ++v)
        if (8 * (v >> 2) < H) mine[acc_row(v, at.lh) * kBiasLd] = acc[v];
    }
    __syncthreads();
    const int j = tid & 31;
    for (int h = tid >> 5; h < H; h += 8) {
      const float* q = part + h * kBiasLd + j;
      const float v = (q[0] + q[32 * kBiasLd]) + (q[2 * 32 * kBiasLd] + q[3 * 32 * kBiasLd]);
      if (j0 + j < N) p.out[(((size_t)b * H + h) * N + i) * N + j0 + j] = v;
    }
  }
}

// ---- out = relu(mean_T LN(t)) W^T over the T templates' planes of 64 channels, 128 outputs: wave = 32 outputs; the
// plain FMA kernel took 160 us for 3 templates of 200^2 positions, at one dot product per thread
constexpr int kTailC = 64, kTailOut = 128;
// 16 outputs of position q from output o0 on with plain fused multiply-adds, for those that are NaN: an infinite or very
// large weight or input has NaN among its three bf16 terms (single_x3_f32.hip).  The sums are kept in the output row, so
// that the kernel needs no registers for them (with 16 more it ran at four work-groups per CU instead of five, 25 us in
// place of 19 for three templates of 200^2).  ln: weights, then biases
__device__ __forceinline__ void plain_tail(const TemplateTailF32Args& p, int b, long q, int o0, const float* ln) {
  constexpr int C = kTailC;
  float* out = p.out + ((size_t)b * p.P + q) * kTailOut + o0;
#pragma unroll 1
  for (int v = 0; v < 16; ++v) out[v] = 0.f;
#pragma unroll 1
  for (int k = 0; k < C; ++k) {
    float x = 0.f;
#pragma unroll 1
    for (int t = 0; t < p.T; ++t) {
      const float* row = p.t + (((size_t)b * p.T + t) * p.P + q) * C;
      if (!p.apply_ln) {
        x += row[k];
        continue;
      }
      float mean = 0.f, var = 0.f;
      for (int c = 0; c < C; ++c) mean += row[c];
      mean *= 1.f / C;
      for (int c = 0; c < C; ++c) var += (row[c] - mean) * (row[c] - mean);
      x += (row[k] - mean) * (1.0f / sqrtf(var * (1.f / C) + kEps)) * ln[k] + ln[C + k];
    }
    x = fmaxf(x / (float)p.T, 0.f);
#pragma unroll 1
    for (int v = 0; v < 16; ++v) out[v] = fmaf(x, p.w[(size_t)(o0 + v) * C + k], out[v]);
  }
}

constexpr size_t kTailLds = (size_t)PassTile<kTailC>::SLOTS * 16 + 2 * kTailC * sizeof(float);
__global__ __launch_bounds__(256, 3) void template_tail_pass(TemplateTailF32Args p, int tiles_per_b, int total) {
  constexpr int C = kTailC, NW = kTailOut / 32, KS = C / 16;
  typedef PassTile<C> Tile;
  extern __shared__ u32x4_t lds[];
  const Tile tile = {lds};
  float* ln = reinterpret_cast<float*>(lds + Tile::SLOTS);
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  if (p.apply_ln)
    for (int c = tid; c < C; c += 64 * NW) ln[c] = p.ln_w[c], ln[C + c] = p.ln_b[c];
  u32x4_t w[KS][3];
#pragma unroll
  for (int s = 0; s < KS; ++s) split_operand(p.w + (size_t)(32 * wave + rowperm16(tid & 31)) * C, s, (tid >> 5) & 1, w[s]);
  __syncthreads();
  RowRegs<C> raw[2];
  auto load_plane = [&](int id, int t) {  // this wave's eight rows of one template's tile
    const Lane here = lane_here();
    const int b = id / tiles_per_b;
    const long p0 = 32L * (id - b * tiles_per_b);
    const float* plane = p.t + ((size_t)b * p.T + t) * p.P * C;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      long q = p0 + 4 * (wave + NW * u) + here.lg;
      q = q < p.P ? q : p.P - 1;
      load_row<C>(plane + q * C, here.li, raw[u]);
    }
  };
  int id = grid_slot();
  if (id < total) load_plane(id, 0);
  for (; id < total; id += gridDim.x) {
    float4 sum[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) sum[u] = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int t = 0; t < p.T; ++t) {  // in template order
      const Lane here = lane_here();
      RowRegs<C> now[2] = {raw[0], raw[1]};
      if (t + 1 < p.T) load_plane(id, t + 1);
      else load_plane(id + (int)gridDim.x < total ? id + gridDim.x : id, 0);
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        float4 y[1] = {now[u].v[0]};
        if (p.apply_ln) norm_row<C>(now[u], ln, here.li, y);
        sum[u].x += y[0].x, sum[u].y += y[0].y, sum[u].z += y[0].z, sum[u].w += y[0].w;
      }
    }
    const float T = (float)p.T;
    {
      const Lane here = lane_here();
#pragma unroll
      for (int u = 0; u < 2; ++u)
        tile.store4(4 * (wave + NW * u) + here.lg, here.li, make_float4(fmaxf(sum[u].x / T, 0.f), fmaxf(sum[u].y / T, 0.f),
                                                                      fmaxf(sum[u].z / T, 0.f), fmaxf(sum[u].w / T, 0.f)));
    }
    __syncthreads();  // the tile is complete
    const f32x16_t acc = unit_product<C, true>(tile, w);
    __syncthreads();  // everybody has read it
    const Lane at = lane_here();
    const int b = id / tiles_per_b;
    const long q = 32L * (id - b * tiles_per_b) + at.l32;
    if (q >= p.P) continue;
    bool again = false;
#pragma unroll
    for (int v = 0; v < 16; ++v) again |= acc[v] != acc[v];
    if (!again) store_row16(nullptr, p.out + ((size_t)b * p.P + q) * kTailOut + 32 * wave + 16 * at.lh, acc, false);
    else plain_tail(p, b, q, 32 * wave + 16 * at.lh, ln);
  }
}

bool aligned16(std::initializer_list<const void*> ptrs) {
  for (const void* q : ptrs)
    if (reinterpret_cast<uintptr_t>(q) % 16 != 0) return false;
  return true;
}

template <int C>
hipError_t launch_pair_bias(const PairBiasF32Args& a, hipStream_t stream) {
  const int panels = (a.N + 31) / 32;
  const int total = a.B * a.N * panels;
  constexpr size_t lds = pair_bias_lds<C>();
  unsigned grid = 0;
  hipError_t e = resident_grid<pair_bias_pass<C>>(256, lds, total, &grid);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(pair_bias_pass<C>, dim3(grid), dim3(256), lds, stream, a, panels, total);
  return hipGetLastError();
}

}  // namespace

bool pair_bias_pass_serves(const PairBiasF32Args& a) {
  return (a.C == 64 || a.C == 128) && a.H <= 32 && aligned16({a.w}) && rows_aligned(a.z, a.z_view) &&
         (long)a.B * a.N * ((a.N + 31) / 32) <= 0x3fffffffL;
}
hipError_t pair_bias_pass_f32(const PairBiasF32Args& a, hipStream_t stream) {
  return a.C == 128 ? launch_pair_bias<128>(a, stream) : launch_pair_bias<64>(a, stream);
}

bool template_tail_pass_serves(const TemplateTailF32Args& a) {
  return a.CT == kTailC && a.CZ == kTailOut && aligned16({a.t, a.w, a.out}) && (long)a.B * ((a.P + 31) / 32) <= 0x3fffffffL;
}
hipError_t template_tail_pass_f32(const TemplateTailF32Args& a, hipStream_t stream) {
  const int tiles_per_b = (int)((a.P + 31) / 32), total = a.B * tiles_per_b;
  unsigned grid = 0;
  hipError_t e = resident_grid<template_tail_pass>(256, kTailLds, total, &grid);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(template_tail_pass, dim3(grid), dim3(256), kTailLds, stream, a, tiles_per_b, total);
  return hipGetLastError();
}

}  // namespace of3
