// Splits weight matrices into the operand order of the split-operand kernels (of3_weight_split.h).
#include "of3_device.h"
#include "of3_split.h"
#include "of3_weight_split.h"

namespace of3 {

namespace {

constexpr int kThreads = 256, kWaves = 4;
constexpr int kAbsent = -(1 << 20);  // the exponent of zero, and of what is no finite number

__device__ __forceinline__ float power_of_two(int e) { return __builtin_ldexpf(1.f, e); }
__device__ __forceinline__ int clamp(int e, int low, int high) { return e < low ? low : e > high ? high : e; }
// the least e with |v| < 2^e
__device__ __forceinline__ int exponent(float v) {
  return v != 0.f && __builtin_fabsf(v) < __builtin_inff() ? __builtin_amdgcn_frexp_expf(v) : kAbsent;
}
__device__ __forceinline__ bool aligned16(const float* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
template <int n>
__device__ __forceinline__ void load(const float* p, bool aligned, float* x) {
  if (aligned) {
#pragma unroll
    for (int e = 0; e < n; e += 4) {
      const float4 v = *reinterpret_cast<const float4*>(p + e);
      x[e] = v.x, x[e + 1] = v.y, x[e + 2] = v.z, x[e + 3] = v.w;
    }
  } else {
#pragma unroll
    for (int e = 0; e < n; ++e) x[e] = p[e];
  }
}

// A row of a matrix [rows][K] behind a LayerNorm, as exponents of two: its own scale, the scale of its inputs, and the bound on its output
// (kAbsent: always zero, or no finite number)
struct Row {
  int weight, input, bound;
};
constexpr int kRowLanes = 4, kItemRows = 64 / kRowLanes;
// of row kItemRows * item + lane / kRowLanes, by one wave
template <int K>
__device__ __forceinline__ Row row_of(const SplitJobs& j, int q, int item) {
  constexpr int kChunks = K / (4 * kRowLanes);
  const int lane = threadIdx.x & 63, part = lane % kRowLanes, norm = j.norm[q];
  int r = kItemRows * item + lane / kRowLanes;
  r = r < j.rows[q] ? r : j.rows[q] - 1;
  const float* src = j.src[q] + (size_t)r * K + 4 * part;
  const float *ln_w = j.ln_w[norm] + 4 * part, *ln_b = j.ln_b[norm] + 4 * part;
  const bool aligned = aligned16(j.src[q]), ln_aligned = aligned16(j.ln_w[norm]) && aligned16(j.ln_b[norm]);
  float x[kChunks][4], w[4], b[4], top = 0.f, top_w = 0.f, top_b = 0.f;
#pragma unroll
  for (int c = 0; c < kChunks; ++c) load<4>(src + 4 * kRowLanes * c, aligned, x[c]);
#pragma unroll
  for (int c = 0; c < kChunks; ++c) {
    load<4>(ln_w + 4 * kRowLanes * c, ln_aligned, w);
    load<4>(ln_b + 4 * kRowLanes * c, ln_aligned, b);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      top = fmaxf(top, __builtin_fabsf(x[c][e]));
      top_w = fmaxf(top_w, __builtin_fabsf(w[e])), top_b = fmaxf(top_b, __builtin_fabsf(b[e]));
    }
  }
  static_assert(kRowLanes == 4, "a quad of lanes");
  auto row_max = [](float v) {
    v = fmaxf(v, dpp_move<0xB1>(v));
    return fmaxf(v, dpp_move<0x4E>(v));
  };
  auto row_sum = [](float v) {
    v += dpp_move<0xB1>(v);
    return v + dpp_move<0x4E>(v);
  };
  top = row_max(top), top_w = row_max(top_w), top_b = row_max(top_b);
  const float root = sqrtf((float)K);
  const int top_e = exponent(top), input_e = exponent(root * top_w + top_b);
  Row row;
  row.weight = top_e == kAbsent ? 80 : clamp(14 - top_e, -110, 80);
  row.input = input_e == kAbsent ? 0 : clamp(14 - input_e, -110, 40);  // 80 + 40: the inverse of the product is a normal number
  const float ws = power_of_two(row.weight), is = power_of_two(row.input);
  float sq = 0.f, dot = 0.f, size = 0.f;
#pragma unroll
  for (int c = 0; c < kChunks; ++c) {
    load<4>(ln_w + 4 * kRowLanes * c, ln_aligned, w);
    load<4>(ln_b + 4 * kRowLanes * c, ln_aligned, b);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float v = x[c][e] * ws, vw = v * (w[e] * is), vb = v * (b[e] * is);
      sq += vw * vw, dot += vb, size += __builtin_fabsf(vb);
    }
  }
  sq = row_sum(sq), dot = row_sum(dot), size = row_sum(size);
  // what rounding leaves of a sum over b that cancels is far below 2^-12 of its terms
  const int bound = exponent(root * sqrtf(sq) + __builtin_fabsf(dot) + 0x1p-12f * size);
  row.bound = top_e == kAbsent || bound == kAbsent ? kAbsent : bound - row.weight - row.input;
  return row;
}

// How a tile of 32 rows is scaled (exponents): the weights and the stored outputs of the lane's row, and what leads from the
// accumulator to these
struct TileScale {
  int weight, output, store;
};
// the rows have one scale
__device__ __forceinline__ TileScale shared_scale(const Row& row, bool logits, int logit_limit) {
  TileScale s;
  s.weight = -wave_max(-row.weight);
  const int bound = wave_max(row.bound);
  s.output = logits && bound != kAbsent ? clamp(14 - bound, -110, logit_limit) : 0;
  s.store = s.output - s.weight - row.input;
  return s;
}
// Or one each: outputs at 2^14, weights as far below 2^14 as that takes with one `store` for all (a wave's rows are in its
// registers: one number in place of 16).  A row that would put the others' weights more than 2^8 lower keeps its own
// and its outputs are lower.
__device__ __forceinline__ TileScale own_scale(const Row& row, int bound) {
  TileScale s;
  const bool live = bound != kAbsent;
  const int want = clamp(14 - bound, -60, 60), lead = want - row.weight - row.input;
  const int most = wave_max(live ? lead : kAbsent), least = -wave_max(live ? -lead : kAbsent);
  s.store = most == kAbsent ? 0 : most < least + 8 ? most : least + 8;
  s.weight = live && want - row.input - s.store < row.weight ? want - row.input - s.store : row.weight;
  // the others give zeros: a scale that takes nothing from the next layer's other columns
  const int top = wave_max(live ? s.weight + row.input + s.store : kAbsent);
  s.output = live ? s.weight + row.input + s.store : top == kAbsent ? 60 : top;
  return s;
}
// of tile t of matrix q, `with`: that of the matrix that its outputs are multiplied with (kUseHidden)
__device__ __forceinline__ TileScale tile_scale(int use, int logit_limit, const Row& row, const Row& with) {
  switch (use) {
    case kUseProduct:
    case kUseValues: return own_scale(row, row.bound);
    case kUseHidden: return own_scale(row, row.bound == kAbsent || with.bound == kAbsent ? kAbsent : row.bound + with.bound);
    default: return shared_scale(row, use == kUseLogits, logit_limit);
  }
}

// of work-group `part`: what is no finite number makes its own products no finite numbers and is left out
__device__ void mask_top(const SplitJobs& j, int part) {
  __shared__ float tops[kWaves];
  const long values = (long)j.B * j.N * j.N;
  float top = 0.f;
  const PairView v = j.mask_view;
  // values one behind the other, in whatever order: eight loads of 16 bytes of a thread in flight (N = 768: the launch 24.4 us with the loop
  // below, 9.7 so, 9.5 without a mask)
  const bool rows = v.stride_k == 1 && v.stride_r == j.N, columns = v.stride_r == 1 && v.stride_k == j.N;
  const bool dense = (rows || columns) && (j.B == 1 || v.stride_b == (int64_t)j.N * j.N) && aligned16(j.mask);
  if (dense) {
    constexpr int kAhead = 8;
    const long chunks = values / 4, step = (long)j.mask_parts * kThreads;
    for (long at = (long)part * kThreads + threadIdx.x; at < chunks; at += kAhead * step) {
      float4 m[kAhead];
#pragma unroll
      for (int e = 0; e < kAhead; ++e) m[e] = reinterpret_cast<const float4*>(j.mask)[at + e * step < chunks ? at + e * step : at];
#pragma unroll
      for (int e = 0; e < kAhead; ++e) {
        const float c[4] = {m[e].x, m[e].y, m[e].z, m[e].w};
#pragma unroll
        for (int k = 0; k < 4; ++k) top = __builtin_fabsf(c[k]) < __builtin_inff() ? fmaxf(top, __builtin_fabsf(c[k])) : top;
      }
    }
    if (part == 0 && 4 * chunks + threadIdx.x < values) {  // up to three more
      const float c = __builtin_fabsf(j.mask[4 * chunks + threadIdx.x]);
      top = c < __builtin_inff() ? fmaxf(top, c) : top;
    }
  }
  auto take = [&](auto number) {
    typedef decltype(number) Index;
    const Index N = j.N, all = values, step = j.mask_parts * kThreads;
#pragma unroll 4
    for (Index at = part * kThreads + threadIdx.x; at < all; at += step) {
      const Index row = at / N, k = at - row * N, b = row / N, r = row - b * N;
      const float m = __builtin_fabsf(j.mask[(long)b * v.stride_b + (long)r * v.stride_r + (long)k * v.stride_k]);
      top = m < __builtin_inff() ? fmaxf(top, m) : top;
    }
  };
  if (!dense && values < 1l << 31) take(0u);  // divisions of 64 bits cost as much as the loads
  else if (!dense) take(0ul);
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) top = fmaxf(top, __shfl_xor(top, d, 64));
  if (threadIdx.x % 64 == 0) tops[threadIdx.x / 64] = top;
  __syncthreads();
  if ((int)threadIdx.x < j.masked) j.mask_top[threadIdx.x]->parts[part] = fmaxf(fmaxf(tops[0], tops[1]), fmaxf(tops[2], tops[3]));
}

// A work-group per tile of 32 rows, or of 32 columns without a LayerNorm before them (fp16 terms), a thread per (row tile,
// step, lane) of it: 8 consecutive k-values, one 16-byte store per term.  fp16 terms: first the bounds of the rows that decide on the
// scales, 16 rows to a wave, four lanes to a row; the matrix then comes from a cache.
__global__ __launch_bounds__(kThreads) void split_weights_f32(SplitJobs j) {
  static_assert(kWaves * kItemRows == 64, "a tile's rows and those that they are multiplied with");
  __shared__ Row bounds[64];
  __shared__ int columns[32];
  __shared__ int tops[kWaves];
  const int tile = blockIdx.x, tid = threadIdx.x;
  if (tile >= j.first[j.n]) return mask_top(j, tile - j.first[j.n]);
  int q = 0, end = j.n;  // the matrix that holds the tile
  while (end - q > 1) {
    const int mid = (q + end) / 2;
    if (tile >= j.first[mid]) q = mid;
    else end = mid;
  }
  const int rows = j.rows[q], K = j.K[q], steps = K / 16, t = tile - j.first[q];
  const int lane = tid & 63, l32 = lane & 31, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool aligned = aligned16(j.src[q]);  // K % 16 == 0: every operand is then 16-byte aligned
  const long plane = packed_elems(rows, K) / 8;
  float x[8];
  auto load_operand = [&](int rt, int s) {
    int row = 32 * rt + l32;
    row = row < rows ? row : rows - 1;  // rows past the end repeat the last one (their results are dropped)
    load<8>(j.src[q] + (size_t)row * K + 16 * s + 8 * (lane >> 5), aligned, x);
  };
  auto operand = [&](int rt, int s) { return reinterpret_cast<u32x4_t*>(j.dst[q]) + ((size_t)rt * steps + s) * 64 + lane; };
  if (j.terms[q] == 3) {
    for (int s = wave; s < steps; s += kWaves) {
      load_operand(t, s);
      u32x4_t h, m, l, *dst = operand(t, s);
      split8(x, h, m, l);
      dst[0] = h;
      dst[plane] = m;
      dst[2 * plane] = l;
    }
    return;
  }
  auto split_store = [&](int rt, int s) {
    u32x4_t h, l, *dst = operand(rt, s);
    split8h(x, h, l);
    dst[0] = h;
    dst[plane] = l;
  };
  WeightScales* out = reinterpret_cast<WeightScales*>(j.dst[q] + 2 * packed_elems(rows, K)) + t;
  const int with = j.with[q];
  const bool normed = j.norm[q] != kNone;
  {
    const int one = normed ? q : with, other = j.use[one] == kUseHidden ? j.with[one] : one, side = wave / 2;
    if (side == 0 || other != one) {
      const int m = side ? other : one, item = 2 * t + wave % 2;
      const Row r = j.K[m] == 128 ? row_of<128>(j, m, item) : row_of<64>(j, m, item);
      if (lane % kRowLanes == 0) bounds[kItemRows * wave + lane / kRowLanes] = r;
    }
    __syncthreads();
    const TileScale scale = tile_scale(j.use[one], j.logit_limit, bounds[l32], bounds[(other != one) * 32 + l32]);
    if (normed) {
      const float ws = power_of_two(scale.weight);
      for (int s = wave; s < steps; s += kWaves) {
        load_operand(t, s);
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] *= ws;
        split_store(t, s);
      }
      if (wave > 0) return;
      const int input = bounds[0].input;
      if (lane < 32) out->rows[lane] = power_of_two(scale.output);
      if (lane == 0) {
        out->unscale = power_of_two(-scale.weight - input);
        out->input = power_of_two(input);
        out->store = power_of_two(scale.store);
        out->output = power_of_two(scale.output);
      }
      return;
    }
    if (tid < 32) columns[tid] = scale.output;
    __syncthreads();
  }
  const int units = 2 * ((rows + 31) / 32), *col = columns + 8 * (lane >> 5);  // a unit: a row tile and one of the two steps
  int top = kAbsent;
  for (int u = wave; u < units; u += kWaves) {
    load_operand(u / 2, 2 * t + u % 2);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int at = exponent(x[e]) - col[16 * (u % 2) + e];
      top = top > at ? top : at;
    }
  }
  top = wave_max(top);
  if (lane == 0) tops[wave] = top;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kWaves; ++w) top = top > tops[w] ? top : tops[w];
  const int scale = top < kAbsent / 2 ? 120 : clamp(14 - top, -120, 120);
  for (int u = wave; u < units; u += kWaves) {
    load_operand(u / 2, 2 * t + u % 2);
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = __builtin_ldexpf(x[e], scale - col[16 * (u % 2) + e]);
    split_store(u / 2, 2 * t + u % 2);
  }
  if (tid == 0) {
    out->unscale = power_of_two(-scale);
    out->input = 1.f;
    out->store = out->output = 0.f;
  }
}

}  // namespace

hipError_t split_weights_launch(const SplitJobs& jobs, hipStream_t stream) {
  hipLaunchKernelGGL(split_weights_f32, dim3((unsigned)(jobs.first[jobs.n] + jobs.mask_parts)), dim3(kThreads), 0, stream, jobs);
  return hipGetLastError();
}

}  // namespace of3
