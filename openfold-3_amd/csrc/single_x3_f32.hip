// fp32 kernels of the single representation on the bf16 matrix instructions (operands split into three
// bf16 terms, of3_split.h): AttentionPairBias of the trunk (attention_pair_bias.py:189-244) and the
// SwiGLU transition over s (transition.py:225-271) at channel counts in multiples of 32 (and head widths
// 8, 16, 24, 32); single_f32.hip serves every other shape with plain FMA kernels.
//
// A few hundred rows of 384 channels are little work (1 to 16 Gflop of products at 768 rows, 10 us of the
// matrix pipes): what bounds these kernels is the latency of one chain load -> LayerNorm -> products ->
// store, and how many compute units the problem reaches.  So a work-group takes one tile of 32 rows x 32
// outputs, its waves share the sum over k (a wave takes every NW-th block of 32 inputs) and their partial
// tiles meet in LDS; 64 rows x 4 * 384 outputs are then 96 work-groups of 4 waves with 3 blocks each.
// The operands are split in registers where they are loaded: lane (row l32, half lh) reads the 16
// consecutive k-values 16 lh .. + 15 of a block (64 bytes, the two halves complete a 128-byte line) as the
// operands of two MFMA steps; weights and rows use the same order of k, which is all a sum over k needs.
// Measured at 64 / 384 / 768 rows, us: see the kernels.
//
// The terms of an infinity, and of a value above the largest bf16 (3.39e38), are an infinity and NaN: an output
// that depends on one comes out as NaN.  Every NaN is therefore computed again with plain fused multiply-adds, in
// the order of single_f32.hip, which keep an infinity; where an operand is NaN itself they give NaN again.
#include "of3_device.h"
#include "of3_kernels.h"
#include "of3_launch.h"
#include "of3_split.h"

namespace of3 {

namespace {

constexpr float kEps = 1e-5f;
constexpr int kPartLd = 36;                 // floats per row of a partial tile in LDS (16-byte aligned rows)
constexpr int kPart = 32 * kPartLd;         // floats per partial tile

__device__ __forceinline__ float sigmoid_f32(float x) { return 1.0f / (1.0f + expf(-x)); }

__device__ __forceinline__ void load16(const float* p, float (&x)[16]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float4 v = *reinterpret_cast<const float4*>(p + 4 * i);
    x[4 * i] = v.x, x[4 * i + 1] = v.y, x[4 * i + 2] = v.z, x[4 * i + 3] = v.w;
  }
}

// one block of 32 inputs: acc[n] (the large terms) and small[n] += W[n]-rows x x-rows.  The weights are the
// MFMA rows: a lane ends with outputs acc_row(v, lh) of row l32.
template <int NT>
__device__ __forceinline__ void block_products(const float (&x)[16], const float (&w)[NT][16], f32x16_t (&acc)[NT],
                                               f32x16_t (&small)[NT]) {
#pragma unroll
  for (int st = 0; st < 2; ++st) {
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = x[8 * st + e];
    u32x4_t x_h, x_m, x_l;
    split8(v, x_h, x_m, x_l);
#pragma unroll
    for (int n = 0; n < NT; ++n) {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = w[n][8 * st + e];
      u32x4_t w_h, w_m, w_l;
      split8(v, w_h, w_m, w_l);
      small[n] = mfma_32x32x16(w_l, x_h, small[n]);
      acc[n] = mfma_32x32x16(w_m, x_h, acc[n]);
      small[n] = mfma_32x32x16(w_h, x_l, small[n]);
      acc[n] = mfma_32x32x16(w_h, x_m, acc[n]);
      small[n] = mfma_32x32x16(w_m, x_m, small[n]);
      acc[n] = mfma_32x32x16(w_h, x_h, acc[n]);
    }
  }
}

// this wave's partial tile n to LDS, [row l32][output]
__device__ __forceinline__ void store_partial(float* part, const f32x16_t& acc, const f32x16_t& small, int l32, int lh) {
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    float4 v;
    v.x = acc[4 * a] + small[4 * a];
    v.y = acc[4 * a + 1] + small[4 * a + 1];
    v.z = acc[4 * a + 2] + small[4 * a + 2];
    v.w = acc[4 * a + 3] + small[4 * a + 3];
    *reinterpret_cast<float4*>(part + l32 * kPartLd + 8 * a + 4 * lh) = v;
  }
}
// outputs 4 c4 .. 4 c4 + 3 of row `row`, summed over the NW waves' partial tiles (stride: floats between them)
template <int NW, int LD = kPartLd>
__device__ __forceinline__ float4 sum_partials(const float* part, int stride, int row, int c4) {
  float4 s = *reinterpret_cast<const float4*>(part + row * LD + 4 * c4);
#pragma unroll
  for (int w = 1; w < NW; ++w) {
    const float4 v = *reinterpret_cast<const float4*>(part + w * stride + row * LD + 4 * c4);
    s.x += v.x, s.y += v.y, s.z += v.z, s.w += v.w;
  }
  return s;
}

__device__ __forceinline__ bool has_nan(const float4& v) { return v.x != v.x || v.y != v.y || v.z != v.z || v.w != v.w; }
// outputs of four rows of W [..][K] for one row of inputs, x(k): inputs 4 k .. + 3
template <class Row>
__device__ __forceinline__ float4 plain_dots(Row&& x, const float* W, int K) {
  float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
  auto add = [](float acc, const float4& a, const float4& w) { return fmaf(a.w, w.w, fmaf(a.z, w.z, fmaf(a.y, w.y, fmaf(a.x, w.x, acc)))); };
  auto weights = [&](int row, int k) { return *reinterpret_cast<const float4*>(W + (size_t)row * K + 4 * k); };
#pragma unroll 1
  for (int k = 0; k < K / 4 && !(s.x != s.x && s.y != s.y && s.z != s.z && s.w != s.w); ++k) {  // NaN stays NaN
    const float4 a = x(k);
    s.x = add(s.x, a, weights(0, k)), s.y = add(s.y, a, weights(1, k)), s.z = add(s.z, a, weights(2, k)), s.w = add(s.w, a, weights(3, k));
  }
  return s;
}

// LayerNorm of rows pos0 .. pos0 + 31 of src [rows][C] times the rows of NT weight matrices (W[n] points at
// the first of the 32 rows): leaves the partial tile of wave w and matrix n in part[(w * NT + n) * kPart].
// The row values stay in registers through the statistics (two-pass, the partial sums of a row meet in
// red[2][kLnWaves][32]); rows past n_rows repeat the last one.  C is a multiple of 32 up to 512.
constexpr int kLnWaves = 4, kLnBlocks = 4;  // 4 waves x 4 blocks x 32 inputs
template <int NT>
__device__ __forceinline__ void ln_products(const float* __restrict__ src, long pos0, long n_rows, int C,
                                            const float* __restrict__ ln_w, const float* __restrict__ ln_b,
                                            const float* const (&W)[NT], float* part, float* red) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, l32 = lane & 31,
            lh = lane >> 5;
  const int blocks = C / 32;
  const int mine = (blocks - wave + kLnWaves - 1) / kLnWaves;  // blocks wave, wave + kLnWaves, ... (may be none)
  const long row = pos0 + l32 < n_rows ? pos0 + l32 : n_rows - 1;
  const float* xp = src + row * C + 32 * wave + 16 * lh;
  float x[kLnBlocks][16];
#pragma unroll
  for (int i = 0; i < kLnBlocks; ++i)
    if (i < mine) load16(xp + 32 * kLnWaves * i, x[i]);
  const long woff = (long)l32 * C + 32 * wave + 16 * lh;
  float w[NT][16], wn[NT][16];
  if (mine > 0) {
#pragma unroll
    for (int n = 0; n < NT; ++n) load16(W[n] + woff, w[n]);
  }
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < kLnBlocks; ++i)
    if (i < mine) {
#pragma unroll
      for (int e = 0; e < 16; ++e) s += x[i][e];
    }
  s += __shfl_xor(s, 32, 64);
  if (lh == 0) red[wave * 32 + l32] = s;
  __syncthreads();
  float mean = 0.f;
#pragma unroll
  for (int q = 0; q < kLnWaves; ++q) mean += red[q * 32 + l32];
  mean /= (float)C;
  s = 0.f;
#pragma unroll
  for (int i = 0; i < kLnBlocks; ++i)
    if (i < mine) {
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        x[i][e] -= mean;
        s += x[i][e] * x[i][e];
      }
    }
  s += __shfl_xor(s, 32, 64);
  if (lh == 0) red[(kLnWaves + wave) * 32 + l32] = s;
  __syncthreads();
  float var = 0.f;
#pragma unroll
  for (int q = 0; q < kLnWaves; ++q) var += red[(kLnWaves + q) * 32 + l32];
  const float rstd = 1.0f / sqrtf(var / (float)C + kEps);

  f32x16_t acc[NT], small[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) acc[n] = small[n] = zero16();
#pragma unroll
  for (int i = 0; i < kLnBlocks; ++i)
    if (i < mine) {
      if (i + 1 < mine) {
#pragma unroll
        for (int n = 0; n < NT; ++n) load16(W[n] + woff + 32 * kLnWaves * (i + 1), wn[n]);
      }
      const int k = 32 * (wave + kLnWaves * i) + 16 * lh;
      float g[16], b[16];
      load16(ln_w + k, g);
      load16(ln_b + k, b);
#pragma unroll
      for (int e = 0; e < 16; ++e) x[i][e] = x[i][e] * rstd * g[e] + b[e];
      block_products<NT>(x[i], w, acc, small);
      if (i + 1 < mine) {
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
          for (int e = 0; e < 16; ++e) w[n][e] = wn[n][e];
      }
    }
#pragma unroll
  for (int n = 0; n < NT; ++n) store_partial(part + (wave * NT + n) * kPart, acc[n], small[n], l32, lh);
  __syncthreads();
}

// the outputs of four rows of W for row pos0 + r (a row that exists) without the matrix instructions; red as ln_products
// has left it
__device__ __forceinline__ float4 ln_plain_dots(const float* __restrict__ src, long pos0, int r, int C, const float* __restrict__ ln_w,
                                                const float* __restrict__ ln_b, const float* W, const float* red) {
  float mean = 0.f, var = 0.f;
#pragma unroll
  for (int q = 0; q < kLnWaves; ++q) mean += red[q * 32 + r], var += red[(kLnWaves + q) * 32 + r];
  mean /= (float)C;
  const float rstd = 1.0f / sqrtf(var / (float)C + kEps);
  const float4* x = reinterpret_cast<const float4*>(src + (pos0 + r) * C);
  const float4 *g = reinterpret_cast<const float4*>(ln_w), *b = reinterpret_cast<const float4*>(ln_b);
  return plain_dots(
      [&](int k) {
        const float4 v = x[k], gk = g[k], bk = b[k];
        return make_float4((v.x - mean) * rstd * gk.x + bk.x, (v.y - mean) * rstd * gk.y + bk.y, (v.z - mean) * rstd * gk.z + bk.z,
                           (v.w - mean) * rstd * gk.w + bk.w);
      },
      W, C);
}

// rows pos0 .. + 31 of src [rows][K] times 32 rows of W [..][K] (W points at the first): the partial tile of
// wave w is left in part[w * kPart].  K a multiple of 32; the next block's operands are in flight meanwhile.
template <int NW>
__device__ __forceinline__ void plain_products(const float* __restrict__ src, long pos0, long n_rows, int K,
                                               const float* __restrict__ W, float* part) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, l32 = lane & 31,
            lh = lane >> 5;
  const int blocks = K / 32;
  const long row = pos0 + l32 < n_rows ? pos0 + l32 : n_rows - 1;
  const float* xp = src + row * K + 16 * lh;
  const float* wp = W + (long)l32 * K + 16 * lh;
  f32x16_t acc[1] = {zero16()}, small[1] = {zero16()};
  float x[16], w[1][16];
  if (wave < blocks) {
    load16(xp + 32 * wave, x);
    load16(wp + 32 * wave, w[0]);
  }
  for (int kb = wave; kb < blocks; kb += NW) {
    const int nb = kb + NW < blocks ? kb + NW : kb;  // the last one is read again: no load under a condition
    float xn[16], wn[16];
    load16(xp + 32 * nb, xn);
    load16(wp + 32 * nb, wn);
    block_products<1>(x, w, acc, small);
#pragma unroll
    for (int e = 0; e < 16; ++e) x[e] = xn[e], w[0][e] = wn[e];
  }
  store_partial(part + wave * kPart, acc[0], small[0], l32, lh);
  __syncthreads();
}

// The same for a tile of 16 rows x 16 outputs: lane (row l16, quarter lq) reads the 8 consecutive k-values 8 lq .. + 7 of a block, the
// operand of one MFMA step, and ends with outputs 4 lq .. + 3 of row l16.
constexpr int kPart16Ld = 20, kPart16 = 16 * kPart16Ld;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4_t;
__device__ __forceinline__ f32x4_t mfma_16x16x32(u32x4_t a, u32x4_t b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}
template <int NW>
__device__ __forceinline__ void plain_products16(const float* __restrict__ src, long pos0, long n_rows, int K,
                                                 const float* __restrict__ W, float* part) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, l16 = lane & 15, lq = lane >> 4;
  const int blocks = K / 32;
  const long row = pos0 + l16 < n_rows ? pos0 + l16 : n_rows - 1;
  const float4* xp = reinterpret_cast<const float4*>(src + row * K + 8 * lq);
  const float4* wp = reinterpret_cast<const float4*>(W + (long)l16 * K + 8 * lq);
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f}, small = acc;
  float4 x[2], w[2];
  auto load = [&](int kb) { x[0] = xp[8 * kb], x[1] = xp[8 * kb + 1], w[0] = wp[8 * kb], w[1] = wp[8 * kb + 1]; };
  if (wave < blocks) load(wave);
  for (int kb = wave; kb < blocks; kb += NW) {
    u32x4_t xo[3], wo[3];
    const float xv[8] = {x[0].x, x[0].y, x[0].z, x[0].w, x[1].x, x[1].y, x[1].z, x[1].w};
    const float wv[8] = {w[0].x, w[0].y, w[0].z, w[0].w, w[1].x, w[1].y, w[1].z, w[1].w};
    load(kb + NW < blocks ? kb + NW : kb);  // the last one is read again: no load under a condition
    split8(xv, xo[0], xo[1], xo[2]);
    split8(wv, wo[0], wo[1], wo[2]);
    small = mfma_16x16x32(wo[2], xo[0], small);
    acc = mfma_16x16x32(wo[1], xo[0], acc);
    small = mfma_16x16x32(wo[0], xo[2], small);
    acc = mfma_16x16x32(wo[0], xo[1], acc);
    small = mfma_16x16x32(wo[1], xo[1], small);
    acc = mfma_16x16x32(wo[0], xo[0], acc);
  }
  *reinterpret_cast<float4*>(part + wave * kPart16 + l16 * kPart16Ld + 4 * lq) =
      make_float4(acc[0] + small[0], acc[1] + small[1], acc[2] + small[2], acc[3] + small[3]);
  __syncthreads();
}

// q (bias added, then / sqrt(D)), k, v and the gate after the sigmoid, all [B*N][H*D]
// (plain FMA kernel 114 / 126 / 187 us at 64 / 384 / 768 rows)
__global__ __launch_bounds__(64 * kLnWaves) void single_proj_x3_f32(SingleAttnF32Args p) {
  __shared__ __align__(16) float part[kLnWaves * kPart];
  __shared__ float red[2 * kLnWaves * 32];
  const long rows = (long)p.B * p.N, pos0 = (long)blockIdx.x * 32;
  const int HD = p.H * p.D, tiles = HD / 32;
  const int kind = blockIdx.y / tiles, o0 = 32 * (blockIdx.y - kind * tiles);
  const float* Wm = kind == 0 ? p.wq : kind == 1 ? p.wk : kind == 2 ? p.wv : p.wg;
  float* dst = kind == 0 ? p.q : kind == 1 ? p.k : kind == 2 ? p.v : p.g;
  const float* const W[1] = {Wm + (size_t)o0 * p.C};
  ln_products<1>(p.a, pos0, rows, p.C, p.ln_w, p.ln_b, W, part, red);
  const int r = threadIdx.x >> 3, c4 = threadIdx.x & 7;
  if (pos0 + r >= rows) return;
  float4 v = sum_partials<kLnWaves>(part, kPart, r, c4);
  if (__builtin_expect(has_nan(v), 0)) v = ln_plain_dots(p.a, pos0, r, p.C, p.ln_w, p.ln_b, W[0] + (size_t)4 * c4 * p.C, red);
  if (kind == 0) {
    const float scale = 1.0f / sqrtf((float)p.D);
    const float* bq = p.bq + o0 + 4 * c4;
    v.x = (v.x + bq[0]) * scale, v.y = (v.y + bq[1]) * scale, v.z = (v.z + bq[2]) * scale, v.w = (v.w + bq[3]) * scale;
  } else if (kind == 3) {
    v.x = sigmoid_f32(v.x), v.y = sigmoid_f32(v.y), v.z = sigmoid_f32(v.z), v.w = sigmoid_f32(v.w);
  }
  *reinterpret_cast<float4*>(dst + (pos0 + r) * HD + o0 + 4 * c4) = v;
}

// exp(x) for x <= 0 (or -inf) from the hardware's exp2: the part of x * log2(e) that one product rounds away
// is carried along and put back (e^(r ln 2) = 1 + r ln 2 for |r| far below 1), so the relative error stays at
// the 1 ulp of the instruction whatever the size of x.  NaN gives NaN: a compare and a select keep -inf out of the
// products, where fmaxf would also turn a NaN logit into the weight 0 of a masked key.
__device__ __forceinline__ float exp_neg(float x) {
  x = x < -1e30f ? -1e30f : x;
  const float t = x * kLog2e;
  const float r = fmaf(x, 1.925963033e-8f, fmaf(x, kLog2e, -t));
  const float e = __builtin_amdgcn_exp2f(t);
  return fmaf(e, r * 0.6931471805599453f, e);
}

// Attention core: work-group = 32 queries of one (batch, head); its four waves take every fourth 32-key tile
// with a running softmax each and merge at the end.  S^T = K Q^T and O^T = V^T P^T as in the pair attention
// (keys, then head channels, are the MFMA rows: a lane holds 16 logits of one query, which are the second
// product's operand).  The head width is padded to 32 channels with zeros.  Logits in the reference's order:
// q.k, then the mask bias, then the pair bias.
// (6.7 / 16.4 us at 64 / 384 tokens; plain FMA kernel 24 / 101 / 200 at 64 / 384 / 768)
constexpr int kAttnWaves = 4;
__global__ __launch_bounds__(64 * kAttnWaves) void single_attn_x3_f32(SingleAttnF32Args p, int pb_vec) {
  __shared__ float merge[kAttnWaves][18][64];
  __shared__ __align__(16) float mbs[kAttnWaves][32];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, l32 = lane & 31, lh = lane >> 5;
  // every pointer and size, asked for at once: one trip to the kernel's arguments instead of three or four in a row
  __asm__ volatile("" ::"s"(p.q), "s"(p.k), "s"(p.v), "s"(p.pair_bias), "s"(p.mask), "s"(p.N), "s"(p.H), "s"(p.D), "s"(p.g), "s"(p.og),
                   "s"(pb_vec));
  const int N = p.N, H = p.H, D = p.D, HD = H * D;
  const int h = blockIdx.y, b = blockIdx.z;
  const int qi = blockIdx.x * 32 + l32;
  const bool q_valid = qi < N;
  const int qrow = q_valid ? qi : N - 1;
  const size_t bN = (size_t)b * N;
  // this lane's 8 channels of step s: 16 s + 8 lh .. + 7 (all inside the head or all outside: D % 8 == 0)
  auto load_row = [&](const float* base, int token, float (&x)[16]) {
    const float* row = base + (bN + token) * HD + h * D;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int d = 16 * s + 8 * lh;
      const float* src = row + (d < D ? d : 0);
      const float4 u = *reinterpret_cast<const float4*>(src), v = *reinterpret_cast<const float4*>(src + 4);
      const float keep = d < D ? 1.f : 0.f;
      x[8 * s] = u.x * keep, x[8 * s + 1] = u.y * keep, x[8 * s + 2] = u.z * keep, x[8 * s + 3] = u.w * keep;
      x[8 * s + 4] = v.x * keep, x[8 * s + 5] = v.y * keep, x[8 * s + 6] = v.z * keep, x[8 * s + 7] = v.w * keep;
    }
  };
  auto split_step = [&](const float (&x)[16], int s, u32x4_t (&op)[3]) {
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = x[8 * s + e];
    split8(v, op[0], op[1], op[2]);
  };
  float xq[16];
  load_row(p.q, qrow, xq);
  const float* pb = p.pair_bias + (((size_t)b * H + h) * N + qrow) * N;
  const float* vcol = p.v + bN * HD + h * D + (l32 < D ? l32 : 0);
  const float vkeep = l32 < D ? 1.f : 0.f;
  const float ninf = -__builtin_inff();

  struct Raw {
    float k[16], v[16], pb[16], mask;
  };
  auto load_tile = [&](int kt, Raw& t) {
    const int k0 = 32 * kt;
    const int key = k0 + l32 < N ? k0 + l32 : N - 1;
    load_row(p.k, key, t.k);
    t.mask = p.mask ? p.mask[bN + key] : 1.f;
#pragma unroll
    for (int a = 0; a < 4; ++a) {  // registers 4 a .. + 3: keys 8 a + 4 lh .. + 3
      const int kk = k0 + 8 * a + 4 * lh;
      if (pb_vec) {  // N % 4 == 0: four keys lie below N or all past it
        const float4 u = *reinterpret_cast<const float4*>(pb + (kk < N ? kk : N - 4));
        t.pb[4 * a] = u.x, t.pb[4 * a + 1] = u.y, t.pb[4 * a + 2] = u.z, t.pb[4 * a + 3] = u.w;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) t.pb[4 * a + e] = pb[kk + e < N ? kk + e : N - 1];
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) t.v[4 * a + e] = vcol[(size_t)(kk + e < N ? kk + e : N - 1) * HD];
    }
  };

  float m_run = ninf, l_run = 0.f;
  f32x16_t oacc = zero16(), osmall = zero16();
  const int nkt = (N + 31) / 32;
  Raw cur, nxt;
  if (wave < nkt) load_tile(wave, cur);
  u32x4_t qop[2][3];  // split behind the first tile's loads, which are under way while the query arrives
  split_step(xq, 0, qop[0]);
  split_step(xq, 1, qop[1]);
  for (int kt = wave; kt < nkt; kt += kAttnWaves) {
    if (kt + kAttnWaves < nkt) load_tile(kt + kAttnWaves, nxt);  // in flight under this tile's arithmetic
    const int k0 = 32 * kt;
    const float mb = k0 + l32 < N ? p.inf * (cur.mask - 1.f) : ninf;
    const bool has_mb = __builtin_amdgcn_ballot_w64(mb != 0.f) != 0;
    f32x16_t s = zero16(), ss = zero16();
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      u32x4_t kop[3];
      split_step(cur.k, st, kop);
      ss = mfma_32x32x16(kop[2], qop[st][0], ss);
      s = mfma_32x32x16(kop[1], qop[st][0], s);
      ss = mfma_32x32x16(kop[0], qop[st][2], ss);
      s = mfma_32x32x16(kop[0], qop[st][1], s);
      ss = mfma_32x32x16(kop[1], qop[st][1], ss);
      s = mfma_32x32x16(kop[0], qop[st][0], s);
    }
#pragma unroll
    for (int v = 0; v < 16; ++v) s[v] += ss[v];
    if (has_mb) {
      if (lh == 0) mbs[wave][l32] = mb;
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        const float4 u = *reinterpret_cast<const float4*>(&mbs[wave][8 * a + 4 * lh]);
        s[4 * a] += u.x, s[4 * a + 1] += u.y, s[4 * a + 2] += u.z, s[4 * a + 3] += u.w;
      }
      __builtin_amdgcn_wave_barrier();
    }
#pragma unroll
    for (int v = 0; v < 16; ++v) s[v] += cur.pb[v];
    float mx = s[0];
#pragma unroll
    for (int v = 1; v < 16; ++v) mx = fmaxf(mx, s[v]);
    const float m_new = fmaxf(m_run, fmaxf(mx, __shfl_xor(mx, 32, 64)));  // of the logits that are numbers
    const float ref = m_new == ninf ? 0.f : m_new;  // all of the pair bias so far was -inf: its keys weigh 0, not NaN
    const float alpha = exp_neg(m_run - ref);       // 0 on the first tile
    m_run = m_new;
    l_run *= alpha;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      s[v] = exp_neg(s[v] - ref);
      l_run += s[v];
      oacc[v] *= alpha;
      osmall[v] *= alpha;
    }
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      float x[8];
      u32x4_t ph, pm, pl, vop[3];
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = s[8 * st + e];
      split8(x, ph, pm, pl);
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = cur.v[8 * st + e] * vkeep;
      split8(x, vop[0], vop[1], vop[2]);
      osmall = mfma_32x32x16(vop[2], ph, osmall);
      oacc = mfma_32x32x16(vop[1], ph, oacc);
      osmall = mfma_32x32x16(vop[0], pl, osmall);
      oacc = mfma_32x32x16(vop[0], pm, oacc);
      osmall = mfma_32x32x16(vop[1], pm, osmall);
      oacc = mfma_32x32x16(vop[0], ph, oacc);
    }
    cur = nxt;
  }
  // ---- merge the waves: common maximum, rescaled sums and accumulators
  const size_t off = (bN + qrow) * HD + h * D + 4 * lh;
  float4 gate[4];
  if (wave == 0) {  // asked for before the barrier: behind the test for NaN they would be waited for
#pragma unroll
    for (int a = 0; a < 4; ++a) gate[a] = *reinterpret_cast<const float4*>(p.g + off + (8 * a < D ? 8 * a : 0));
  }
  merge[wave][16][lane] = m_run;  // -inf for a wave without tiles
  merge[wave][17][lane] = l_run + __shfl_xor(l_run, 32, 64);
#pragma unroll
  for (int v = 0; v < 16; ++v) merge[wave][v][lane] = oacc[v] + osmall[v];
  __syncthreads();
  if (wave != 0) return;
  float m_tot = merge[0][16][lane];  // -inf only where no key of the query weighs anything (the row is NaN then)
#pragma unroll
  for (int w = 1; w < kAttnWaves; ++w) m_tot = fmaxf(m_tot, merge[w][16][lane]);
  float l_tot = 0.f;
#pragma unroll
  for (int v = 0; v < 16; ++v) oacc[v] = 0.f;
#pragma unroll
  for (int w = 0; w < kAttnWaves; ++w) {
    const float sc = exp_neg(merge[w][16][lane] - m_tot);  // 0 for a wave without tiles
    l_tot += merge[w][17][lane] * sc;
#pragma unroll
    for (int v = 0; v < 16; ++v) oacc[v] += merge[w][v][lane] * sc;
  }
  if (!q_valid) return;
  bool again = l_tot != l_tot;
#pragma unroll
  for (int v = 0; v < 16; ++v) again |= oacc[v] != oacc[v];
  if (again) {  // the query without the matrix instructions: the maximum, then the weighted sum of this lane's channels
    const float* qr = p.q + (bN + qrow) * HD + h * D;
    auto logit = [&](int key) {
      const float* kr = p.k + (bN + key) * HD + h * D;
      float acc = 0.f;
      for (int d = 0; d < D; ++d) acc = fmaf(qr[d], kr[d], acc);
      return acc + p.inf * ((p.mask ? p.mask[bN + key] : 1.f) - 1.f) + pb[key];
    };
    m_tot = ninf, l_tot = 0.f;
#pragma unroll
    for (int v = 0; v < 16; ++v) oacc[v] = 0.f;
    bool lost = false;  // a logit that is NaN, or +inf: so is the whole row
#pragma unroll 1
    for (int key = 0; key < N && !lost; ++key) {
      const float x = logit(key);
      lost = !(x < __builtin_inff());
      m_tot = lost ? x - x : fmaxf(m_tot, x);
    }
#pragma unroll 1
    for (int key = 0; key < (lost ? 1 : N); ++key) {
      const float w = exp_neg(logit(key) - m_tot);
      const float* vr = p.v + (bN + key) * HD + h * D + 4 * lh;
      l_tot += w;
#pragma unroll
      for (int v = 0; v < 16; ++v)
        if (8 * (v >> 2) < D) oacc[v] = fmaf(w, vr[8 * (v >> 2) + (v & 3)], oacc[v]);
    }
  }
  const float inv = 1.0f / l_tot;
#pragma unroll
  for (int a = 0; a < 4; ++a)
    if (8 * a < D) {  // registers 4 a .. + 3 are head channels 8 a + 4 lh .. + 3
      const float4 g = gate[a];
      *reinterpret_cast<float4*>(p.og + off + 8 * a) = make_float4(oacc[4 * a] * inv * g.x, oacc[4 * a + 1] * inv * g.y,
                                                                   oacc[4 * a + 2] * inv * g.z, oacc[4 * a + 3] * inv * g.w);
    }
}

// outputs 4 c4 .. + 3 of row r of a tile of T x T, for the threads that have one
template <int T, int NW>
__device__ __forceinline__ bool tile_products(const float* src, long pos0, long n_rows, int K, const float* W, float* part, int& r, int& c4,
                                              float4& v) {
  if (T == 32) plain_products<NW>(src, pos0, n_rows, K, W, part);
  else plain_products16<NW>(src, pos0, n_rows, K, W, part);
  r = threadIdx.x / (T / 4), c4 = threadIdx.x % (T / 4);
  if (threadIdx.x >= T * T / 4 || pos0 + r >= n_rows) return false;
  v = sum_partials<NW, T == 32 ? kPartLd : kPart16Ld>(part, T == 32 ? kPart : kPart16, r, c4);
  if (__builtin_expect(has_nan(v), 0)) {
    const float4* x = reinterpret_cast<const float4*>(src + (pos0 + r) * K);
    v = plain_dots([&](int k) { return x[k]; }, W + (size_t)4 * c4 * K, K);
  }
  return true;
}

// out = [a +] og Wo^T (plain FMA kernel 41 / 45 / 49 us at 64 / 384 / 768 rows)
template <int T>
constexpr int kOutWaves = T == 32 ? 4 : 8;
template <int T>  // rows and outputs of a tile, 32 or 16
__global__ __launch_bounds__(64 * kOutWaves<T>) void single_out_x3_f32(SingleAttnF32Args p) {
  __shared__ __align__(16) float part[kOutWaves<T> * (T == 32 ? kPart : kPart16)];
  const long rows = (long)p.B * p.N, pos0 = (long)blockIdx.x * T;
  const int HD = p.H * p.D, o0 = T * blockIdx.y;
  int r, c4;
  float4 v;
  if (!tile_products<T, kOutWaves<T>>(p.og, pos0, rows, HD, p.wo + (size_t)o0 * HD, part, r, c4, v)) return;
  const size_t off = (pos0 + r) * p.C + o0 + 4 * c4;
  if (p.add_residual) {
    const float4 x = *reinterpret_cast<const float4*>(p.a + off);
    v.x = x.x + v.x, v.y = x.y + v.y, v.z = x.z + v.z, v.w = x.w + v.w;
  }
  *reinterpret_cast<float4*>(p.out + off) = v;
}

// h = silu(LN(x) Wa^T) * (LN(x) Wb^T), [rows][HID] (the transition in one plain FMA kernel: 320 / 348 / 448 us
// at 64 / 384 / 768 rows)
__global__ __launch_bounds__(64 * kLnWaves) void row_hidden_x3_f32(RowTransitionF32Args p) {
  __shared__ __align__(16) float part[kLnWaves * 2 * kPart];
  __shared__ float red[2 * kLnWaves * 32];
  const long pos0 = (long)blockIdx.x * 32;
  const int o0 = 32 * blockIdx.y;
  const float* const W[2] = {p.wa + (size_t)o0 * p.C, p.wb + (size_t)o0 * p.C};
  ln_products<2>(p.x, pos0, p.rows, p.C, p.ln_w, p.ln_b, W, part, red);
  const int r = threadIdx.x >> 3, c4 = threadIdx.x & 7;
  if (pos0 + r >= p.rows) return;
  float4 a = sum_partials<kLnWaves>(part, 2 * kPart, r, c4), b = sum_partials<kLnWaves>(part + kPart, 2 * kPart, r, c4);
  if (__builtin_expect(has_nan(a), 0)) a = ln_plain_dots(p.x, pos0, r, p.C, p.ln_w, p.ln_b, W[0] + (size_t)4 * c4 * p.C, red);
  if (__builtin_expect(has_nan(b), 0)) b = ln_plain_dots(p.x, pos0, r, p.C, p.ln_w, p.ln_b, W[1] + (size_t)4 * c4 * p.C, red);
  float4 v;
  v.x = a.x * sigmoid_f32(a.x) * b.x;
  v.y = a.y * sigmoid_f32(a.y) * b.y;
  v.z = a.z * sigmoid_f32(a.z) * b.z;
  v.w = a.w * sigmoid_f32(a.w) * b.w;
  *reinterpret_cast<float4*>(p.hidden + (pos0 + r) * p.HID + o0 + 4 * c4) = v;
}

// out = [x +] (h Wout^T) * mask; the sum over up to 2048 hidden channels is dealt to 16 waves
constexpr int kRowOutWaves = 16;
template <int T>  // rows and outputs of a tile, 32 or 16
__global__ __launch_bounds__(64 * kRowOutWaves) void row_out_x3_f32(RowTransitionF32Args p) {
  extern __shared__ __align__(16) float part[];  // [kRowOutWaves][kPart or kPart16]
  const long pos0 = (long)blockIdx.x * T;
  const int o0 = T * blockIdx.y;
  int r, c4;
  float4 v;
  if (!tile_products<T, kRowOutWaves>(p.hidden, pos0, p.rows, p.HID, p.wout + (size_t)o0 * p.HID, part, r, c4, v)) return;
  if (p.mask) {
    const float m = p.mask[pos0 + r];
    v.x *= m, v.y *= m, v.z *= m, v.w *= m;
  }
  const size_t off = (pos0 + r) * p.C + o0 + 4 * c4;
  if (p.add_residual) {
    const float4 x = *reinterpret_cast<const float4*>(p.x + off);
    v.x = x.x + v.x, v.y = x.y + v.y, v.z = x.z + v.z, v.w = x.w + v.w;
  }
  *reinterpret_cast<float4*>(p.out + off) = v;
}

// The output products in tiles of 16 x 16 where all of these run at once, two to a CU: a tile of 32 x 32 splits and multiplies for twice as
// long and reads twice as much through its CU's L1, on a quarter of the CUs.  Tiles of 32 / 16, us, at 24 / 64 / 150 / 256 / 300 | 384 / 640
// rows: the transition's two kernels 24.6 / 26.2 / 28.5 / 33.3 / 33.0 | 39.6 / 46.4, 17.4 / 17.7 / 20.5 / 30.0 / 30.1 | 41.6 / 53.8; the attention's
// three, 22.7 / 24.2 / 31.3 / 41.6 / 46.1 | 59.2 and 19.6 / 20.8 / 28.2 / 39.8 / 44.3 | 58.3 (512 rows 74.5, 75.7).
hipError_t small_tiles(long rows, int C, bool* small) {
  static int cache[kMaxDevices];
  int cus = 0;
  const hipError_t e = per_device(cache, [](int dev, int* v) { return cu_count(dev, v); }, &cus);
  *small = (rows + 15) / 16 * (C / 16) <= 2l * cus;
  return e;
}

bool aligned16(std::initializer_list<const void*> ptrs) {
  for (const void* q : ptrs)
    if (reinterpret_cast<uintptr_t>(q) % 16 != 0) return false;
  return true;
}

}  // namespace

bool single_attn_x3_serves(const SingleAttnF32Args& a) {
  const int HD = a.H * a.D;
  return a.C % 32 == 0 && a.C <= 32 * kLnWaves * kLnBlocks && HD % 32 == 0 && a.D % 8 == 0 && a.D <= 32 &&
         4 * HD / 32 <= 65535 &&
         aligned16({a.a, a.ln_w, a.ln_b, a.wq, a.wk, a.wv, a.wg, a.wo, a.q, a.k, a.v, a.g, a.og, a.out});
}

hipError_t single_attn_x3_fwd_f32(const SingleAttnF32Args& a, hipStream_t stream) {
  const long rows = (long)a.B * a.N;
  const long row_tiles = (rows + 31) / 32;
  if (row_tiles > 0x7fffffffl) return hipErrorInvalidValue;
  const int HD = a.H * a.D;
  if (a.phases & kSingleProject) {
    hipLaunchKernelGGL(single_proj_x3_f32, dim3((unsigned)row_tiles, 4 * HD / 32), dim3(64 * kLnWaves), 0, stream, a);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  if (!(a.phases & kSingleAttend)) return hipSuccess;
  const int pb_vec = a.N % 4 == 0 && aligned16({a.pair_bias}) ? 1 : 0;
  hipLaunchKernelGGL(single_attn_x3_f32, dim3((a.N + 31) / 32, a.H, a.B), dim3(64 * kAttnWaves), 0, stream, a, pb_vec);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  bool small = false;
  e = small_tiles(rows, a.C, &small);
  if (e != hipSuccess) return e;
  if (small)
    hipLaunchKernelGGL(single_out_x3_f32<16>, dim3((unsigned)((rows + 15) / 16), a.C / 16), dim3(64 * kOutWaves<16>), 0, stream, a);
  else
    hipLaunchKernelGGL(single_out_x3_f32<32>, dim3((unsigned)row_tiles, a.C / 32), dim3(64 * kOutWaves<32>), 0, stream, a);
  return hipGetLastError();
}

bool row_transition_x3_serves(const RowTransitionF32Args& a) {
  return a.hidden && a.C % 32 == 0 && a.C <= 32 * kLnWaves * kLnBlocks && a.HID % 32 == 0 &&
         aligned16({a.x, a.ln_w, a.ln_b, a.wa, a.wb, a.wout, a.hidden, a.out});
}

hipError_t row_transition_x3_fwd_f32(const RowTransitionF32Args& a, hipStream_t stream) {
  const long row_tiles = (a.rows + 31) / 32;
  if (row_tiles > 0x7fffffffl) return hipErrorInvalidValue;
  constexpr size_t lds = (size_t)kRowOutWaves * kPart * sizeof(float);
  hipError_t e = allow_dynamic_lds<row_out_x3_f32<32>>(lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(row_hidden_x3_f32, dim3((unsigned)row_tiles, a.HID / 32), dim3(64 * kLnWaves), 0, stream, a);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  bool small = false;
  e = small_tiles(a.rows, a.C, &small);
  if (e != hipSuccess) return e;
  if (small)
    hipLaunchKernelGGL(row_out_x3_f32<16>, dim3((unsigned)((a.rows + 15) / 16), a.C / 16), dim3(64 * kRowOutWaves),
                       kRowOutWaves * kPart16 * sizeof(float), stream, a);
  else
    hipLaunchKernelGGL(row_out_x3_f32<32>, dim3((unsigned)row_tiles, a.C / 32), dim3(64 * kRowOutWaves), lds, stream, a);
  return hipGetLastError();
}

}  // namespace of3
