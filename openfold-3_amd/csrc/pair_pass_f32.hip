// Position-wise passes of the two fp32 triangle modules at 64 and 128 channels (c_z = c_hidden = heads x width:
// the template stack's and the trunk's), products on the fp16 matrix instructions with operands split into two
// fp16 terms (of3_split.h).  pair_f32.hip has the passes for every other shape.
//
// What bounded the passes of pair_f32.hip at these widths: every group of 32 positions read all split weights
// again from L2 (6 KB per k-step of a wave against 12 MFMAs, 64 bytes per clock and compute unit: the rate of the
// L1), and LayerNorm, products and epilogue ran one after the other.  Here the weights stay on the chip:
// persistent work-groups whose waves each own one 32-output tile of one or two matrices and keep its split
// operands in registers (64 registers per matrix at 128 channels, 32 at 64) for all the tiles they process; a tile
// of 32 positions goes through LDS once (two fp16 planes, 16-byte chunks XOR-swizzled by the position), read by
// all waves.  The next tile's rows are in flight meanwhile, in registers.  At small N the weights are a
// one-time 3 us instead of a latency in every k-step.
#include <type_traits>

#include "of3_device.h"
#include "of3_kernels.h"
#include "of3_launch.h"
#include "of3_pair_f32.h"
#include "of3_pass_f32.h"
#include "of3_split.h"
#include "of3_weight_split.h"

namespace of3 {

namespace {

using namespace pass_f32;

// the odd rows of 16 lanes of `even` change places with the even rows of `odd`
__device__ __forceinline__ void swap_rows(uint32_t& even, uint32_t& odd) {
  const u32x2_t r = __builtin_amdgcn_permlane16_swap(even, odd, false, false);
  even = r[0], odd = r[1];
}

// ---- triangle multiplication, input pass: a, b = mask * sigmoid(LN(z) Wg^T) * (LN(z) Wp^T) ------------------
// Wave = gate and projection of one 32-channel tile of a or b: two matrices, 128 registers of split operands at 128
// channels.  At 64 channels a work-group of four waves has a and b.  At 128 it has a and b in eight waves, so that a tile is read
// and normalised once, as long as there is more than a tile per CU; below that four waves of one of the two, which
// spread over all CUs (us, four / eight waves: pair stack N = 80 116.8 / 117.9, 200 310.0 / 309.3, 768 4590 / 4465, trunk 384 1260 / 1204).
// Bytes per tile: 16 KB read, 32 KB written; N = 768 359 us with two barriers per tile and every tile read by two work-groups,
// 324 now (212 without the products, 267 without the stores: matrix and vector time and the transfers still add up, at the clock
// that they allow together).
// Tile = 32 columns k of one row; four
// consecutive rows of a panel are consecutive tiles of one XCD, so that the 64-byte pieces a tile writes per channel
// and term meet in L2 as whole lines.
template <int C>
struct ProjLds {
  static constexpr size_t kBytes = (size_t)2 * HalfTile<C>::SLOTS * 16 + (2 * C + 128) * sizeof(float);
};

template <int C, int NW>
__global__ __launch_bounds__(64 * NW, 2) void trimul_proj_pass(TrimulF32 p, int panels, int row_groups, int total) {
  typedef HalfTile<C> Tile;
  constexpr int KS = C / 16, OT = C / 32, TASKS = 8 / NW;
  constexpr bool kOneSide = OT == NW;  // a and b in work-groups of their own
  constexpr bool kStagger = NW == 8;
  extern __shared__ u32x4_t lds[];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  float* ln = reinterpret_cast<float*>(lds + 2 * Tile::SLOTS);  // [2][C], times the scale of the activations
  float* msk = ln + 2 * C;                                 // [4][32]
  const int slot = grid_slot(), N = p.N, pair = kOneSide ? slot & 1 : wave / OT, ot = wave % OT;
  const WeightX3 Wg = pair ? p.s_bg : p.s_ag, Wp = pair ? p.s_bp : p.s_ap;
  const WeightScales &sg = Wg.scales()[ot], &sp = Wp.scales()[ot];
  const float in_scale = sg.input, g_unscale = sg.unscale, out_scale = sp.store;
  MaskExponent mask_top;
  u32x4_t wg[KS][2], wp[KS][2];
  load_unit<C, 2>(Wg, ot, lane, wg);
  load_unit<C, 2>(Wp, ot, lane, wp);
  mask_top.load(p);
  for (int c = tid; c < C; c += 64 * NW) ln[c] = p.ln_in_w[c] * in_scale, ln[C + c] = p.ln_in_b[c] * in_scale;
  wait_vmcnt<0>();  // the weights have landed: no wait for them, and with it for the rows in flight, inside the loop
  const int mask_e = mask_top.of_wave();
  __syncthreads();

  struct Place {
    int b, r, k0;
  };
  auto place = [&](int id) {
    Place t;
    const int q = id & 3, rest = id >> 2, per_b = row_groups * panels;
    t.b = rest / per_b;
    const int rem = rest - t.b * per_b, rg = rem / panels;
    t.r = 4 * rg + q;
    t.k0 = 32 * (rem - rg * panels);
    return t;
  };
  RowRegs<C> raw[TASKS];
  float mraw = 1.f;
  auto load_tile = [&](int id) {  // addresses clamped to real positions: no load is under a condition
    const Lane here = lane_here();
    const int li = here.li, lg = here.lg, l32 = here.l32;
    const Place t = place(id);
    const int r = t.r < N ? t.r : N - 1;
    const float* base = p.z + t.b * p.zv.stride_b + r * p.zv.stride_r;
#pragma unroll
    for (int u = 0; u < TASKS; ++u) {
      int k = t.k0 + 4 * (wave + NW * u) + lg;
      k = k < N ? k : N - 1;
      load_row<C>(base + k * p.zv.stride_k, li, raw[u]);
    }
    int k = t.k0 + l32;
    k = k < N ? k : N - 1;
    if (p.mask) mraw = p.mask[t.b * p.mv.stride_b + r * p.mv.stride_r + k * p.mv.stride_k];
  };

  const int step = kOneSide ? gridDim.x / 2 : gridDim.x, first_id = kOneSide ? slot >> 1 : slot;
  // rows of the n-th tile of this work-group, in registers, to its LDS tile; requests those of the next one
  auto normalise = [&](int n) {
    const int id = first_id + n * step;
    const Tile xn = {lds + (n & 1) * Tile::SLOTS};
    const Place t = place(id);
    const Lane here = lane_here();
#pragma unroll
    for (int u = 0; u < TASKS; ++u) {
      const int li = here.li, pos = 4 * (wave + NW * u) + here.lg;
      float4 y[C / 64];
      norm_row<C>(raw[u], ln, li, y);
#pragma unroll
      for (int e = 0; e < C / 64; ++e) xn.store4(pos, li + 16 * e, y[e]);
    }
    // the panel's padding holds zeros
    if (tid < 32) msk[32 * (n & 3) + tid] = t.k0 + tid < N ? __builtin_ldexpf(mraw, -mask_e) : 0.f;
    load_tile(id + step < total ? id + step : id);
  };
  if (first_id >= total) return;  // the whole work-group
  const int count = (total - first_id + step - 1) / step;
  // Interval n lies between the barrier that completes tile n and the next one.  In it the early half of a work-group of eight waves
  // finishes tile n - 1, normalises tile n + 1 and takes the products of tile n, the late half takes the products first, so that
  // of the two waves of a SIMD (w and w + 4) one has vector work while the other has matrix work: 4500 -> 4470 us per pair stack N = 768.
  const bool early = kStagger && wave < NW / 2;
  load_tile(first_id);
  normalise(0);
  __syncthreads();
  if (early && count > 1) normalise(1);
  for (int n = 0; n < count; ++n) {
    const Tile xn = {lds + (n & 1) * Tile::SLOTS};
    const Place t = place(first_id + n * step);
    HalfSum<C, false> sum_g, sum_p;
    const Lane at = lane_here();
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const u32x4_t* x = xn.s + Tile::slot(at.l32, 2 * s + at.lh);
      const u32x4_t op[2] = {x[0], x[Tile::PLANE]};
      sum_g.step(wg[s], op);
      sum_p.step(wp[s], op);
    }
    const f32x16_t ag = sum_g.total(), ap = sum_p.total();
    if (early && n + 1 < count) __syncthreads();
    wait_vmcnt<0>();  // the rows in flight since a product ago, ahead of the stores, so that nobody waits for these
    // channels in the lanes, positions in the registers: registers 8 st .. + 7 are the k-values 16 st + 8 (e >> 2)
    // + 4 lh + (e & 3), stored as the 8 consecutive columns 16 st + 8 lh .. of the panel row (a and b in the same
    // order, which is all a sum over k needs); positions past N are copies of a real row, and the zeros of msk make the
    // panel's padding of them
    if (t.r < N) {
      const Lane out = lane_here();
      const int l32 = out.l32, lh = out.lh;
      const int l16 = l32 & 15;
      const int rot0 = panel_rotation(32 * ot + l16, p.Np), rot1 = panel_rotation(32 * ot + 16 + l16, p.Np);
      u32x4_t op[2][2];
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        float x[8];
#pragma unroll
        for (int a = 0; a < 2; ++a) {
          const float4 m4 = *reinterpret_cast<const float4*>(msk + 32 * (n & 3) + 16 * st + 8 * a + 4 * lh);
          const float m[4] = {m4.x, m4.y, m4.z, m4.w};
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int v = 8 * st + 4 * a + e;
            x[4 * a + e] = m[e] * sigmoid_hw_f32(ag[v], g_unscale) * (ap[v] * out_scale);
          }
        }
        split8h(x, op[st][0], op[st][1]);
      }
      // Lane l32, half lh has the chunks lh and 2 + lh of channel l32.  Rows of 16 lanes exchange one, so that one store writes the 64 bytes of
      // channels 0..15 and the next those of 16..31 (32-byte pieces of every channel otherwise: twice the requests).  Eight instructions in the place
      // of the 32 of an exchange between neighbouring lanes, which selected by lane before and after.
#pragma unroll
      for (int pl = 0; pl < 2; ++pl)
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          uint32_t a = op[0][pl][w], b = op[1][pl][w];
          swap_rows(a, b);
          op[0][pl][w] = a, op[1][pl][w] = b;
        }
      const size_t chan = (size_t)p.Np * p.Np, pn = (size_t)(t.k0 >> 5) * p.Np;
      bf16_t* lp = (pair ? p.bs : p.as) + ((size_t)t.b * C + 32 * ot + l16) * chan + 8 * lh + (l32 & 16);
      bf16_t* lp0 = lp + (pn + panel_row(t.r, rot0, p.Np)) * 32;
      bf16_t* lp1 = lp + 16 * chan + (pn + panel_row(t.r, rot1, p.Np)) * 32;
#pragma unroll
      for (int pl = 0; pl < 2; ++pl) {
        *reinterpret_cast<u32x4_t*>(lp0 + pl * p.ab_plane) = op[0][pl];
        *reinterpret_cast<u32x4_t*>(lp1 + pl * p.ab_plane) = op[1][pl];
      }
    }
    if (n + (early ? 2 : 1) < count) normalise(n + (early ? 2 : 1));
    if (!early && n + 1 < count) __syncthreads();
  }
  // block 0 has a tile.  Not ahead of the rows, whose wait would be for this store too (0.5 us of 8 at one tile per work-group)
  if (blockIdx.x == 0 && tid == 0) MaskTop::of(p.s_ap)->exponent = mask_e;
}

// ---- output passes ------------------------------------------------------------------------------------------
// Wave = one 32-channel tile of the gate and the same tile of the output projection, weights in registers as in the input
// passes.  One LDS tile holds LayerNorm(z) for the gates, another LayerNorm(x) or the gated attention output: two barriers per tile.
// Every load of a tile is requested before the product ahead of its use and nothing waits for a store (N = 768, 268 -> 251 and
// 256 -> 239 us); the rows leave whole, by way of the residual's place in LDS, after the next tile's first barrier (RowTile: -> 235 and 221; lanes
// that load and store 64 bytes of their own row each kept the address unit busy for 54 and 64 % of the time).
// Four waves per work-group at 128 channels, two
// work-groups per CU; two waves at 64.
template <int C>
struct OutLds {
  static constexpr int NW = C / 32;
  static constexpr size_t kTrimul = (size_t)(2 * HalfTile<C>::SLOTS + RowTile<C>::SLOTS) * 16 + (2 * 32 * 2 * NW + 4 * C) * sizeof(float);
  static constexpr size_t kTriattn = (size_t)(2 * HalfTile<C>::SLOTS + RowTile<C>::SLOTS) * 16 + 2 * C * sizeof(float);
};
// the two matrices of an output wave, outputs dealt by rowperm16: lane (position l32, half lh) ends with the outputs
// 32 ot + 16 lh + v
template <int C>
struct OutWeights {
  static constexpr int KS = C / 16;
  u32x4_t g[KS][2], o[KS][2];
  __device__ __forceinline__ void load(const WeightX3& Wg, const WeightX3& Wo, int ot, int l32, int lh) {
    const int src = rowperm16(l32) + 32 * lh;
    load_unit<C, 2>(Wg, ot, src, g);
    load_unit<C, 2>(Wo, ot, src, o);
  }
};
// ---- triangle multiplication, output pass: out = [z +] (LN(x) Wz^T) * sigmoid(LN(z) Wg^T)
// x is channel-major: thread (position tid % 32, group tid / 32) holds 16 channels of a position; the statistics are
// combined from the groups' means and squared deviations (one exchange).
template <int C>
__global__ __launch_bounds__(2 * C, 2) void trimul_out_pass(TrimulF32 p, int panels, int total) {
  typedef HalfTile<C> Tile;
  constexpr int NW = C / 32, TASKS = 8 / NW, NG = 2 * NW;
  extern __shared__ u32x4_t lds[];
  const Tile tile = {lds}, second = {lds + Tile::SLOTS};
  const RowTile<C> rows = {reinterpret_cast<float4*>(lds + 2 * Tile::SLOTS)};
  float* red = reinterpret_cast<float*>(lds + 2 * Tile::SLOTS + RowTile<C>::SLOTS);  // [NG][32] means, [NG][32] squared deviations
  float* ln = red + 2 * 32 * NG;                             // LayerNorm of z [2][C], of x [2][C], times the activations' scales
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, l32 = lane & 31, lh = lane >> 5;
  const int N = p.N;
  const WeightScales &sg = p.s_g.scales()[wave], &sz = p.s_z.scales()[wave];
  const float g_in = sg.input, g_unscale = sg.unscale, z_in = sz.input, z_unscale = sz.unscale;
  OutWeights<C> w;
  w.load(p.s_g, p.s_z, wave, l32, lh);
  for (int c = tid; c < C; c += 64 * NW) {
    ln[c] = p.ln_in_w[c] * g_in, ln[C + c] = p.ln_in_b[c] * g_in;
    ln[2 * C + c] = p.ln_out_w[c] * z_in, ln[3 * C + c] = p.ln_out_b[c] * z_in;
  }
  wait_vmcnt<0>();  // the weights
  __syncthreads();

  struct Place {
    int b, i, j0;
  };
  auto place = [&](int id) {
    Place t;
    const int bi = id / panels;
    t.j0 = 32 * (id - bi * panels);
    t.b = bi / N;
    t.i = bi - t.b * N;
    return t;
  };
  const int xpos = tid & 31, xg = tid >> 5;
  RowRegs<C> zraw[TASKS];
  float xraw[16];  // channels 8 xg .. + 7 and C / 2 + 8 xg .. + 7
  const size_t NN = (size_t)N * N;
  auto load_z = [&](int id) {
    const Lane here = lane_here();
    const int li = here.li, lg = here.lg;
    const Place t = place(id);
    const float* base = p.z + t.b * p.zc.stride_b + t.i * p.zc.stride_r;
#pragma unroll
    for (int u = 0; u < TASKS; ++u) {
      int j = t.j0 + 4 * (wave + NW * u) + lg;
      j = j < N ? j : N - 1;
      load_row<C>(base + j * p.zc.stride_k, li, zraw[u]);
    }
  };
  auto load_x = [&](int id) {
    const Place t = place(id);
    int j = t.j0 + xpos;
    j = j < N ? j : N - 1;
    const float* xp = p.x + (((size_t)t.b * C + 8 * xg) * N + t.i) * N + j;
#pragma unroll
    for (int e = 0; e < 8; ++e) xraw[e] = xp[e * NN], xraw[8 + e] = xp[(C / 2 + e) * NN];
  };

  // result rows of a tile, as the threads have normalised them
  auto store_rows = [&](const Place& t) {
    const Lane here = lane_here();
    float* base = p.out + t.b * p.zc.stride_b + t.i * p.zc.stride_r;
#pragma unroll
    for (int u = 0; u < TASKS; ++u) {
      const int pos = 4 * (wave + NW * u) + here.lg;
      if (t.j0 + pos < N) rows.store(base + (t.j0 + pos) * p.zc.stride_k, pos, here.li);
    }
  };
  int id = grid_slot();
  bool first = true;
  Place before = {};
  if (id < total) load_z(id), load_x(id);
  for (; id < total; id += gridDim.x) {
    const Place t = place(id);
    const int next = id + (int)gridDim.x < total ? id + (int)gridDim.x : id;
    const Lane here = lane_here();
#pragma unroll
    for (int u = 0; u < TASKS; ++u) {
      const int li = here.li, pos = 4 * (wave + NW * u) + here.lg;
      float4 y[C / 64];
      norm_row<C>(zraw[u], ln, li, y);
#pragma unroll
      for (int e = 0; e < C / 64; ++e) tile.store4(pos, li + 16 * e, y[e]);
    }
    {
      float s = 0.f, q = 0.f;
#pragma unroll
      for (int e = 0; e < 16; ++e) s += xraw[e];
      s *= 0.0625f;
#pragma unroll
      for (int e = 0; e < 16; ++e) q += (xraw[e] - s) * (xraw[e] - s);
      red[xg * 32 + xpos] = s;
      red[(NG + xg) * 32 + xpos] = q;
    }
    __syncthreads();  // LayerNorm(z) and the rows of the tile before are complete, and everybody has finished with the second tile
    if (!first) store_rows(before);
    if (p.add_residual) {
      const Lane at = lane_here();
#pragma unroll
      for (int u = 0; u < TASKS; ++u) rows.put(4 * (wave + NW * u) + at.lg, at.li, zraw[u]);
    }
    load_z(next);
    const f32x16_t gate = unit_product<C, true>(tile, w.g);
    {
      // mean of the groups' means; squared deviations = within the groups + 16 x those of the groups' means
      float mg[NG], mean = 0.f, q = 0.f;
#pragma unroll
      for (int g = 0; g < NG; ++g) mean += mg[g] = red[g * 32 + xpos];
      mean *= 1.f / NG;
#pragma unroll
      for (int g = 0; g < NG; ++g) q += red[(NG + g) * 32 + xpos] + 16.f * ((mg[g] - mean) * (mg[g] - mean));
      const float rstd = rsqrt_f32(q * (1.f / C) + kEps);
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) {
        const float* wv = ln + 2 * C + hf * (C / 2) + 8 * xg;
        float y[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) y[e] = (xraw[8 * hf + e] - mean) * rstd * wv[e] + wv[C + e];
        second.store8(xpos, hf * (C / 16) + xg, y);
      }
    }
    load_x(next);
    __syncthreads();  // LayerNorm(x) is complete, and everybody has finished with the first tile
    f32x16_t acc = unit_product<C, true>(second, w.o);
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] = acc[v] * z_unscale * sigmoid_hw_f32(gate[v], g_unscale);
    rows.add(wave, acc, p.add_residual);
    before = t;
    first = false;
  }
  if (first) return;  // the whole work-group
  __syncthreads();
  store_rows(before);
}

// ---- triangle attention, input pass: q / sqrt(D), k, v^T as split operands of the core, triangle bias --------
// Wave = one 32-channel tile of q, k or v (12 waves at 128 channels, three per SIMD).  Tile = one 32-position panel;
// double buffered, one barrier per tile (three panels per barrier: 417 against 385 us at N = 768).  The H rows of the
// triangle bias are dot products taken on the normalised rows while they are in registers.
// PARTS work-groups share a tile, each with every output tile's PARTS-th and as many of the bias rows, where there are CUs left:
// what bounds a launch of one tile per CU is the 192 KB of weights through the CU's L1 (3 us) and the products of three waves
// per SIMD.
template <int C>
struct AttProjLds {
  static constexpr size_t kBytes = (size_t)2 * HalfTile<C>::SLOTS * 16 + (2 * C + 8 * C) * sizeof(float);
};

template <int C, int PARTS>
__global__ __launch_bounds__(6 * C / PARTS) void triattn_proj_pass(TriattnF32 p, int panels, int total) {
  typedef HalfTile<C> Tile;
  constexpr int OT = C / 32 / PARTS, NW = 3 * OT, KS = C / 16, TASKS = (8 + NW - 1) / NW;
  extern __shared__ u32x4_t lds[];
  float* ln = reinterpret_cast<float*>(lds + 2 * Tile::SLOTS);  // [2][C], times the scale of the activations
  float* wb = ln + 2 * C;                                       // [H][C], H <= 8, times the scale of the logits over that of the activations
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int slot = grid_slot(), part = slot % PARTS;
  const int N = p.N, H = p.H, kind = wave / OT, ot = part * OT + wave % OT;
  const int h0 = H * part / PARTS, h1 = H * (part + 1) / PARTS;  // this work-group's heads of the bias
  const bool narrow = p.D == 16;
  const WeightX3 W = kind == 0 ? p.s_q : kind == 1 ? p.s_k : p.s_v;
  const WeightScales& sc = W.scales()[ot];
  const float in_scale = sc.input;
  // q / sqrt(c) after the projection (attention.py:283-284)
  const float out_scale = sc.store * (kind == 0 ? 1.0f / sqrtf((float)p.D) : 1.f);
  u32x4_t w[KS][2];
  load_unit<C, 2>(W, ot, tid & 63, w);
  for (int c = tid; c < C; c += 64 * NW) ln[c] = p.ln_w[c] * in_scale, ln[C + c] = p.ln_b[c] * in_scale;
  for (int c = tid; c < H * C; c += 64 * NW) {
    const int t = c / C * p.D / 32;  // the head's tile of q and k
    wb[c] = p.w_b[c] * (p.s_q.scales()[t].output * p.s_k.scales()[t].output / in_scale);
  }
  wait_vmcnt<0>();  // the weights
  __syncthreads();

  // panel -> its row (b N + i) and first position
  auto row_of = [&](int pn, int& j0) {
    const int bi = pn / panels;
    j0 = 32 * (pn - bi * panels);
    return bi;
  };
  RowRegs<C> raw[TASKS];  // task u of this wave: rows 4 (wave + NW u) .. + 3, where these are below 32
  auto load_tile = [&](int pn) {
    const Lane here = lane_here();
    int j0;
    const int bi = row_of(pn, j0), b = bi / N, i = bi - b * N;
#pragma unroll
    for (int u = 0; u < TASKS; ++u)
      if (wave + NW * u < 8) {
        int j = j0 + 4 * (wave + NW * u) + here.lg;
        j = j < N ? j : N - 1;
        load_row<C>(p.x + b * p.xv.stride_b + i * p.xv.stride_r + j * p.xv.stride_k, here.li, raw[u]);
      }
  };
  // the operands of a step are read one step ahead, no further: read as early as the compiler would have it, they do
  // not fit the registers of three waves per SIMD
  auto product = [&](auto w_rows, const Tile& t) {
    HalfSum<C, decltype(w_rows)::value> sum;
    u32x4_t nxt[2];
    const Lane at = lane_here();
    auto read = [&](int s) {
      const u32x4_t* x = t.s + Tile::slot(at.l32, 2 * s + at.lh);
      nxt[0] = x[0], nxt[1] = x[Tile::PLANE];
    };
    read(0);
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const u32x4_t op[2] = {nxt[0], nxt[1]};
      if (s + 1 < KS) read(s + 1);
      __builtin_amdgcn_sched_barrier(0);
      sum.step(w[s], op);
      __builtin_amdgcn_sched_barrier(0);
    }
    return sum.total();
  };
  auto split_store = [&](bf16_t* dst, long second, size_t slot, const f32x16_t& acc, int st) {
    float x[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = acc[8 * st + e] * out_scale;
    u32x4_t h, lo;
    split8h(x, h, lo);
    u32x4_t* d4 = reinterpret_cast<u32x4_t*>(dst) + slot;
    d4[0] = h;
    d4[second] = lo;
  };

  const int step = (int)gridDim.x / PARTS;
  int pn = slot / PARTS, buf = 0;
  if (pn < total) load_tile(pn);
  wait_vmcnt<0>();
  for (; pn < total; pn += step, buf ^= 1) {
    const Tile xn = {lds + buf * Tile::SLOTS};
    const Lane here = lane_here();
    int j0;
    const int bi = row_of(pn, j0);
#pragma unroll
    for (int u = 0; u < TASKS; ++u) {
      if (wave + NW * u >= 8) continue;
      const int li = here.li, pos = 4 * (wave + NW * u) + here.lg;
      float4 y[C / 64];
      norm_row<C>(raw[u], ln, li, y);
#pragma unroll
      for (int e = 0; e < C / 64; ++e) xn.store4(pos, li + 16 * e, y[e]);
      float bias = 0.f;  // of head li
      for (int h = h0; h < h1; ++h) {
        float d = 0.f;
#pragma unroll
        for (int e = 0; e < C / 64; ++e) {
          const float4 v = *reinterpret_cast<const float4*>(wb + h * C + 64 * e + 4 * li);
          d += y[e].x * v.x, d += y[e].y * v.y, d += y[e].z * v.z, d += y[e].w * v.w;
        }
        d = group_sum<16>(d);
        bias = li == h ? d : bias;
      }
      if (li >= h0 && li < h1) {  // rows padded to whole panels with zeros
        const int b = bi / N, i = bi - b * N;
        p.tb[(((size_t)b * H + li) * N + i) * p.Jp + j0 + pos] = j0 + pos < N ? bias : 0.f;
      }
    }
    load_tile(pn + step < total ? pn + step : pn);
    __syncthreads();  // this tile is complete, and everybody has finished with the other buffer
    const Lane out = lane_here();
    const int l32 = out.l32, lh = out.lh, lane = l32 + 32 * lh, nt = p.Jp / 32, jt = j0 / 32;
    const size_t row = bi;
    // A 32-column tile of the projections is one head, or two of width 16.  q and k: head channels in the
    // registers, positions in the lanes; v the other way round.  Registers 8 st .. + 7 of a lane are its operand
    // for step st (narrow heads: q, k have one step, that of head 2 ot + st; lane l32 of the v tile is row
    // l32 % 16 of head 2 ot + l32 / 16, its second term row 16 + l32 % 16).
    // Positions past N store copies of the last real one: their keys and values are the reader's to leave out (a bias of -infinity there in the
    // core, which gives them no weight; a value that is not a number makes its real copy's result one as well), their queries' results nobody stores.
    f32x16_t acc;
    bf16_t* dst;
    long second;
    size_t first, next;  // slots of steps 0 and 1
    if (kind < 2) {
      acc = product(std::true_type{}, xn);
      dst = kind == 0 ? p.qs : p.ks;
      second = p.qk_plane / 8;
      first = (row * H + (narrow ? 2 * ot : ot)) * nt + jt;
      first = (narrow ? first : 2 * first) * 64 + lane;
      next = first + (narrow ? (size_t)nt * 64 : 64);
    } else {
      acc = product(std::false_type{}, xn);
      const int head = narrow ? 2 * ot + (l32 >> 4) : ot, vrow = narrow ? (l32 & 15) : l32;
      dst = p.vs;
      second = narrow ? 16 : p.v_plane / 8;
      first = ((row * H + head) * nt + jt) * 2 * 64 + vrow + 32 * lh;
      next = first + 64;
    }
    // The rows in flight, ahead of the stores, and on the way of every wave: with a wait in each branch the compiler saw a way round both and waited at the
    // top of the loop, for the stores as well.  us a launch, before / now: N = 384 78.4 / 76.3, 512 128.7 / 124.6, 768 267 / 261; templates 3 x 200
    // 37.0 / 35.4, 4 x 384 177 / 140.
    wait_vmcnt<0>();
    split_store(dst, second, first, acc, 0);
    split_store(dst, second, next, acc, 1);
  }
}

// ---- triangle attention, output pass: out = [x +] (o * sigmoid(LN(x) Wg^T)) Wo^T
// A wave's 16 channels of a position are consecutive: 64 bytes of o, and two chunks of the second product's operand.
template <int C>
__global__ __launch_bounds__(2 * C, 2) void triattn_out_pass(TriattnF32 p, int panels, int total) {
  typedef HalfTile<C> Tile;
  constexpr int NW = C / 32, TASKS = 8 / NW;
  extern __shared__ u32x4_t lds[];
  const Tile tile = {lds}, second = {lds + Tile::SLOTS};
  const RowTile<C> rows = {reinterpret_cast<float4*>(lds + 2 * Tile::SLOTS)};
  float* ln = reinterpret_cast<float*>(lds + 2 * Tile::SLOTS + RowTile<C>::SLOTS);  // [2][C], times the scale of the activations
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, l32 = lane & 31, lh = lane >> 5;
  const int N = p.N;
  const WeightScales& sg = p.s_g.scales()[wave];
  const float g_in = sg.input, g_unscale = sg.unscale, tile_unscale = p.s_o.scales()[wave].unscale;
  OutWeights<C> w;
  w.load(p.s_g, p.s_o, wave, l32, lh);
  ColumnScales so(p.s_o, NW);
  for (int c = tid; c < C; c += 64 * NW) ln[c] = p.ln_w[c] * g_in, ln[C + c] = p.ln_b[c] * g_in;
  wait_vmcnt<0>();  // the weights
  __syncthreads();

  auto place = [&](int id, int& b, int& i) {  // returns the first position
    const int bi = id / panels;
    b = bi / N;
    i = bi - b * N;
    return 32 * (id - bi * panels);
  };
  RowRegs<C> raw[TASKS];
  float4 oraw[4];
  auto load_rows = [&](int id) {
    const Lane here = lane_here();
    const int li = here.li, lg = here.lg;
    int b, i;
    const int j0 = place(id, b, i);
#pragma unroll
    for (int u = 0; u < TASKS; ++u) {
      int j = j0 + 4 * (wave + NW * u) + lg;
      j = j < N ? j : N - 1;
      load_row<C>(p.x + b * p.xv.stride_b + i * p.xv.stride_r + j * p.xv.stride_k, li, raw[u]);
    }
  };
  auto load_o = [&](int id) {
    const Lane here = lane_here();
    int b, i;
    const int j0 = place(id, b, i);
    const int j = j0 + here.l32 < N ? j0 + here.l32 : N - 1;
    const float* op = p.o + (((size_t)b * N + i) * N + j) * C + 32 * wave + 16 * here.lh;
#pragma unroll
    for (int a = 0; a < 4; ++a) oraw[a] = *reinterpret_cast<const float4*>(op + 4 * a);
  };

  auto store_rows = [&](int id) {
    const Lane here = lane_here();
    int b, i;
    const int j0 = place(id, b, i);
    float* base = p.out + b * p.xv.stride_b + i * p.xv.stride_r;
#pragma unroll
    for (int u = 0; u < TASKS; ++u) {
      const int pos = 4 * (wave + NW * u) + here.lg;
      if (j0 + pos < N) rows.store(base + (j0 + pos) * p.xv.stride_k, pos, here.li);
    }
  };
  int id = grid_slot();
  const int first = id;
  if (id < total) load_rows(id), load_o(id);
  so.finish();  // beside the first tile's loads
  const float o_scale = so.of(tile_unscale), unscale = so.total;
  for (; id < total; id += gridDim.x) {
    const int next = id + (int)gridDim.x < total ? id + (int)gridDim.x : id;
    int b, i;
    const int j0 = place(id, b, i);
    const Lane here = lane_here();
#pragma unroll
    for (int u = 0; u < TASKS; ++u) {
      const int li = here.li, pos = 4 * (wave + NW * u) + here.lg;
      float4 y[C / 64];
      norm_row<C>(raw[u], ln, li, y);
#pragma unroll
      for (int e = 0; e < C / 64; ++e) tile.store4(pos, li + 16 * e, y[e]);
    }
    __syncthreads();  // LayerNorm(x) and the rows of the tile before are complete, and everybody has finished with the second tile
    if (id != first) store_rows(id - gridDim.x);
    if (p.add_residual) {
      const Lane at = lane_here();
#pragma unroll
      for (int u = 0; u < TASKS; ++u) rows.put(4 * (wave + NW * u) + at.lg, at.li, raw[u]);
    }
    load_rows(next);
    const f32x16_t gate = unit_product<C, true>(tile, w.g);
    const Lane mid = lane_here();
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
      const float4 o0 = oraw[2 * hf], o1 = oraw[2 * hf + 1];
      const float ov[8] = {o0.x, o0.y, o0.z, o0.w, o1.x, o1.y, o1.z, o1.w};
      float y[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) y[e] = ov[e] * o_scale * sigmoid_hw_f32(gate[8 * hf + e], g_unscale);
      second.store8(mid.l32, 4 * wave + 2 * mid.lh + hf, y);
    }
    load_o(next);
    __syncthreads();  // the gated output is complete, and everybody has finished with the first tile
    f32x16_t acc = unit_product<C, true>(second, w.o);
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] *= unscale;
    rows.add(wave, acc, p.add_residual);
  }
  if (first >= total) return;  // the whole work-group
  __syncthreads();
  store_rows(id - gridDim.x);
}

template <int C, int NW>
hipError_t launch_trimul_proj(const TrimulF32& p, int panels, int row_groups, long total, hipStream_t stream) {
  constexpr bool kOneSide = C / 32 == NW;
  unsigned grid = 0;
  hipError_t e = resident_grid<trimul_proj_pass<C, NW>>(64 * NW, ProjLds<C>::kBytes, kOneSide ? 2 * total : total, &grid);
  if (e != hipSuccess) return e;
  if (kOneSide) grid &= ~1u;  // a and b
  hipLaunchKernelGGL((trimul_proj_pass<C, NW>), dim3(grid), dim3(64 * NW), ProjLds<C>::kBytes, stream, p, panels, row_groups, (int)total);
  return hipGetLastError();
}
template <int C>
hipError_t launch_trimul_proj(const TrimulF32& p, hipStream_t stream) {
  const int panels = p.Np / 32, row_groups = (p.N + 3) / 4;
  const long total = (long)p.B * row_groups * panels * 4;
  if (total > 0x3fffffffL) return hipErrorInvalidValue;
  if constexpr (C == 128) {
    static int cache[kMaxDevices];
    int cus = 0;
    const hipError_t e = per_device(cache, [](int dev, int* v) { return cu_count(dev, v); }, &cus);
    if (e != hipSuccess) return e;
    if (total > cus) return launch_trimul_proj<C, 8>(p, panels, row_groups, total, stream);
  }
  return launch_trimul_proj<C, 4>(p, panels, row_groups, total, stream);
}

template <int C>
hipError_t launch_trimul_out(const TrimulF32& p, hipStream_t stream) {
  const int panels = p.Np / 32;
  const long total = (long)p.B * p.N * panels;
  if (total > 0x3fffffffL) return hipErrorInvalidValue;
  unsigned grid = 0;
  hipError_t e = resident_grid<trimul_out_pass<C>>(2 * C, OutLds<C>::kTrimul, total, &grid);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(trimul_out_pass<C>, dim3(grid), dim3(2 * C), OutLds<C>::kTrimul, stream, p, panels, (int)total);
  return hipGetLastError();
}

template <int C, int PARTS>
hipError_t launch_triattn_proj(const TriattnF32& p, int panels, long total, hipStream_t stream) {
  unsigned grid = 0;
  hipError_t e = resident_grid<triattn_proj_pass<C, PARTS>>(6 * C / PARTS, AttProjLds<C>::kBytes, PARTS * total, &grid);
  if (e != hipSuccess) return e;
  grid -= grid % PARTS;
  hipLaunchKernelGGL((triattn_proj_pass<C, PARTS>), dim3(grid), dim3(6 * C / PARTS), AttProjLds<C>::kBytes, stream, p, panels,
                     (int)total);
  return hipGetLastError();
}
template <int C>
hipError_t launch_triattn_proj(const TriattnF32& p, hipStream_t stream) {
  const int panels = p.Jp / 32;
  const long total = (long)p.B * p.N * panels;
  if (total > 0x3fffffffL) return hipErrorInvalidValue;
  static int cache[kMaxDevices];
  int cus = 0;
  const hipError_t e = per_device(cache, [](int dev, int* v) { return cu_count(dev, v); }, &cus);
  if (e != hipSuccess) return e;
  // One / two / four work-groups per tile, us: four trunk blocks at N = 64 615 / 612 / 624, 45 599 / 591 / 599, 30 558 / 546 / 551, a pair stack
  // at 64 112 / 110 / 111, and with more tiles than half of the CUs, at 80, 137 / 142 / 143.
  if (C == 128 && 2 * total <= cus) return launch_triattn_proj<C, C == 128 ? 2 : 1>(p, panels, total, stream);
  return launch_triattn_proj<C, 1>(p, panels, total, stream);
}

template <int C>
hipError_t launch_triattn_out(const TriattnF32& p, hipStream_t stream) {
  const int panels = p.Jp / 32;
  const long total = (long)p.B * p.N * panels;
  if (total > 0x3fffffffL) return hipErrorInvalidValue;
  unsigned grid = 0;
  hipError_t e = resident_grid<triattn_out_pass<C>>(2 * C, OutLds<C>::kTriattn, total, &grid);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(triattn_out_pass<C>, dim3(grid), dim3(2 * C), OutLds<C>::kTriattn, stream, p, panels, (int)total);
  return hipGetLastError();
}

}  // namespace

bool trimul_pass_serves(const TrimulF32& p) {
  return trimul_half_shapes(p.B, p.N, p.C, p.CH) && rows_aligned(p.z, p.zv) && rows_aligned(p.out, p.zc);
}
hipError_t trimul_proj_pass_f32(const TrimulF32& p, hipStream_t stream) {
  return p.C == 128 ? launch_trimul_proj<128>(p, stream) : launch_trimul_proj<64>(p, stream);
}
hipError_t trimul_out_pass_f32(const TrimulF32& p, hipStream_t stream) {
  return p.C == 128 ? launch_trimul_out<128>(p, stream) : launch_trimul_out<64>(p, stream);
}

bool triattn_pass_serves(const TriattnF32& p) {
  return triattn_half_shapes(p.B, p.N, p.C, p.H, p.D) && rows_aligned(p.x, p.xv) && rows_aligned(p.out, p.xv);
}
hipError_t triattn_proj_pass_f32(const TriattnF32& p, hipStream_t stream) {
  return p.C == 128 ? launch_triattn_proj<128>(p, stream) : launch_triattn_proj<64>(p, stream);
}
hipError_t triattn_out_pass_f32(const TriattnF32& p, hipStream_t stream) {
  return p.C == 128 ? launch_triattn_out<128>(p, stream) : launch_triattn_out<64>(p, stream);
}

}  // namespace of3
