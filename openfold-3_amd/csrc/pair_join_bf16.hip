// bf16: the output pass of one triangle module and the input pass of the next in one launch, for the lengths at which a
// work-group's share of the pair tensor is one tile.
//
// Between two cores (contraction, attention) a pair stack ends one module and begins the next, position by position: gate,
// output projection, residual, LayerNorm, projections.  As two launches (trimul_out / triattn_out, trimul_proj / triattn_proj)
// each costs 2 us to launch, 2.7 us until its 64 to 164 KB of weights and its tile have come through the L1 (64 B per clock
// and CU), and a trip of z to memory and back; up to N = 220 that is half of their time.  Here a work-group of 8 waves takes R rows
// x one 32-position panel in the frame of the second module, R chosen so that every CU has one tile (two at 64 channels), and
// keeps it: the updated z goes to memory and, through LDS, into the second half.  The second half's weights are requested before
// the first half's products.  The contraction before a join of two multiplications writes x in the second one's frame,
// so that both halves walk rows of the same frame.
// Same operations and rounding points as the passes by themselves (the same bits).  What bounds it: up to two rows the chain of
// loads, LayerNorms, barriers and products (9 us of kernel at N = 80: 2.4 until the loads are issued, 1.1 the first LayerNorm,
// 1.3 x, 1.1 the update, 1.5 LayerNorm and projections); at six rows the vector instructions of the three LayerNorms (6.5 of
// 25 us) and the gates beside the products.
#include "of3_device.h"
#include "of3_kernels.h"
#include "of3_launch.h"
#include "of3_pass_bf16.h"

#include <type_traits>

namespace of3 {

namespace {

using namespace pass_bf16;

constexpr int kWaves = 8;

template <int C>
constexpr int waves_per_simd() {  // one work-group per CU at 128 channels, two at 64
  return C == 128 ? 2 : 4;
}

// LayerNorm tasks of a tile of R panels: an instruction's positions, `task` of the wave's u-th
template <int C, int R>
struct Tasks {
  static constexpr int PER_PANEL = 32 / LnLane<C>::PPI, ALL = R * PER_PANEL, MINE = (ALL + kWaves - 1) / kWaves;
  __device__ __forceinline__ static bool exists(int task) { return ALL % kWaves == 0 || task < ALL; }
  __device__ __forceinline__ static int panel(int task) { return task / PER_PANEL; }
  __device__ __forceinline__ static int pos(int task) { return task % PER_PANEL * LnLane<C>::PPI + LnLane<C>::pos(); }
};

template <int C>
__device__ __forceinline__ int plain_slot(int panel, int pos, int chunk) {
  return panel * PanelTile<C, false>::SLOTS + PanelTile<C, false>::slot(pos, chunk);
}

struct JoinTile {
  int b, r0, k0;        // batch element, first row, first column, in the frame of the second half
  int64_t sb, sr, sk;   // of z in that frame
};

// the lanes' share of an updated panel: added to the residual, rounded, to memory and back into the residual's slots
template <int C>
__device__ __forceinline__ void finish_update(bf16_t* out, const JoinTile& t, int N, int add_residual, u32x4_t* rtile,
                                              int q, int ot, int l32, int lh, float (&res)[16]) {
  u32x4_t* const s0 = rtile + plain_slot<C>(q, l32, 4 * ot + 2 * lh);
  u32x4_t* const s1 = rtile + plain_slot<C>(q, l32, 4 * ot + 2 * lh + 1);
  if (add_residual) {
    float r[8];
    unpack8(*s0, r);
#pragma unroll
    for (int v = 0; v < 8; ++v) res[v] += r[v];
    unpack8(*s1, r);
#pragma unroll
    for (int v = 0; v < 8; ++v) res[8 + v] += r[v];
  }
  u32x4_t o[2];
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    o[0][w] = pack_bf16(res[2 * w], res[2 * w + 1]);
    o[1][w] = pack_bf16(res[8 + 2 * w], res[8 + 2 * w + 1]);
  }
  *s0 = o[0];
  *s1 = o[1];
  if (t.r0 + q < N && t.k0 + l32 < N) {
    bf16_t* dst = out + t.b * t.sb + (t.r0 + q) * t.sr + (t.k0 + l32) * t.sk + 32 * ot + 16 * lh;
    *reinterpret_cast<u32x4_t*>(dst) = o[0];
    *reinterpret_cast<u32x4_t*>(dst + 8) = o[1];
  }
}

// ---- first halves -------------------------------------------------------------------------------------------
// load: what is read before the weights; stage: into LDS; then (after a barrier) middle, (after another) update.
template <int C, int R>
struct TrimulEnd {
  typedef TrimulOutArgs Args;
  static constexpr int KS = C / 16, OT = C / 32, GROUPS = kWaves / OT;  // waves that share an output tile take every GROUPS-th panel
  static constexpr int ITEMS = C / 2 * 4 * R, XR = (ITEMS + 511) / 512;  // channel pairs x 8-position groups
  u32x4_t xa[XR], xb[XR], wg[KS], wz[KS];
  LnLane<C> lz, lx;
  __device__ __forceinline__ void load(const Args& p, const JoinTile& t) {
    const size_t plane = (size_t)p.Np * p.Np;
#pragma unroll
    for (int u = 0; u < XR; ++u) {
      const int item = u * 512 + threadIdx.x;
      if (ITEMS % 512 != 0 && item >= ITEMS) break;
      const int q = item / (C * 2), cp = item % (C * 2) >> 2, pg = item & 3;
      const int r = t.r0 + q < p.N ? t.r0 + q : p.N - 1;
      const bf16_t* src = p.x + ((size_t)t.b * C + 2 * cp) * plane + (size_t)r * p.Np + t.k0 + 8 * pg;  // rows are padded to Np
      xa[u] = *reinterpret_cast<const u32x4_t*>(src);
      xb[u] = *reinterpret_cast<const u32x4_t*>(src + plane);
    }
  }
  __device__ __forceinline__ void load_weights(const Args& p, int wave, int lane) {
    lz = ln_lane<C>(p.ln_in_w, p.ln_in_b, lane);
    lx = ln_lane<C>(p.ln_out_w, p.ln_out_b, lane);
    if (R < GROUPS && wave / OT >= R) return;  // has no panel
    load_unit<C>(p.w_z, wave % OT, rowperm16(lane & 31), lane >> 5, 1, wz);
    load_unit<C>(p.w_g, wave % OT, rowperm16(lane & 31), lane >> 5, 1, wg);
  }
  // x channel-major into position-major order, 4-byte (channel pair) writes
  __device__ __forceinline__ void stage(u32x4_t* xtile) {
    uint32_t* const x32 = reinterpret_cast<uint32_t*>(xtile);
#pragma unroll
    for (int u = 0; u < XR; ++u) {
      const int item = u * 512 + threadIdx.x;
      if (ITEMS % 512 != 0 && item >= ITEMS) break;
      const int q = item / (C * 2), cp = item % (C * 2) >> 2, pg = item & 3;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const uint32_t ua = xa[u][e >> 1], ub = xb[u][e >> 1];
        x32[plain_slot<C>(q, 8 * pg + e, cp >> 2) * 4 + (cp & 3)] =
            __builtin_amdgcn_perm(ub, ua, (e & 1) ? 0x07060302u : 0x05040100u);
      }
    }
  }
  __device__ __forceinline__ void middle(u32x4_t* /*ntile*/, u32x4_t* xtile, int wave) {  // LayerNorm of x in place
    typedef Tasks<C, R> T;
    float lw[8], lb[8];
    lx.template unpacked<false>(lw, lb);
    int slot[T::MINE];
    u32x4_t x[T::MINE];  // all of them read before the first is written: the compiler cannot tell that they do not overlap
#pragma unroll
    for (int u = 0; u < T::MINE; ++u) {
      const int task = wave + kWaves * u;
      slot[u] = T::exists(task) ? plain_slot<C>(T::panel(task), T::pos(task), LnLane<C>::chunk()) : 0;
      x[u] = xtile[slot[u]];
    }
#pragma unroll
    for (int u = 0; u < T::MINE; ++u)
      if (T::exists(wave + kWaves * u)) xtile[slot[u]] = layer_norm_chunk<C>(x[u], lw, lb);
  }
  __device__ __forceinline__ void update(const Args& p, const JoinTile& t, u32x4_t* ntile, u32x4_t* xtile, u32x4_t* rtile, int wave) {
    const int ot = wave % OT;
#pragma unroll
    for (int q0 = 0; q0 < R; q0 += GROUPS) {
      const int q = q0 + wave / OT;
      if (R % GROUPS != 0 && q >= R) break;
      const Lane at = lane_here();
      const int l32 = at.l32, lh = at.lh;
      f32x16_t ag = zero16(), az = zero16();
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const int slot = plain_slot<C>(q, l32, 2 * s + lh);
        az = mfma_32x32x16(wz[s], xtile[slot], az);
        ag = mfma_32x32x16(wg[s], ntile[slot], ag);
      }
      float res[16];
#pragma unroll
      for (int e = 0; e < 16; ++e) res[e] = az[e] * sigmoid_from_scaled(ag[e]);
      finish_update<C>(p.out, t, p.N, p.add_residual, rtile, q, ot, l32, lh, res);
    }
  }
};

template <int C, int R>
struct TriattnEnd {
  typedef TriattnOutArgs Args;
  static constexpr int KS = C / 16, OT = C / 32, GROUPS = kWaves / OT, MINE = (R + GROUPS - 1) / GROUPS;
  u32x4_t o[MINE][2], wg[KS], wo[KS];
  LnLane<C> lz;
  __device__ __forceinline__ void load(const Args& p, const JoinTile& t) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const Lane at = lane_here();
    // o [B][N][N][C] is a tensor of the attention's frame; the module after an attention walks the transposed one
    const int64_t o_r = C, o_k = (int64_t)p.N * C;
    const int k = t.k0 + at.l32 < p.N ? t.k0 + at.l32 : p.N - 1;
#pragma unroll
    for (int m = 0; m < MINE; ++m) {
      const int q = m * GROUPS + wave / OT;
      const int r = t.r0 + q < p.N ? t.r0 + q : p.N - 1;
      const bf16_t* src = p.o + (int64_t)t.b * p.N * p.N * C + r * o_r + k * o_k + 32 * (wave % OT) + 16 * at.lh;
      o[m][0] = *reinterpret_cast<const u32x4_t*>(src);
      o[m][1] = *reinterpret_cast<const u32x4_t*>(src + 8);
    }
  }
  __device__ __forceinline__ void load_weights(const Args& p, int wave, int lane) {
    lz = ln_lane<C>(p.ln_w, p.ln_b, lane);
    if (R < GROUPS && wave / OT >= R) return;  // has no panel
    load_unit<C>(p.w_g, wave % OT, rowperm16(lane & 31), lane >> 5, 1, wg);
    load_unit<C>(p.w_o, wave % OT, rowperm16(lane & 31), lane >> 5, 1, wo);
  }
  __device__ __forceinline__ void stage(u32x4_t* /*otile*/) {}
  __device__ __forceinline__ void middle(u32x4_t* ntile, u32x4_t* otile, int wave) {  // o times its gate
    const int ot = wave % OT;
#pragma unroll
    for (int m = 0; m < MINE; ++m) {
      const int q = m * GROUPS + wave / OT;
      if (R % GROUPS != 0 && q >= R) break;
      const Lane at = lane_here();
      const int l32 = at.l32, lh = at.lh;
      f32x16_t acc = zero16();
#pragma unroll
      for (int s = 0; s < KS; ++s) acc = mfma_32x32x16(wg[s], ntile[plain_slot<C>(q, l32, 2 * s + lh)], acc);
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        float ov[8];
        unpack8(o[m][half], ov);
#pragma unroll
        for (int v = 0; v < 8; ++v) ov[v] *= sigmoid_from_scaled(acc[8 * half + v]);
        otile[plain_slot<C>(q, l32, 4 * ot + 2 * lh + half)] = pack8(ov);
      }
    }
  }
  __device__ __forceinline__ void update(const Args& p, const JoinTile& t, u32x4_t* /*ntile*/, u32x4_t* otile, u32x4_t* rtile, int wave) {
    const int ot = wave % OT;
#pragma unroll
    for (int m = 0; m < MINE; ++m) {
      const int q = m * GROUPS + wave / OT;
      if (R % GROUPS != 0 && q >= R) break;
      const Lane at = lane_here();
      const int l32 = at.l32, lh = at.lh;
      f32x16_t acc = zero16();
#pragma unroll
      for (int s = 0; s < KS; ++s) acc = mfma_32x32x16(wo[s], otile[plain_slot<C>(q, l32, 2 * s + lh)], acc);
      float res[16];
#pragma unroll
      for (int v = 0; v < 16; ++v) res[v] = acc[v];
      finish_update<C>(p.out, t, p.N, p.add_residual, rtile, q, ot, l32, lh, res);
    }
  }
};

// ---- second halves ------------------------------------------------------------------------------------------
template <int C, int R>
struct TrimulStart {
  typedef TrimulProjArgs Args;
  static constexpr int KS = C / 16, OT = C / 32, GROUPS = kWaves / (2 * OT);
  u32x4_t wg[KS], wp[KS];
  __device__ __forceinline__ static JoinTile frame(const Args& p) { return {0, 0, 0, p.z_view.stride_b, p.z_view.stride_r, p.z_view.stride_k}; }
  __device__ __forceinline__ void load_weights(const Args& p, int wave, int lane) {
    const bool pair = wave / OT & 1;
    load_unit<C>(pair ? p.w_bg : p.w_ag, wave % OT, lane & 31, lane >> 5, 1, wg);
    load_unit<C>(pair ? p.w_bp : p.w_ap, wave % OT, lane & 31, lane >> 5, 1, wp);
  }
  __device__ __forceinline__ void take_mask(const Args& p, const JoinTile& t, int q, int pos, float m, float* msk) {
    msk[32 * q + pos] = t.k0 + pos < p.N ? m : 0.f;
  }
  __device__ __forceinline__ void project(const Args& p, const JoinTile& t, u32x4_t* ntile, const float* msk, int wave) {
    typedef PanelTile<C, true> Tile;
    const int ot = wave % OT, pair = wave / OT & 1;
#pragma unroll
    for (int q0 = 0; q0 < R; q0 += GROUPS) {
      const int q = q0 + wave / (2 * OT);
      if ((R % GROUPS != 0 && q >= R) || t.r0 + q >= p.N) break;
      const Tile tile = {ntile + q * Tile::SLOTS};
      const Lane at = lane_here();
      const int l32 = at.l32, lh = at.lh;
      const bool masked = __builtin_amdgcn_ballot_w64(msk[32 * q + l32] != 1.f) != 0;
      f32x16_t ag = zero16(), ap = zero16();
      const int pos = rowperm16(l32);
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const u32x4_t x = tile.s[Tile::slot(pos, 2 * s + lh)];
        ag = mfma_32x32x16(x, wg[s], ag);
        ap = mfma_32x32x16(x, wp[s], ap);
      }
      float res[16];
      if (masked) {
#pragma unroll
        for (int a = 0; a < 4; ++a) {
          const float4 m = *reinterpret_cast<const float4*>(msk + 32 * q + 16 * lh + 4 * a);
          const float mv[4] = {m.x, m.y, m.z, m.w};
#pragma unroll
          for (int e = 0; e < 4; ++e) res[4 * a + e] = (mv[e] * sigmoidf_fast(ag[4 * a + e])) * ap[4 * a + e];
        }
      } else {
#pragma unroll
        for (int v = 0; v < 16; ++v) res[v] = sigmoidf_fast(ag[v]) * ap[v];
      }
      bf16_t* dst = (pair ? p.b : p.a) + ((size_t)t.b * C + 32 * ot + l32) * ((size_t)p.Np * p.Np) + (size_t)(t.k0 >> 5) * (p.Np * 32) +
                    (t.r0 + q) * 32 + 16 * lh;
      store16(dst, res);
    }
  }
};

template <int C, int R>
struct TriattnStart {
  typedef TriattnProjArgs Args;
  static constexpr int KS = C / 16, OT = C / 32, D = C / 4;
  // 128 channels: waves 0..3 a tile of q and of k, 4..7 one of v and the triangle bias of every fourth panel;
  // 64: waves 0..5 a tile of q, k or v, 6 and 7 the bias
  u32x4_t w0[KS], w1[KS];
  __device__ __forceinline__ static JoinTile frame(const Args& p) { return {0, 0, 0, p.x_view.stride_b, p.x_view.stride_r, p.x_view.stride_k}; }
  __device__ __forceinline__ void load_weights(const Args& p, int wave, int lane) {
    if (C == 128) {
      load_attention_unit<C>(p, wave < 4 ? 0 : 2, wave % 4, lane, w0);
      load_attention_unit<C>(p, wave < 4 ? 1 : 3, wave % 4, lane, w1);
    } else {
      load_attention_unit<C>(p, wave / 2, wave % 2, lane, w0);
    }
  }
  __device__ __forceinline__ void take_mask(const Args& p, const JoinTile& t, int q, int pos, float m, float* /*msk*/) {
    if (t.r0 + q < p.N) store_mask_bias(p, t.b * p.N + t.r0 + q, t.k0 + pos, m);
  }
  __device__ __forceinline__ void project(const Args& p, const JoinTile& t, u32x4_t* ntile, const float* /*msk*/, int wave) {
    typedef PanelTile<C, true> Tile;
#pragma unroll
    for (int q = 0; q < R; ++q) {
      if (t.r0 + q >= p.N) break;
      const Tile tile = {ntile + q * Tile::SLOTS};
      const int bi = t.b * p.N + t.r0 + q;
      if (C == 128) {
        if (wave < 4) {
          project_panel<C, D>(p, w0, tile, 0, wave, bi, t.k0);
          project_panel<C, D>(p, w1, tile, 1, wave, bi, t.k0);
        } else {
          project_panel<C, D>(p, w0, tile, 2, wave - 4, bi, t.k0);
          if (q % 4 == wave - 4) project_panel<C, D>(p, w1, tile, 3, 0, bi, t.k0);
        }
      } else if (wave < 6) {
        project_panel<C, D>(p, w0, tile, wave / 2, wave % 2, bi, t.k0);
      } else if (q % 2 == wave - 6) {
        project_panel<C, D>(p, w0, tile, 3, 0, bi, t.k0);
      }
    }
  }
};

template <int C, int R, template <int, int> class End, template <int, int> class Start>
__global__ __launch_bounds__(64 * kWaves, waves_per_simd<C>()) void pair_join(typename End<C, R>::Args e, typename Start<C, R>::Args s,
                                                                             Division by_panels, Division by_batch) {
  typedef Tasks<C, R> T;
  typedef LnLane<C> Ln;
  constexpr int TILE = R * PanelTile<C, false>::SLOTS;
  extern __shared__ u32x4_t lds[];
  u32x4_t* const ntile = lds;              // LayerNorm(z), then LayerNorm of the updated z
  u32x4_t* const xtile = lds + TILE;       // x or o
  u32x4_t* const rtile = lds + 2 * TILE;   // z, then the updated z
  float* const msk = reinterpret_cast<float*>(lds + 3 * TILE);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int N = e.N;
  JoinTile t = Start<C, R>::frame(s);
  {
    const int id = grid_slot();
    t.b = by_batch.quotient(id);
    const int rem = id - t.b * by_batch.d, rg = by_panels.quotient(rem);
    t.r0 = R * rg;
    t.k0 = 32 * (rem - rg * by_panels.d);
  }
  End<C, R> end;
  Start<C, R> start;
  u32x4_t raw[T::MINE];
  float mraw[T::MINE];
  const bf16_t* z;
  if constexpr (std::is_same<typename End<C, R>::Args, TrimulOutArgs>::value) z = e.z;
  else z = e.x;
#pragma unroll
  for (int u = 0; u < T::MINE; ++u) {
    const int task = wave + kWaves * u;
    mraw[u] = 1.f;
    if (!T::exists(task)) break;
    int r = t.r0 + T::panel(task), k = t.k0 + T::pos(task);  // clamped to real positions
    r = r < N ? r : N - 1;
    k = k < N ? k : N - 1;
    raw[u] = *reinterpret_cast<const u32x4_t*>(z + t.b * t.sb + r * t.sr + k * t.sk + 8 * Ln::chunk());
    if (s.mask) mraw[u] = s.mask[t.b * s.mask_view.stride_b + r * s.mask_view.stride_r + k * s.mask_view.stride_k];
  }
  end.load(e, t);
  end.load_weights(e, wave, lane);
  const Ln ln = ln_lane<C>(s.ln_w, s.ln_b, lane);

  float lw[8], lb[8];
  end.lz.template unpacked<true>(lw, lb);
#pragma unroll
  for (int u = 0; u < T::MINE; ++u) {
    const int task = wave + kWaves * u;
    if (!T::exists(task)) break;
    const int slot = plain_slot<C>(T::panel(task), T::pos(task), Ln::chunk());
    ntile[slot] = layer_norm_chunk<C>(raw[u], lw, lb);
    rtile[slot] = raw[u];
    if (Ln::chunk() == 0) start.take_mask(s, t, T::panel(task), T::pos(task), mraw[u], msk);
  }
  end.stage(xtile);
  __syncthreads();
  start.load_weights(s, wave, lane);  // they arrive under the first half
  end.middle(ntile, xtile, wave);
  __syncthreads();
  end.update(e, t, ntile, xtile, rtile, wave);
  __syncthreads();
  ln.template unpacked<false>(lw, lb);
#pragma unroll
  for (int u = 0; u < T::MINE; ++u) {
    const int task = wave + kWaves * u;
    if (!T::exists(task)) break;
    // positions past the end are copies of the last one, as where the pass reads them itself
    int q = T::panel(task), pos = T::pos(task);
    q = t.r0 + q < N ? q : N - 1 - t.r0;
    pos = t.k0 + pos < N ? pos : N - 1 - t.k0;
    raw[u] = rtile[plain_slot<C>(q, pos, Ln::chunk())];
  }
#pragma unroll
  for (int u = 0; u < T::MINE; ++u) {
    const int task = wave + kWaves * u;
    if (!T::exists(task)) break;
    ntile[T::panel(task) * PanelTile<C, true>::SLOTS + PanelTile<C, true>::slot(T::pos(task), Ln::chunk())] = layer_norm_chunk<C>(raw[u], lw, lb);
  }
  __syncthreads();
  start.project(s, t, ntile, msk, wave);
}

template <int C, int R>
constexpr size_t join_lds() {
  return (size_t)3 * R * PanelTile<C, false>::SLOTS * 16 + R * 32 * sizeof(float);
}

template <int C, int R, template <int, int> class End, template <int, int> class Start>
hipError_t launch_rows(const typename End<C, R>::Args& e, const typename Start<C, R>::Args& s, hipStream_t stream) {
  constexpr size_t lds = join_lds<C, R>();
  const hipError_t err = allow_dynamic_lds<pair_join<C, R, End, Start>>(lds);
  if (err != hipSuccess) return err;
  const int panels = (e.N + 31) / 32, row_groups = (e.N + R - 1) / R;
  hipLaunchKernelGGL((pair_join<C, R, End, Start>), dim3((unsigned)(e.B * panels * row_groups)), dim3(64 * kWaves), lds, stream, e, s,
                     Division::by(panels), Division::by(panels * row_groups));
  return hipGetLastError();
}

template <int C, template <int, int> class End, template <int, int> class Start>
hipError_t launch(const typename End<C, 1>::Args& e, const typename Start<C, 1>::Args& s, hipStream_t stream) {
  if (e.B != s.B || e.N != s.N) return hipErrorInvalidValue;
  int rows = 0;
  const hipError_t err = join_rows(e.B, e.N, C, &rows);
  if (err != hipSuccess) return err;
  switch (rows) {
    case 1: return launch_rows<C, 1, End, Start>(e, s, stream);
    case 2: return launch_rows<C, 2, End, Start>(e, s, stream);
    case 3: return launch_rows<C, 3, End, Start>(e, s, stream);
    case 4: return launch_rows<C, 4, End, Start>(e, s, stream);
    case 5: return launch_rows<C, 5, End, Start>(e, s, stream);
    case 6: return launch_rows<C, 6, End, Start>(e, s, stream);
  }
  return hipErrorInvalidValue;
}

}  // namespace

hipError_t join_rows(int B, int N, int C, int* rows) {
  *rows = 0;
  if ((C != 128 && C != 64) || N > kJoinTokens) return hipSuccess;
  static int cache[kMaxDevices];
  int cus = 0;
  const hipError_t e = per_device(cache, [](int dev, int* v) { return cu_count(dev, v); }, &cus);
  if (e != hipSuccess) return e;
  // The fewest rows with which all tiles run at once (one work-group per CU at 128 channels, two at 64).  Three joins against
  // their six passes, us, 256 CUs, packed weights; 128 channels: N = 40 24 / 30, 80 32 / 38, 128 45 / 56, 160 62 / 70, 200 (six
  // rows) 82 / 86; 64 channels: 2 x 100 39 / 46, 2 x 187 57 / 72, 2 x 205 66 / 87, 1 x 256 50 / 78.  At 64 channels, where two
  // work-groups cover each other's waits, four rows stay the better up to three rounds (3 x 220 100 / 118, 4 x 187 96 / 110), which
  // is also what the workspace has room for (join_room).  At four, 4 x 256, the launches are level (168 / 169 in a trace) and the
  // contraction that writes x transposed takes 27 us in place of 21: two blocks 788 / 782; in between, 4 x 225 (3.6 rounds), they would
  // still gain, 712 / 742.  At 128 a second round costs what the join saves.
  const long slots = (C == 128 ? 1 : 2) * (long)cus, panels = (N + 31) / 32;
  auto tiles = [&](int r) { return B * (long)((N + r - 1) / r) * panels; };
  for (int r = 1; r <= 6 && *rows == 0; ++r)
    if (tiles(r) <= slots) *rows = r;
  if (*rows == 0 && C == 64 && tiles(4) <= 3 * slots) *rows = 4;
  return hipSuccess;
}
hipError_t trimul_trimul_launch(const TrimulOutArgs& e, const TrimulProjArgs& s, int C, hipStream_t stream) {
  return C == 128 ? launch<128, TrimulEnd, TrimulStart>(e, s, stream) : launch<64, TrimulEnd, TrimulStart>(e, s, stream);
}
hipError_t trimul_triattn_launch(const TrimulOutArgs& e, const TriattnProjArgs& s, int C, hipStream_t stream) {
  return C == 128 ? launch<128, TrimulEnd, TriattnStart>(e, s, stream) : launch<64, TrimulEnd, TriattnStart>(e, s, stream);
}
hipError_t triattn_triattn_launch(const TriattnOutArgs& e, const TriattnProjArgs& s, int C, hipStream_t stream) {
  return C == 128 ? launch<128, TriattnEnd, TriattnStart>(e, s, stream) : launch<64, TriattnEnd, TriattnStart>(e, s, stream);
}
// Only blocks whose attentions come first have this boundary.  Such blocks, us, with this launch / its two passes / no join at all: 64
// channels 64 57.2 / 60.2 / 65.0, 2 x 100 86.6 / 88.5 / 99.8, 2 x 187 161.1 / 164.4 / 170.8, 4 x 187 245.5 / 250.0 / 257.8; 128 channels
// 64 64.1 / 67.5 / 74.7, 160 138.1 / 140.8 / 145.1, 200 188.1 / 190.9 / 193.4.
hipError_t triattn_trimul_launch(const TriattnOutArgs& e, const TrimulProjArgs& s, int C, hipStream_t stream) {
  return C == 128 ? launch<128, TriattnEnd, TrimulStart>(e, s, stream) : launch<64, TriattnEnd, TrimulStart>(e, s, stream);
}

}  // namespace of3
