// bf16 position-wise passes of the two triangle modules on tiles of 32 positions, for short sequences.
//
// The passes of trimul_proj / trimul_out / triattn_proj / triattn_out.hip walk tiles of 128 positions with one
// work-group per CU, the right split once every CU has several tiles.  A pair tensor of 40 tokens is 13 such tiles and
// one of 200 tokens 313 on 256 CUs: most of the chip idles, or waits for a second, nearly empty round, and every step of
// the chain load -> LayerNorm -> products -> stores is four times as long as it has to be.  Here a tile is one
// 32-position panel of a row, a wave owns one 32-output tile of one or two matrices (64 registers of weights at 128
// channels, about 100 registers in all), and two or more work-groups share a CU.  Same operations and rounding points.
// The launchers of the 128-position passes say up to where these are the faster ones.
#include "of3_device.h"
#include "of3_kernels.h"
#include "of3_launch.h"
#include "of3_pass_bf16.h"

namespace of3 {

namespace {

using namespace pass_bf16;

// ---- triangle multiplication, input pass (trimul_proj.hip) ---------------------------------------------------
// Wave = gate and projection of one 32-channel tile of a or b.  The positions are the MFMA rows, dealt by rowperm16: a
// lane ends with 16 consecutive k of one channel, 32 bytes of the panel row.
template <int C>
__global__ __launch_bounds__(4 * C, 4) void trimul_proj_panels(TrimulProjArgs p, int panels, int row_groups, int total) {
  typedef PanelTile<C, true> Tile;
  constexpr int NW = C / 16, KS = C / 16, OT = C / 32;
  __shared__ u32x4_t tiles[2][Tile::SLOTS];
  __shared__ __align__(16) float msk[2][32];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int pair = wave / OT, ot = wave % OT, N = p.N, Np = p.Np;
  const LnLane<C> ln = ln_lane<C>(p.ln_w, p.ln_b, lane);
  u32x4_t wg[KS], wp[KS];
  load_unit<C>(pair ? p.w_bg : p.w_ag, ot, lane & 31, lane >> 5, p.packed, wg);
  load_unit<C>(pair ? p.w_bp : p.w_ap, ot, lane & 31, lane >> 5, p.packed, wp);

  struct Place {
    int b, r, k0;
  };
  auto place = [&](int id) {  // four consecutive rows of a panel are consecutive tiles
    Place t;
    const int q = id & 3, rest = id >> 2, per_b = row_groups * panels;
    t.b = rest / per_b;
    const int rem = rest - t.b * per_b, rg = rem / panels;
    t.r = 4 * rg + q;
    t.k0 = 32 * (rem - rg * panels);
    return t;
  };
  u32x4_t raw;
  float mraw = 1.f;
  auto load_tile = [&](int id) {
    const int ln_chunk = ln.chunk(), ln_pos = ln.pos();
    const Lane here = lane_here();
    const int l32 = here.l32;
    // addresses clamped to real positions: no load is under a condition
    const Place t = place(id);
    const int r = t.r < N ? t.r : N - 1;
    int k = t.k0 + wave * ln.PPI + ln_pos;
    k = k < N ? k : N - 1;
    raw = *reinterpret_cast<const u32x4_t*>(p.z + t.b * p.z_view.stride_b + r * p.z_view.stride_r + k * p.z_view.stride_k + 8 * ln_chunk);
    k = t.k0 + l32 < N ? t.k0 + l32 : N - 1;
    if (p.mask) mraw = p.mask[t.b * p.mask_view.stride_b + r * p.mask_view.stride_r + k * p.mask_view.stride_k];
  };

  int id = grid_slot(), buf = 0;
  if (id < total) load_tile(id);
  for (; id < total; id += gridDim.x, buf ^= 1) {
    const Place t = place(id);
    const Tile tile = {tiles[buf]};
    tile.s[Tile::slot(wave * ln.PPI + ln.pos(), ln.chunk())] = ln.template normalised<false>(raw);
    if (tid < 32) msk[buf][tid] = t.k0 + tid < N ? mraw : 0.f;
    load_tile(id + (int)gridDim.x < total ? id + gridDim.x : id);
    __syncthreads();  // the tile is complete, everybody has finished with the other one
    if (t.r >= N) continue;
    const Lane at = lane_here();
    const int l32 = at.l32, lh = at.lh;
    const bool masked = __builtin_amdgcn_ballot_w64(msk[buf][l32] != 1.f) != 0;
    f32x16_t ag = zero16(), ap = zero16();
    const int pos = rowperm16(l32);
    u32x4_t next = tile.s[Tile::slot(pos, lh)];
#pragma unroll
    for (int s = 0; s < KS; ++s) {  // operands one step ahead, no further: 128 registers
      const u32x4_t x = next;
      if (s + 1 < KS) next = tile.s[Tile::slot(pos, 2 * (s + 1) + lh)];
      __builtin_amdgcn_sched_barrier(0);
      ag = mfma_32x32x16(x, wg[s], ag);
      ap = mfma_32x32x16(x, wp[s], ap);
      __builtin_amdgcn_sched_barrier(0);
    }
    float res[16];
    if (masked) {
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        const float4 m = *reinterpret_cast<const float4*>(&msk[buf][16 * lh + 4 * a]);
        const float mv[4] = {m.x, m.y, m.z, m.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) res[4 * a + e] = (mv[e] * sigmoidf_fast(ag[4 * a + e])) * ap[4 * a + e];
      }
    } else {
#pragma unroll
      for (int v = 0; v < 16; ++v) res[v] = sigmoidf_fast(ag[v]) * ap[v];
    }
    bf16_t* dst = (pair ? p.b : p.a) + ((size_t)t.b * C + 32 * ot + l32) * ((size_t)Np * Np) + (size_t)(t.k0 >> 5) * (Np * 32) +
                  t.r * 32 + 16 * lh;
    store16(dst, res);
  }
}

// ---- triangle multiplication, output pass (trimul_out.hip) ---------------------------------------------------
// Wave = one 32-channel tile of the gate and of the output projection.  x is channel-major: thread (position pair
// tid % 16, chunk tid / 16) holds 8 channels of two positions, which go into position-major order through LDS.
template <int C>
__global__ __launch_bounds__(2 * C, 3) void trimul_out_panels(TrimulOutArgs p, int panels, int total) {
  typedef PanelTile<C, false> Tile;
  constexpr int NW = C / 32, KS = C / 16, TASKS = 32 / LnLane<C>::PPI / NW;
  __shared__ u32x4_t ztiles[2][Tile::SLOTS], xtiles[2][Tile::SLOTS];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int N = p.N, Np = p.Np;
  const LnLane<C> ln = ln_lane<C>(p.ln_in_w, p.ln_in_b, lane), lx = ln_lane<C>(p.ln_out_w, p.ln_out_b, lane);
  const int xp = tid & 15, xc = tid >> 4;  // position pair and chunk of x
  u32x4_t wg[KS], wz[KS];
  load_unit<C>(p.w_g, wave, rowperm16(lane & 31), lane >> 5, p.packed, wg);
  load_unit<C>(p.w_z, wave, rowperm16(lane & 31), lane >> 5, p.packed, wz);

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
  u32x4_t raw[TASKS];
  uint32_t xraw[8];
  auto load_tile = [&](int id) {
    const int ln_chunk = ln.chunk(), ln_pos = ln.pos();
    const Place t = place(id);
    const bf16_t* base = p.z + t.b * p.z_view.stride_b + t.i * p.z_view.stride_r + 8 * ln_chunk;
#pragma unroll
    for (int u = 0; u < TASKS; ++u) {
      int j = t.j0 + (wave + NW * u) * ln.PPI + ln_pos;
      j = j < N ? j : N - 1;
      raw[u] = *reinterpret_cast<const u32x4_t*>(base + j * p.z_view.stride_k);
    }
    const bf16_t* x = p.x + (((size_t)t.b * C + 8 * xc) * Np + t.i) * Np + t.j0 + 2 * xp;  // planes are padded: always inside
#pragma unroll
    for (int e = 0; e < 8; ++e) xraw[e] = *reinterpret_cast<const uint32_t*>(x + (size_t)e * Np * Np);
  };

  int id = grid_slot(), buf = 0;
  if (id < total) load_tile(id);
  for (; id < total; id += gridDim.x, buf ^= 1) {
    const Place t = place(id);
    const Tile zn = {ztiles[buf]}, xn = {xtiles[buf]};
#pragma unroll
    for (int u = 0; u < TASKS; ++u) zn.s[Tile::slot((wave + NW * u) * ln.PPI + ln.pos(), ln.chunk())] = ln.template normalised<true>(raw[u]);
    {  // x as it is into position-major order: a thread holds one chunk of two positions
      u32x4_t lo, hi;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        lo[q] = __builtin_amdgcn_perm(xraw[2 * q + 1], xraw[2 * q], 0x05040100u);
        hi[q] = __builtin_amdgcn_perm(xraw[2 * q + 1], xraw[2 * q], 0x07060302u);
      }
      xn.s[Tile::slot(2 * xp, xc)] = lo;
      xn.s[Tile::slot(2 * xp + 1, xc)] = hi;
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < TASKS; ++u) {  // LayerNorm in place
      u32x4_t& x = xn.s[Tile::slot((wave + NW * u) * ln.PPI + ln.pos(), ln.chunk())];
      x = lx.template normalised<false>(x);
    }
    load_tile(id + (int)gridDim.x < total ? id + gridDim.x : id);
    __syncthreads();  // both tiles are complete; the ones before may be overwritten after this
    const Lane at = lane_here();
    const int l32 = at.l32, lh = at.lh;
    f32x16_t ag = zero16(), az = zero16();
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const int slot = Tile::slot(l32, 2 * s + lh);
      az = mfma_32x32x16(wz[s], xn.s[slot], az);
      ag = mfma_32x32x16(wg[s], zn.s[slot], ag);
    }
    // lane (position l32, half lh): channels 32 wave + 16 lh + v
    if (t.j0 + l32 < N) {
      const int64_t off = t.b * p.z_view.stride_b + t.i * p.z_view.stride_r + (t.j0 + l32) * p.z_view.stride_k + 32 * wave + 16 * lh;
      float res[16];
#pragma unroll
      for (int e = 0; e < 16; ++e) res[e] = az[e] * sigmoid_from_scaled(ag[e]);
      if (p.add_residual) add16(p.z + off, res);
      store16(p.out + off, res);
    }
  }
}

// ---- triangle attention, input pass (triattn_proj.hip) -------------------------------------------------------
// Wave = one 32-channel tile of q, k or v (kind 0, 1, 2), the last wave the triangle bias (4 rows, the others of its tile
// zero).
template <int C, int D>
__global__ __launch_bounds__(6 * C + 64) void triattn_proj_panels(TriattnProjArgs p, int panels, int total) {
  typedef PanelTile<C, true> Tile;
  constexpr int H = 4, OT = C / 32, KS = C / 16, NTASK = 32 / LnLane<C>::PPI;
  static_assert(H * D == C && NTASK <= 3 * OT, "");
  __shared__ u32x4_t tiles[2][Tile::SLOTS];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int kind = wave / OT, ot = wave % OT, N = p.N;
  const LnLane<C> ln = ln_lane<C>(p.ln_w, p.ln_b, lane);
  u32x4_t w[KS];
  load_attention_unit<C>(p, kind, ot, lane, w);

  u32x4_t raw;
  float mraw = 1.f;
  auto load_tile = [&](int pn) {
    const int ln_chunk = ln.chunk(), ln_pos = ln.pos();
    const int bi = pn / panels, b = bi / N, i = bi - b * N;
    int j = 32 * (pn - bi * panels) + wave * ln.PPI + ln_pos;
    j = j < N ? j : N - 1;
    if (wave < NTASK) {
      raw = *reinterpret_cast<const u32x4_t*>(p.x + b * p.x_view.stride_b + i * p.x_view.stride_r + j * p.x_view.stride_k + 8 * ln_chunk);
      if (p.mask) mraw = p.mask[b * p.mask_view.stride_b + i * p.mask_view.stride_r + j * p.mask_view.stride_k];
    }
  };
  int pn = grid_slot(), buf = 0;
  if (pn < total) load_tile(pn);
  for (; pn < total; pn += gridDim.x, buf ^= 1) {
    const Tile tile = {tiles[buf]};
    const int bi = pn / panels, j0 = 32 * (pn - bi * panels);
    if (wave < NTASK) {
      const int ln_chunk = ln.chunk(), pos = wave * ln.PPI + ln.pos();
      tile.s[Tile::slot(pos, ln_chunk)] = ln.template normalised<false>(raw);
      if (ln_chunk == 0) store_mask_bias(p, bi, j0 + pos, mraw);
    }
    load_tile(pn + (int)gridDim.x < total ? pn + gridDim.x : pn);
    __syncthreads();  // the tile is complete, everybody has finished with the other one
    project_panel<C, D>(p, w, tile, kind, ot, bi, j0);
  }
}

// ---- triangle attention, output pass (triattn_out.hip) -------------------------------------------------------
template <int C>
__global__ __launch_bounds__(2 * C, 4) void triattn_out_panels(TriattnOutArgs p, int panels, int total) {
  typedef PanelTile<C, false> Tile;
  constexpr int NW = C / 32, KS = C / 16, TASKS = 32 / LnLane<C>::PPI / NW;
  __shared__ u32x4_t xtile[Tile::SLOTS], otile[Tile::SLOTS];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int N = p.N;
  const LnLane<C> ln = ln_lane<C>(p.ln_w, p.ln_b, lane);
  u32x4_t wg[KS], wo[KS];
  load_unit<C>(p.w_g, wave, rowperm16(lane & 31), lane >> 5, p.packed, wg);
  load_unit<C>(p.w_o, wave, rowperm16(lane & 31), lane >> 5, p.packed, wo);
  auto place = [&](int id, int& b, int& i) {
    const int bi = id / panels;
    b = bi / N;
    i = bi - b * N;
    return 32 * (id - bi * panels);
  };
  u32x4_t raw[TASKS], oraw[2];
  auto load_tile = [&](int id) {
    const int ln_chunk = ln.chunk(), ln_pos = ln.pos();
    const Lane here = lane_here();
    const int l32 = here.l32, lh = here.lh;
    int b, i;
    const int j0 = place(id, b, i);
    const bf16_t* base = p.x + b * p.x_view.stride_b + i * p.x_view.stride_r + 8 * ln_chunk;
#pragma unroll
    for (int u = 0; u < TASKS; ++u) {
      int j = j0 + (wave + NW * u) * ln.PPI + ln_pos;
      j = j < N ? j : N - 1;
      raw[u] = *reinterpret_cast<const u32x4_t*>(base + j * p.x_view.stride_k);
    }
    const int j = j0 + l32 < N ? j0 + l32 : N - 1;
    const bf16_t* op = p.o + (((size_t)b * N + i) * N + j) * C + 32 * wave + 16 * lh;
    oraw[0] = *reinterpret_cast<const u32x4_t*>(op);
    oraw[1] = *reinterpret_cast<const u32x4_t*>(op + 8);
  };
  int id = grid_slot();
  if (id < total) load_tile(id);
  for (; id < total; id += gridDim.x) {
    int b, i;
    const int j0 = place(id, b, i);
#pragma unroll
    for (int u = 0; u < TASKS; ++u) xtile[Tile::slot((wave + NW * u) * ln.PPI + ln.pos(), ln.chunk())] = ln.template normalised<true>(raw[u]);
    __syncthreads();  // LayerNorm(x) is complete; everybody has finished with the gated output before
    {
      const Lane at = lane_here();
      const int l32 = at.l32, lh = at.lh;
      f32x16_t acc = zero16();
#pragma unroll
      for (int s = 0; s < KS; ++s) acc = mfma_32x32x16(wg[s], xtile[Tile::slot(l32, 2 * s + lh)], acc);
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        float ov[8];
        unpack8(oraw[half], ov);
#pragma unroll
        for (int v = 0; v < 8; ++v) ov[v] *= sigmoid_from_scaled(acc[8 * half + v]);
        otile[Tile::slot(l32, 4 * wave + 2 * lh + half)] = pack8(ov);
      }
    }
    load_tile(id + (int)gridDim.x < total ? id + gridDim.x : id);
    __syncthreads();  // the gated output is complete; everybody has read LayerNorm(x)
    const Lane at = lane_here();
    const int l32 = at.l32, lh = at.lh;
    f32x16_t acc = zero16();
#pragma unroll
    for (int s = 0; s < KS; ++s) acc = mfma_32x32x16(wo[s], otile[Tile::slot(l32, 2 * s + lh)], acc);
    if (j0 + l32 < N) {
      const int64_t off = b * p.x_view.stride_b + i * p.x_view.stride_r + (j0 + l32) * p.x_view.stride_k + 32 * wave + 16 * lh;
      float res[16];
#pragma unroll
      for (int v = 0; v < 16; ++v) res[v] = acc[v];
      if (p.add_residual) add16(p.x + off, res);
      store16(p.out + off, res);
    }
  }
}

template <auto Kern>
hipError_t panel_grid(int threads, long tiles, unsigned* grid) {
  static int cache[kMaxDevices];
  int fit = 0;
  hipError_t e = per_device(cache, [&](int dev, int* v) { return resident_blocks(Kern, threads, dev, v); }, &fit);
  *grid = (unsigned)(tiles < fit ? tiles : fit);
  return e;
}

template <int C>
hipError_t launch_trimul_proj(const TrimulProjArgs& a, hipStream_t stream) {
  const int panels = (a.N + 31) / 32, row_groups = (a.N + 3) / 4;
  const long total = (long)a.B * row_groups * panels * 4;
  unsigned grid = 0;
  hipError_t e = panel_grid<trimul_proj_panels<C>>(4 * C, total, &grid);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(trimul_proj_panels<C>, dim3(grid), dim3(4 * C), 0, stream, a, panels, row_groups, (int)total);
  return hipGetLastError();
}
template <int C>
hipError_t launch_trimul_out(const TrimulOutArgs& a, hipStream_t stream) {
  const int panels = (a.N + 31) / 32;
  const long total = (long)a.B * a.N * panels;
  unsigned grid = 0;
  hipError_t e = panel_grid<trimul_out_panels<C>>(2 * C, total, &grid);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(trimul_out_panels<C>, dim3(grid), dim3(2 * C), 0, stream, a, panels, (int)total);
  return hipGetLastError();
}
template <int C, int D>
hipError_t launch_triattn_proj(const TriattnProjArgs& a, hipStream_t stream) {
  const int panels = (a.N + 31) / 32;
  const long total = (long)a.B * a.N * panels;
  unsigned grid = 0;
  hipError_t e = panel_grid<triattn_proj_panels<C, D>>(6 * C + 64, total, &grid);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((triattn_proj_panels<C, D>), dim3(grid), dim3(6 * C + 64), 0, stream, a, panels, (int)total);
  return hipGetLastError();
}
template <int C>
hipError_t launch_triattn_out(const TriattnOutArgs& a, hipStream_t stream) {
  const int panels = (a.N + 31) / 32;
  const long total = (long)a.B * a.N * panels;
  unsigned grid = 0;
  hipError_t e = panel_grid<triattn_out_panels<C>>(2 * C, total, &grid);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(triattn_out_panels<C>, dim3(grid), dim3(2 * C), 0, stream, a, panels, (int)total);
  return hipGetLastError();
}

}  // namespace

hipError_t trimul_proj_panels_launch(const TrimulProjArgs& a, int C, hipStream_t stream) {
  return C == 128 ? launch_trimul_proj<128>(a, stream) : launch_trimul_proj<64>(a, stream);
}
hipError_t trimul_out_panels_launch(const TrimulOutArgs& a, int C, hipStream_t stream) {
  return C == 128 ? launch_trimul_out<128>(a, stream) : launch_trimul_out<64>(a, stream);
}
hipError_t triattn_proj_panels_launch(const TriattnProjArgs& a, int C, hipStream_t stream) {
  return C == 128 ? launch_triattn_proj<128, 32>(a, stream) : launch_triattn_proj<64, 16>(a, stream);
}
hipError_t triattn_out_panels_launch(const TriattnOutArgs& a, int C, hipStream_t stream) {
  return C == 128 ? launch_triattn_out<128>(a, stream) : launch_triattn_out<64>(a, stream);
}

}  // namespace of3
