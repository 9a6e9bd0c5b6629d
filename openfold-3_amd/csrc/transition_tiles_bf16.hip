// bf16 pair transition (transition.hip has the operation and its rounding points) on tiles of 32, 64, 128 or 160
// positions, for short sequences.
//
// transition.hip gives a wave 32 positions and the whole hidden dimension: 256 positions per work-group and about 24 us
// for one of them, whether a call has seven of them (40 tokens) or one for every CU.  Here the eight waves of a
// work-group share a tile's hidden dimension, a wave to each tile of 32 hidden channels of a slice of 32 S; the hidden
// activations go through LDS (double buffered, one barrier per slice), and a wave owns one 32-channel tile of the
// output.  The sums run over the hidden channels in the same order and groups as there: the results are the same bits.
// The weights come from L2 for every tile (384 KB at C = 128, n = 4, as long as its products on 64 positions), requested
// one slice ahead.
// The longer tiles are for the lengths at which one of them per CU is all there is to do: 24 us for 128 positions, 28 for
// 160 (their hidden slices are of 128 channels, two or three position tiles to a wave; LDS has no room for more).
#include "of3_device.h"
#include "of3_kernels.h"
#include "of3_launch.h"
#include "of3_pass_bf16.h"

namespace of3 {

namespace {

using namespace pass_bf16;

constexpr int kWaves = 8;

// S hidden tiles per slice, P tiles of 32 positions per work-group (P = 5, S = 4, C = 128: all of the 160 KB)
template <int C, int S, int P>
constexpr size_t lds_slots() {
  return (size_t)P * (2 * PanelTile<C, false>::SLOTS + 2 * 32 * 4 * S);
}

// BIAS: and ends with the pair bias of the block's attention over s (pair_bias.hip), from the rows that it has just finished; the positions
// of a tile are as contiguous there as in z.  Four trunk blocks at N = 40 / 85 / 128 / 151 / 200 364 / 397 / 476 / 610 / 865 us, so 347 / 375 / 457 /
// 592 / 847 (a launch, and z read once more from memory).
// AFTER: the tile begins with the output pass of the triangle attention before it (the ending node's: its frame is the transposed one),
// whose result goes from LDS to LDS; one tile per work-group, weights packed.  Saves a launch, the tile's trip to memory and back and the wait for the
// first tile: four trunk blocks at N = 40 / 85 / 128 / 150 / 200 353 / 410 / 491 / 617 / 881 us, so 324 / 395 / 477 / 603 / 855; templates 4 x 60 152 /
// 134, 2 x 90 166 / 160, 1 x 180 223 / 219.
template <int C, int S, int P, bool AFTER, bool BIAS>
__global__ __launch_bounds__(64 * kWaves) void transition_tiles(TransitionArgs p, int packed, int tiles_per_row, int total, TriattnOutArgs e,
                                                                Division by_n, PairBiasArgs pb) {
  typedef PanelTile<C, false> XTile;
  constexpr int KS = C / 16, OT = C / 32, HCH = 4 * S;  // 16-byte chunks of a position's hidden slice
  constexpr int TASKS = P * 32 / LnLane<C>::PPI;        // LayerNorm instructions of a tile
  constexpr int LPW = (TASKS + kWaves - 1) / kWaves;
  // first product: hidden tile of the wave and the position tiles it covers; second: output and position tile
  // (tiles pt_a, pt_a + GA ... and pt_b, pt_b + GB ...; the two waves of a SIMD differ in pt_a and pt_b)
  constexpr int GA = kWaves / S, GB = kWaves / OT, APT = (P + GA - 1) / GA, BPT = (P + GB - 1) / GB;
  static_assert(S == 8 || S == 4, "");
  // The next slice's first weights requested before the slice's barrier, where the registers are there (one tile per work-group): four trunk blocks
  // at N = 140 / 160 / 180 569 / 601 / 675 us, so 561 / 593 / 666; 128 and 200 451 and 801, 449 and 799; with one position tile no difference.
  constexpr bool EARLY = AFTER && P > 1;
  extern __shared__ u32x4_t lds[];
  u32x4_t* const xn = lds;                             // [P][XTile::SLOTS] LayerNorm(x)
  u32x4_t* const xr = xn + P * XTile::SLOTS;           // x as loaded: the residual
  u32x4_t* const hid = xr + P * XTile::SLOTS;          // [2][P][32 * HCH]
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int ht = wave % S, pt_a = wave / S;
  const int ot = wave % OT, pt_b = wave / OT;
  const bool first = pt_a < P, second = pt_b < P;  // wave-uniform
  const int L = p.N, slices = p.HID / (32 * S);
  const LnLane<C> ln = ln_lane<C>(p.ln_w, p.ln_b, lane);
  const int arow = rowperm16(lane & 31), half = lane >> 5;

  auto hid_slot = [](int pos, int chunk) { return pos * HCH + (chunk ^ (pos & 15)); };
  auto place = [&](int id, int& b, int& i) {
    const int per_b = p.R * tiles_per_row;
    b = id / per_b;
    const int rem = id - b * per_b;
    i = rem / tiles_per_row;
    return (rem - i * tiles_per_row) * 32 * P;
  };
  u32x4_t raw[LPW];
  float mval[BPT];
#pragma unroll
  for (int q = 0; q < BPT; ++q) mval[q] = 1.f;
  auto load_tile = [&](int id) {
    const int ln_chunk = ln.chunk(), ln_pos = ln.pos();
    int b, i;
    const int j0 = place(id, b, i);
    const bf16_t* row = p.x + b * p.x_view.stride_b + i * p.x_view.stride_r + 8 * ln_chunk;
#pragma unroll
    for (int u = 0; u < LPW; ++u) {
      const int task = wave + kWaves * u;
      int j = j0 + (task < TASKS ? task : 0) * ln.PPI + ln_pos;
      j = j < L ? j : L - 1;
      raw[u] = *reinterpret_cast<const u32x4_t*>(row + j * p.x_view.stride_k);
    }
    if (p.mask) {
#pragma unroll
      for (int q = 0; q < BPT; ++q) {
        int j = j0 + (second ? 32 * (pt_b + GB * q) : 0) + lane_here().l32;
        j = j < L ? j : L - 1;
        mval[q] = p.mask[b * p.mask_view.stride_b + i * p.mask_view.stride_r + j * p.mask_view.stride_k];
      }
    }
  };
  // operands of hidden tile t of Wa and Wb, and of the output tile's columns of a slice.  The second product's k-step s
  // of a hidden tile takes hidden channels 16 lh + 8 s + (0 .. 7) of it, the order in which a lane holds them.
  u32x4_t wa[KS], wb[KS], wo[2 * S];
  auto load_first = [&](int slice) {
    const int t = slice * S + ht;
    load_unit<C>(p.w_a, t, arow, half, packed, wa);
    load_unit<C>(p.w_b, t, arow, half, packed, wb);
  };
  auto load_second = [&](int slice) {
    const bf16_t* base = packed ? p.w_out + (((ot * (p.HID / 16) + half) * 64) + arow) * 8 : p.w_out + (32 * ot + arow) * p.HID + 16 * half;
    const int step_t = packed ? 1024 : 32, step_s = packed ? 256 : 8;
#pragma unroll
    for (int t = 0; t < S; ++t)
#pragma unroll
      for (int s = 0; s < 2; ++s) wo[2 * t + s] = *reinterpret_cast<const u32x4_t*>(base + (slice * S + t) * step_t + s * step_s);
  };

  int id = AFTER ? grid_slot() : blockIdx.x;
  if (id >= total) return;
  load_tile(id);
  if (!AFTER && first) load_first(0);
  for (; id < total; id += gridDim.x) {
    int b, i;
    const int j0 = place(id, b, i);
    auto ln_slot = [&](int u) {
      const int pos = (wave + kWaves * u) * ln.PPI + ln.pos();
      return (pos >> 5) * XTile::SLOTS + XTile::slot(pos & 31, ln.chunk());
    };
    if constexpr (AFTER) {
      // the same steps and rounding points as triattn_out.hip
      constexpr int MINE = (P + GB - 1) / GB;
      u32x4_t o[MINE][2], wg[KS], wz[KS];
      const LnLane<C> lz = ln_lane<C>(e.ln_w, e.ln_b, lane);
#pragma unroll
      for (int q = 0; q < MINE; ++q) {
        const int pos = j0 + 32 * (pt_b + GB * q) + (lane & 31), f = pos < L ? pos : L - 1;
        const int r = by_n.quotient(f), k = f - r * by_n.d;
        const bf16_t* src = e.o + (((int64_t)b * by_n.d + k) * by_n.d + r) * C + 32 * ot + 16 * half;
        o[q][0] = *reinterpret_cast<const u32x4_t*>(src);
        o[q][1] = *reinterpret_cast<const u32x4_t*>(src + 8);
      }
      if (second) {
        load_unit<C>(e.w_g, ot, arow, half, 1, wg);
        load_unit<C>(e.w_o, ot, arow, half, 1, wz);
      }
#pragma unroll
      for (int u = 0; u < LPW; ++u) {
        if (wave + kWaves * u >= TASKS) continue;
        const int slot = ln_slot(u);
        xn[slot] = lz.template normalised<true>(raw[u]);
        xr[slot] = raw[u];
      }
      __syncthreads();
      if (second) {
#pragma unroll
        for (int q = 0; q < MINE; ++q) {  // the attention's output times its gate
          const int pt = pt_b + GB * q;
          if (P % GB != 0 && pt >= P) break;
          const Lane at = lane_here();
          f32x16_t acc = zero16();
#pragma unroll
          for (int s = 0; s < KS; ++s) acc = mfma_32x32x16(wg[s], xn[pt * XTile::SLOTS + XTile::slot(at.l32, 2 * s + at.lh)], acc);
#pragma unroll
          for (int hf = 0; hf < 2; ++hf) {
            float ov[8];
            unpack8(o[q][hf], ov);
#pragma unroll
            for (int v = 0; v < 8; ++v) ov[v] *= sigmoid_from_scaled(acc[8 * hf + v]);
            hid[pt * XTile::SLOTS + XTile::slot(at.l32, 4 * ot + 2 * at.lh + hf)] = pack8(ov);
          }
        }
      }
      __syncthreads();
      if (first) load_first(0);
      if (second) {
#pragma unroll
        for (int q = 0; q < MINE; ++q) {
          const int pt = pt_b + GB * q;
          if (P % GB != 0 && pt >= P) break;
          const Lane at = lane_here();
          f32x16_t acc = zero16();
#pragma unroll
          for (int s = 0; s < KS; ++s) acc = mfma_32x32x16(wz[s], hid[pt * XTile::SLOTS + XTile::slot(at.l32, 2 * s + at.lh)], acc);
#pragma unroll
          for (int hf = 0; hf < 2; ++hf) {
            u32x4_t* const s = xr + pt * XTile::SLOTS + XTile::slot(at.l32, 4 * ot + 2 * at.lh + hf);
            float r[8];
            unpack8(*s, r);
#pragma unroll
            for (int v = 0; v < 8; ++v) r[v] = acc[8 * hf + v] + r[v];
            *s = pack8(r);
          }
        }
      }
      __syncthreads();
#pragma unroll
      for (int u = 0; u < LPW; ++u)
        if (wave + kWaves * u < TASKS) raw[u] = xr[ln_slot(u)];
    }
#pragma unroll
    for (int u = 0; u < LPW; ++u) {
      if (wave + kWaves * u >= TASKS) continue;
      const int slot = ln_slot(u);
      xn[slot] = ln.template normalised<false>(raw[u]);
      if (!AFTER) xr[slot] = raw[u];
    }
    float mtile[BPT];
    f32x16_t oacc[BPT];
#pragma unroll
    for (int q = 0; q < BPT; ++q) mtile[q] = mval[q], oacc[q] = zero16();
    __syncthreads();
    for (int slice = 0; slice < slices; ++slice) {
      u32x4_t* const h = hid + (slice & 1) * P * 32 * HCH;
      const Lane at = lane_here();
      const int l32 = at.l32, lh = at.lh;
      if (second) load_second(slice);
      if (first) {
#pragma unroll
        for (int q = 0; q < APT; ++q) {
          const int pt = pt_a + GA * q;
          if (P % GA != 0 && P > GA && pt >= P) break;  // wave-uniform
          const u32x4_t* x = xn + pt * XTile::SLOTS;
          f32x16_t ca = zero16(), cb = zero16();
#pragma unroll
          for (int s = 0; s < KS; ++s) {
            const u32x4_t xb = x[XTile::slot(l32, 2 * s + lh)];
            ca = mfma_32x32x16(wa[s], xb, ca);
            cb = mfma_32x32x16(wb[s], xb, cb);
          }
          float hv[16];
#pragma unroll
          for (int e = 0; e < 16; ++e) hv[e] = ca[e] * fast_rcp(1.f + fast_exp2(-kLog2e * ca[e])) * cb[e];
          u32x4_t* dst = h + pt * 32 * HCH;
#pragma unroll
          for (int s = 0; s < 2; ++s) {
            u32x4_t o;
#pragma unroll
            for (int v = 0; v < 4; ++v) o[v] = pack_bf16(hv[8 * s + 2 * v], hv[8 * s + 2 * v + 1]);
            dst[hid_slot(l32, 4 * ht + 2 * lh + s)] = o;
          }
        }
      }
      if (EARLY && first && slice + 1 < slices) load_first(slice + 1);
      __syncthreads();  // the slice is complete, and nobody reads the one before any more
      if (!EARLY && first) load_first(slice + 1 < slices ? slice + 1 : 0);
      if (!AFTER && slice + 1 == slices) load_tile(id + (int)gridDim.x < total ? id + gridDim.x : id);
      if (second) {
#pragma unroll
        for (int q = 0; q < BPT; ++q) {
          const int pt = pt_b + GB * q;
          if (P % GB != 0 && P > GB && pt >= P) break;  // wave-uniform
          const u32x4_t* src = h + pt * 32 * HCH;
#pragma unroll
          for (int t = 0; t < S; ++t)
#pragma unroll
            for (int s = 0; s < 2; ++s) oacc[q] = mfma_32x32x16(wo[2 * t + s], src[hid_slot(l32, 4 * t + 2 * lh + s)], oacc[q]);
        }
      }
    }
    if (second) {
#pragma unroll
      for (int q = 0; q < BPT; ++q) {
        const int pt = pt_b + GB * q;
        if (P % GB != 0 && P > GB && pt >= P) break;  // wave-uniform
        const Lane at = lane_here();
        const int l32 = at.l32, lh = at.lh, j = j0 + 32 * pt + l32;
        u32x4_t* const s0 = xr + pt * XTile::SLOTS + XTile::slot(l32, 4 * ot + 2 * lh);
        u32x4_t* const s1 = xr + pt * XTile::SLOTS + XTile::slot(l32, 4 * ot + 2 * lh + 1);
        float r0[8], r1[8];
        unpack8(*s0, r0);
        unpack8(*s1, r1);
        if (!p.add_residual) {
#pragma unroll
          for (int e = 0; e < 8; ++e) r0[e] = r1[e] = 0.f;
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          r0[e] += oacc[q][e] * mtile[q];
          r1[e] += oacc[q][8 + e] * mtile[q];
        }
        const u32x4_t o0 = pack8(r0), o1 = pack8(r1);
        if (BIAS) *s0 = o0, *s1 = o1;
        if (j < L) {
          bf16_t* dst = p.out + b * p.x_view.stride_b + i * p.x_view.stride_r + j * p.x_view.stride_k + 32 * ot + 16 * lh;
          *reinterpret_cast<u32x4_t*>(dst) = o0;
          *reinterpret_cast<u32x4_t*>(dst + 8) = o1;
        }
      }
    }
    if constexpr (BIAS) {
      LnLane<C> lb;
      const int chunk = lane % LnLane<C>::NCH;
      lb.w = *reinterpret_cast<const u32x4_t*>(pb.ln_w + 8 * chunk);
      lb.b = u32x4_t{0u, 0u, 0u, 0u};
      if (pb.ln_b) lb.b = *reinterpret_cast<const u32x4_t*>(pb.ln_b + 8 * chunk);
      u32x4_t wh[KS];
      const int head = lane & 31;
      if (wave < P) {
#pragma unroll
        for (int s = 0; s < KS; ++s) {
          wh[s] = u32x4_t{0u, 0u, 0u, 0u};
          if (head < pb.H) wh[s] = *reinterpret_cast<const u32x4_t*>(pb.w + head * C + 16 * s + 8 * half);
        }
      }
      __syncthreads();  // the tile's rows are complete
#pragma unroll
      for (int u = 0; u < LPW; ++u) {
        if (wave + kWaves * u >= TASKS) continue;
        const int slot = ln_slot(u);
        xn[slot] = lb.template normalised<false>(xr[slot]);
      }
      __syncthreads();
      if (wave < P) {
        f32x16_t acc = zero16();
#pragma unroll
        for (int s = 0; s < KS; ++s) acc = mfma_32x32x16(xn[wave * XTile::SLOTS + XTile::slot(arow, 2 * s + half)], wh[s], acc);
        // lane (head, half): 16 positions
        const int f = j0 + 32 * wave + 16 * half;
        if (head < pb.H && f < L) store_run16(pb.out + ((int64_t)b * pb.H + head) * L + f, acc, L - f, L % 8 == 0);
      }
    }
    if (AFTER) return;
    __syncthreads();  // both tiles of x are rewritten by the next one
  }
}

template <int C, int S, int P, bool AFTER = false, bool BIAS = false>
hipError_t launch(const TransitionArgs& a, hipStream_t stream, const TriattnOutArgs& end = {}, const PairBiasArgs& bias = {}) {
  constexpr size_t lds = lds_slots<C, S, P>() * 16;
  constexpr auto kernel = transition_tiles<C, S, P, AFTER, BIAS>;
  static int cache[kMaxDevices];
  int fit = 0;
  hipError_t e = allow_dynamic_lds<kernel>(lds);
  if (e == hipSuccess)
    e = per_device(
        cache,
        [&](int dev, int* v) {
          int cus = 0, per_cu = 0;
          hipError_t s = cu_count(dev, &cus);
          if (s == hipSuccess) s = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, 64 * kWaves, lds);
          *v = cus * (per_cu > 0 ? per_cu : 1);
          return s;
        },
        &fit);
  if (e != hipSuccess) return e;
  const int tiles_per_row = (a.N + 32 * P - 1) / (32 * P);
  const long total = (long)a.B * a.R * tiles_per_row;
  TransitionArgs k = a;
  const int packed = a.operands[0] ? 1 : 0;
  if (packed) k.w_a = a.operands[0], k.w_b = a.operands[1], k.w_out = a.operands[2];
  if (AFTER && (!packed || a.R != 1 || a.N != end.N * end.N || a.B != end.B)) return hipErrorInvalidValue;
  hipLaunchKernelGGL(kernel, dim3((unsigned)(AFTER || total < fit ? total : fit)), dim3(64 * kWaves), lds, stream, k, packed, tiles_per_row, (int)total,
                     end, Division::by(AFTER ? end.N : 1), bias);
  return hipGetLastError();
}

}  // namespace

template <int C, bool BIAS>
static hipError_t launch_after(const TriattnOutArgs& end, const TransitionArgs& a, const PairBiasArgs& bias, int position_tiles, hipStream_t stream) {
  const bool wide = a.HID % 256 == 0;
  if (position_tiles == 1)
    return wide ? launch<C, 8, 1, true, BIAS>(a, stream, end, bias) : launch<C, 4, 1, true, BIAS>(a, stream, end, bias);
  if (position_tiles == 2)
    return wide ? launch<C, 8, 2, true, BIAS>(a, stream, end, bias) : launch<C, 4, 2, true, BIAS>(a, stream, end, bias);
  if constexpr (C == 128) {
    if (position_tiles == 4) return launch<128, 4, 4, true, BIAS>(a, stream, end, bias);
    if (position_tiles == 5) return launch<128, 4, 5, true, BIAS>(a, stream, end, bias);
  }
  return hipErrorInvalidValue;
}
hipError_t triattn_transition_tiles_launch(const TriattnOutArgs& end, const TransitionArgs& a, const PairBiasArgs* bias, int C,
                                           int position_tiles, hipStream_t stream) {
  if (bias && (bias->B != a.B || bias->N * bias->N != a.N || bias->H > 32 || C != 128)) return hipErrorInvalidValue;
  if (C == 64) return launch_after<64, false>(end, a, {}, position_tiles, stream);
  return bias ? launch_after<128, true>(end, a, *bias, position_tiles, stream) : launch_after<128, false>(end, a, {}, position_tiles, stream);
}

hipError_t transition_tiles_launch(const TransitionArgs& a, int C, int position_tiles, hipStream_t stream) {
  if (position_tiles > 2) {
    if (C != 128) return hipErrorInvalidValue;
    return position_tiles == 4 ? launch<128, 4, 4>(a, stream) : launch<128, 4, 5>(a, stream);
  }
  const bool one = position_tiles == 1;
  if (a.HID % 256 == 0) {
    if (C == 128) return one ? launch<128, 8, 1>(a, stream) : launch<128, 8, 2>(a, stream);
    return one ? launch<64, 8, 1>(a, stream) : launch<64, 8, 2>(a, stream);
  }
  if (C == 128) return one ? launch<128, 4, 1>(a, stream) : launch<128, 4, 2>(a, stream);
  return one ? launch<64, 4, 1>(a, stream) : launch<64, 4, 2>(a, stream);
}

}  // namespace of3
