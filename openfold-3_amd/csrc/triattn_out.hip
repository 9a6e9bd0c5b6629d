// Triangle-attention output pass (attention.py:288-302 plus the caller's residual add of
// base_blocks.py:364-378 when requested):
//     out = [x +] (o * sigmoid(LayerNorm(x) Wg^T)) Wo^T
// o is the flash kernel's [b][i][j][H*D] output in the module frame; x / out are addressed
// through the PairView (transposed for the ending node).  The gate is recomputed from x
// rather than stored by the input pass (one z-sized write and read less).
//
// Reads o and x once, writes out once: at N = 768 (128 channels) 4.3 to 4.8 TB/s, a large copy's rate, with the vector pipe 56 % busy; up
// to three rounds of tiles bound by a tile's chain of LayerNorm, products and barriers.  Two MFMA passes per tile of 128 or 64 positions:
// gate tile -> multiplied into the o tile in LDS in place -> output projection.
// A tile is consecutive positions of the flattened [B][N][N] index space of the module frame, so it
// may run over the end of a row (or of a batch element): a token count off the multiples of 128 costs
// no partly filled tile per row, only one at the very end.
#include "of3_device.h"
#include "of3_kernels.h"
#include "of3_launch.h"
#include "of3_pass_bf16.h"

#include <type_traits>

namespace of3 {

namespace {

// TP: positions of a tile (out_tile_positions in of3_tiles.h); PART: of the pieces that the tiles of the last round are dealt in (last_round), TP:
// whole tiles only
template <int C, int HD, int MODE, int PART, int TP>
__global__ __launch_bounds__(4 * TP, C == 64 ? 4 : 2) void triattn_out_kernel(TriattnOutArgs p, uint32_t total_pos, int whole_tiles, int total_items) {
  static_assert(C == HD, "o tile shares the x tile geometry");
  // Unconditional loads and stores and rows that leave whole, as in trimul_out.hip, in launches without pieces.  Past the end, which only the last
  // tile of all has, the last position is loaded and stored again.  us a launch, before / now, 64 channels: three templates of 256 19.3 / 18.1, of 400
  // 39.0 / 37.0, of 500 56.9 / 53.1, four of 384 45.7 / 41.5, of 512 78.7 / 70.8.  128 channels, tiles of 64 inside one row: N = 384 30.9 / 30.3, 512
  // 53.3 / 50.8, 768 105.7 / 101.2; where a tile may lie in two rows level (451 42.5 / 43.2, 1100 208 / 208), and on tiles of 128 1700 491 / 496.
  constexpr bool ROWS = PART == TP && (C == 64 ? MODE < 2 : MODE == 0 && TP == 64);
  constexpr int NCH = C / 8;
  constexpr int LPP = NCH;
  constexpr int PPI = 64 / LPP;
  constexpr int NW = TP / 16;            // waves per work-group
  constexpr int LN_ITERS = (TP / NW) / PPI;
  constexpr int KS = C / 16;
  constexpr int NOT = C / 32;
  constexpr int WPG = NW / NOT;
  constexpr int LN_STEP = NW * PPI;      // positions that the waves normalise at a time, PPI consecutive ones each

  __shared__ u32x4_t xtile[TP * NCH];  // LayerNorm(x), bf16
  __shared__ u32x4_t otile[TP * NCH];  // o, then o * gate
  __shared__ u32x4_t rtile[TP * NCH];  // x as loaded: the residual of the output phase

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, l32 = lane & 31, lh = lane >> 5;
  const int ln_chunk = lane % LPP, ln_pp = lane / LPP;

  // LayerNorm(x) feeds the gate only: its weight and bias carry the factor -log2(e) of the gate's
  // base-2 exponential, one multiplication per gate value less
  float lw[8], lb[8];
  load_affine8(p.ln_w, ln_chunk, lw);
  load_affine8(p.ln_b, ln_chunk, lb);
#pragma unroll
  for (int e = 0; e < 8; ++e) lw[e] *= -kLog2e, lb[e] *= -kLog2e;

  const int ot = wave % NOT;
  u32x4_t wg[KS], wo[KS];
  {
    pass_bf16::load_unit<C>(p.w_g, ot, rowperm16(l32), lh, p.packed, wg);
    pass_bf16::load_unit<HD>(p.w_o, ot, rowperm16(l32), lh, p.packed, wo);
  }

  const int N = p.N;
  // A tile starts at position p0 = (b0, i0, j0) (wave-uniform: scalar divisions); with N >= TP it holds
  // positions of at most two rows, whose offsets in the view are scalars, and position d of the tile costs a
  // compare and two selects (of3_tiles.h).
  typedef FlatTile Origin;
  auto tile_origin = [&](int tile_id) { return flat_tile<TP>(tile_id, N, p.x_view.stride_b, p.x_view.stride_r); };
  auto view_offset = [&](const Origin& t, int d) -> int64_t {
    return flat_offset<MODE>(t, d, N, p.x_view.stride_b, p.x_view.stride_r, p.x_view.stride_k);
  };

  // The loads of a tile are issued one tile ahead (right after the previous tile's values have
  // been consumed by the LayerNorm phase) and travel under that tile's two MFMA phases.
  // LayerNorm-phase position `it` of this lane, from the item's first one: TP / NW consecutive positions per wave in whole
  // tiles, in pieces LN_STEP by all waves at a time, so that a piece is the first iterations
  auto ln_position = [&](bool in_piece, int it) {
    return in_piece ? it * LN_STEP + wave * PPI + ln_pp : wave * (TP / NW) + it * PPI + ln_pp;
  };
  u32x4_t xraw[LN_ITERS], oraw[LN_ITERS];
  auto load_tile = [&](int item) {
    const TilePiece piece = tile_piece<PART, TP>(item, whole_tiles);
    const Origin t = tile_origin(piece.tile);
    const uint32_t p0 = (uint32_t)piece.tile * TP;
#pragma unroll
    for (int it = 0; it < LN_ITERS; ++it) {
      int d = piece.first + ln_position(piece.count < TP, it);
      if (ROWS) {
        if (MODE != 0) d = p0 + d < total_pos ? d : (int)(total_pos - 1 - p0);
        xraw[it] = *reinterpret_cast<const u32x4_t*>(p.x + view_offset(t, d) + 8 * ln_chunk);
        oraw[it] = *reinterpret_cast<const u32x4_t*>(p.o + (size_t)(p0 + d) * HD + 8 * ln_chunk);
        continue;
      }
      u32x4_t vx = {0u, 0u, 0u, 0u}, vo = {0u, 0u, 0u, 0u};
      if ((PART == TP || it * LN_STEP < piece.count) && p0 + d < total_pos) {
        vx = *reinterpret_cast<const u32x4_t*>(p.x + view_offset(t, d) + 8 * ln_chunk);
        vo = *reinterpret_cast<const u32x4_t*>(p.o + (size_t)(p0 + d) * HD + 8 * ln_chunk);  // o is [B][N][N][HD]
      }
      xraw[it] = vx;
      oraw[it] = vo;
    }
  };
  if constexpr (C == 64 && !ROWS) {
    // no early return here: with one, launches with pieces take longer, us: one tensor of 300 12.8 / 12.1, two of 200 12.4 / 11.7, three of 170 12.8 / 12.2, four
    // of 150 12.5 / 12.0 (128 channels: 200 11.9 / 12.1, 300 level)
    if ((int)blockIdx.x < total_items) load_tile(blockIdx.x);
  } else {
    if ((int)blockIdx.x >= total_items) return;
    load_tile(blockIdx.x);
  }
  if (ROWS) {  // the weights count as used here
#pragma unroll
    for (int s = 0; s < KS; ++s) __asm__ volatile("" : "+v"(wg[s]), "+v"(wo[s]));
  }

  auto do_tile = [&](auto positions, int item) {
    constexpr int P = decltype(positions)::value;
    constexpr int T = P / 32 >= WPG ? P / 32 / WPG : 1;  // position tiles per wave
    const TilePiece piece = tile_piece<PART, TP>(item, whole_tiles);
    const int first = P == TP ? 0 : piece.first;
    const bool multiplies = P == TP || wave / NOT * T < P / 32;
    const Origin t = tile_origin(piece.tile);
    const uint32_t p0 = (uint32_t)piece.tile * TP;

    // ---- LayerNorm of this tile's values, then the next tile's loads
#pragma unroll
    for (int it = 0; it < LN_ITERS; ++it) {
      const int pos = first + ln_position(P < TP, it);
      if (P < TP && pos >= first + P) break;
      const int slot = tile_slot<NCH, 0>(pos, ln_chunk);
      xtile[slot] = layer_norm_chunk<C>(xraw[it], lw, lb);
      rtile[slot] = xraw[it];
      otile[slot] = oraw[it];
    }
    __syncthreads();
    if (P == TP && item + (int)gridDim.x < total_items) load_tile(item + gridDim.x);

    // ---- gate: lane owns gate channels 32*ot + 16*lh + v of position 32*t + l32
#pragma unroll
    for (int tt = 0; tt < T; ++tt) {
      if (!multiplies) break;
      const int pos = first + 32 * (wave / NOT * T + tt) + l32;
      f32x16_t acc = zero16();
#pragma unroll
      for (int s = 0; s < KS; ++s) acc = mfma_32x32x16(wg[s], xtile[tile_slot<NCH, 0>(pos, 2 * s + lh)], acc);
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        const int slot = tile_slot<NCH, 0>(pos, 4 * ot + 2 * lh + half);
        float ov[8];
        unpack8(otile[slot], ov);
#pragma unroll
        for (int v = 0; v < 8; ++v) ov[v] *= sigmoid_from_scaled(acc[8 * half + v]);
        otile[slot] = pack8(ov);
      }
    }
    __syncthreads();

    // ---- output projection (+ residual)
    if (!multiplies) return;  // nothing comes after a piece
#pragma unroll
    for (int tt = 0; tt < T; ++tt) {
      const int pos = first + 32 * (wave / NOT * T + tt) + l32;
      f32x16_t acc = zero16();
#pragma unroll
      for (int s = 0; s < KS; ++s) acc = mfma_32x32x16(wo[s], otile[tile_slot<NCH, 0>(pos, 2 * s + lh)], acc);
      if (ROWS || p0 + pos < total_pos) {
        bf16_t* outrow = p.out;
        const int64_t off = ROWS ? 0 : view_offset(t, pos) + 32 * ot + 16 * lh;
        float res[16];
#pragma unroll
        for (int v = 0; v < 16; ++v) res[v] = acc[v];
        if (p.add_residual) {
          const u32x4_t r0 = rtile[tile_slot<NCH, 0>(pos, 4 * ot + 2 * lh)];
          const u32x4_t r1 = rtile[tile_slot<NCH, 0>(pos, 4 * ot + 2 * lh + 1)];
          float xr[8];
          unpack8(r0, xr);
#pragma unroll
          for (int v = 0; v < 8; ++v) res[v] += xr[v];
          unpack8(r1, xr);
#pragma unroll
          for (int v = 0; v < 8; ++v) res[8 + v] += xr[v];
        }
        u32x4_t o0, o1;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          o0[q] = pack_bf16(res[2 * q], res[2 * q + 1]);
          o1[q] = pack_bf16(res[8 + 2 * q], res[8 + 2 * q + 1]);
        }
        if (ROWS) {
          rtile[tile_slot<NCH, 0>(pos, 4 * ot + 2 * lh)] = o0;
          rtile[tile_slot<NCH, 0>(pos, 4 * ot + 2 * lh + 1)] = o1;
        } else {
          *reinterpret_cast<u32x4_t*>(outrow + off) = o0;
          *reinterpret_cast<u32x4_t*>(outrow + off + 8) = o1;
        }
      }
    }
    if (P == TP) __syncthreads();
    if (ROWS) {
#pragma unroll
      for (int it = 0; it < LN_ITERS; ++it) {
        int d = ln_position(false, it);
        if (MODE != 0) d = p0 + d < total_pos ? d : (int)(total_pos - 1 - p0);
        *reinterpret_cast<u32x4_t*>(p.out + view_offset(t, d) + 8 * ln_chunk) = rtile[tile_slot<NCH, 0>(d, ln_chunk)];
      }
    }
  };
  typedef std::integral_constant<int, TP> Whole;
  int item = blockIdx.x;
  if constexpr (ROWS) {
    do_tile(Whole{}, item);  // peeled: the loop proper is only entered with a tile's stores in flight
    item += gridDim.x;
  }
  for (; item < whole_tiles; item += gridDim.x) do_tile(Whole{}, item);
  if constexpr (PART < TP) {
    if (item < total_items) do_tile(std::integral_constant<int, PART>{}, item);  // one piece: the last round
  }
}

template <int C, int HD, int MODE, int TP>
hipError_t launch(const TriattnOutArgs& a, hipStream_t stream) {
  static int cache[kMaxDevices];
  int grid_cap = 0;
  hipError_t e =
      per_device(cache, [&](int dev, int* v) { return resident_blocks(triattn_out_kernel<C, HD, MODE, TP, TP>, 4 * TP, dev, v); }, &grid_cap);
  if (e != hipSuccess) return e;
  const long positions = (long)a.B * a.N * a.N;
  if (positions <= 0 || positions > 0x7fffffffL) return hipErrorInvalidValue;
  const int tiles = (int)((positions + TP - 1) / TP);
  constexpr bool kManyRounds = C == 128 && TP == 128;
  const LastRound r = kManyRounds ? LastRound{tiles, tiles, TP} : last_round<TP>(tiles, grid_cap);
  const int grid = r.items < grid_cap ? r.items : grid_cap;
  auto go = [&](auto kern) { hipLaunchKernelGGL(kern, dim3(grid), dim3(4 * TP), 0, stream, a, (uint32_t)positions, r.whole, r.items); };
  if constexpr (!kManyRounds) {
    if (r.piece == 32) {
      go(triattn_out_kernel<C, HD, MODE, 32, TP>);
      return hipGetLastError();
    }
    if (r.piece != TP) {
      go(triattn_out_kernel<C, HD, MODE, 64, TP>);
      return hipGetLastError();
    }
  }
  go(triattn_out_kernel<C, HD, MODE, TP, TP>);
  return hipGetLastError();
}
// a tile lies in one row (N a multiple of its positions), in at most two (N no less), or anywhere
template <int C, int TP>
hipError_t launch_tiles(const TriattnOutArgs& a, hipStream_t stream) {
  if (a.N % TP == 0) return launch<C, C, 0, TP>(a, stream);
  if (a.N >= TP) return launch<C, C, 1, TP>(a, stream);
  if constexpr (C == 64 || TP == 64) return launch<C, C, 2, TP>(a, stream);
  return hipErrorInvalidValue;  // tiles of 128 at 128 channels are for long sequences only
}

}  // namespace

hipError_t triattn_out_launch(const TriattnOutArgs& args, int C, int HD, hipStream_t stream) {
  if ((C != 128 && C != 64) || HD != C) return hipErrorInvalidValue;
  // Short sequences on 32-position tiles, under the rule of the triangle multiplication's output pass (C = 128, packed, us,
  // 128- against 32-position tiles: N = 40 7.7 / 4.5, 64 7.6 / 4.6, 96 8.4 / 6.7, 128 7.6 / 7.2, 160 8.8 / 9.4).
  bool small = false;
  const hipError_t e = small_pass(args.B, args.N, C == 128 ? 2 : 1, &small);
  if (e != hipSuccess) return e;
  if (small) return triattn_out_panels_launch(args, C, stream);
  if (C == 64) return launch_tiles<64, 128>(args, stream);
  return out_tile_positions(args.N, false) == 64 ? launch_tiles<128, 64>(args, stream) : launch_tiles<128, 128>(args, stream);
}

}  // namespace of3
