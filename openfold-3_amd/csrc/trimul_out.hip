// Triangle-multiplication output pass
//     out = [z +] (LayerNorm_out(x) Wz^T) * sigmoid(LayerNorm_in(z) Wg^T)
// (triangular_multiplicative_update.py:498-501; the optional residual is the caller's
// "z = z + update" of base_blocks.py:329-335 fused in).  x arrives channel-major
// [b][c][i][j] from the contraction and is transposed to position-major on its way into
// LDS; the gate is recomputed from z instead of being stored by the input pass, which
// saves one full write and one full read of a z-sized tensor.
//
// Reads x and z once, writes out once.  Bound by its instructions beside the bytes: at N = 768 (128 channels) 4.1 TB/s, where a large copy has 4.8, with the
// vector pipe 64 % busy.
//
// Tiles are TP = 128 or 64 positions: the whole TP-wide pieces of every row first, then, when N is not a multiple
// of TP, the remaining columns in pieces of 2^s columns x TP / 2^s consecutive rows (2^s the smallest
// power of two >= 8 that covers them), so that the ragged end of the rows costs a few tiles per batch
// element rather than one more tile per row.
#include "of3_device.h"
#include "of3_kernels.h"
#include "of3_launch.h"
#include "of3_pass_bf16.h"

#include <type_traits>

namespace of3 {

namespace {

// TP: positions of a tile (out_tile_positions in of3_tiles.h); PART: of the pieces that the tiles of the last round are dealt in (last_round), TP:
// whole tiles only
template <int C, int CH, bool RAGGED, int PART, int TP>
__global__ __launch_bounds__(4 * TP, C == 64 && TP == 64 ? 3 : 2) void trimul_out_kernel(TrimulOutArgs p, int full_per_row, int tail_shift, int tiles_per_batch,
                                                           int whole_tiles, int total_items) {
  static_assert(C == CH, "position-major x tile shares the z tile geometry");
  // 64 channels, tiles of 64: every tile issues the same loads and stores (indices past the end are clamped, a store past the end is beyond its
  // buffer), so that the compiler's wait for a tile's values counts the stores of the tile before it and leaves them in flight; with a load or a store
  // under a condition it waits for all of them.  Rows leave whole: the waves put their channels in the residual's place and the lanes that loaded a
  // row store it, 1 KB of it per instruction in the place of 16 bytes of each of 64 pieces of rows.  us a launch, before / now: three templates of 400
  // 46.1 / 44.2, of 500 68.3 / 65.0, four of 384 53.5 / 51.2, of 512 88.5 / 81.8; up to three rounds level.  At 128 channels the counted waits
  // are within 2 % (N = 300 23.3 / 23.5, 768 117.5 / 118.3) and whole rows lose 4 % (768 122): two work-groups to a CU, all registers taken.
  constexpr bool ROWS = C == 64 && TP == 64;
  constexpr int NCH = C / 8;
  constexpr int LPP = NCH;
  constexpr int PPI = 64 / LPP;
  constexpr int WHOLE = TP == 128 ? 7 : 6;  // log2 of its width where it lies in one row
  constexpr int NW = TP / 16, NTH = 64 * NW;  // waves and threads per work-group
  constexpr int LN_ITERS = (TP / NW) / PPI;
  constexpr int KS = C / 16;
  constexpr int NOT = C / 32;            // output-channel tiles
  constexpr int WPG = NW / NOT;          // waves sharing one output tile (2 or 4)
  constexpr int LN_STEP = NW * PPI;      // positions that the waves normalise at a time, PPI consecutive ones each
  constexpr int XROUNDS = (CH / 2) * (TP / 8) / NTH;  // (channel pair, 8-position group) items per thread

  __shared__ u32x4_t ztile[TP * NCH];
  __shared__ u32x4_t xtile[TP * NCH];
  __shared__ u32x4_t rtile[TP * NCH];  // z as loaded: the residual of the output phase

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, l32 = lane & 31, lh = lane >> 5;
  const int ln_chunk = lane % LPP, ln_pp = lane / LPP;

  float iw[8], ib[8], ow[8], ob[8];
  load_affine8(p.ln_in_w, ln_chunk, iw);
  load_affine8(p.ln_in_b, ln_chunk, ib);
  load_affine8(p.ln_out_w, ln_chunk, ow);
  load_affine8(p.ln_out_b, ln_chunk, ob);
  // LayerNorm_in(z) feeds the gate only: its weight and bias carry the factor -log2(e) of the gate's
  // base-2 exponential, one multiplication per gate value less
#pragma unroll
  for (int e = 0; e < 8; ++e) iw[e] *= -kLog2e, ib[e] *= -kLog2e;

  // A operands: logical output channel of A-row r is 32*ot + rowperm16(r), so that a lane
  // ends up with the 16 consecutive channels 32*ot + 16*lh + v
  const int ot = wave % NOT;
  u32x4_t wz[KS], wgt[KS];
  {
    pass_bf16::load_unit<CH>(p.w_z, ot, rowperm16(l32), lh, p.packed, wz);
    pass_bf16::load_unit<C>(p.w_g, ot, rowperm16(l32), lh, p.packed, wgt);
  }

  const int N = p.N, Np = p.Np;
  // tile -> batch element, first row, first column, log2 of its width (all wave-uniform); the last ragged
  // piece may run past the last row: those positions are left out below
  auto tile_origin = [&](int tile_id, int& b, int& i0, int& j0, int& shift) {
    const TilePlace t = tile_place<RAGGED, TP>(tile_id, N, full_per_row, tail_shift, tiles_per_batch, false);
    b = t.b, i0 = t.i0, j0 = t.j0, shift = t.shift;
  };
  // LayerNorm-phase position `it` of this lane, from the item's first one: TP / NW consecutive positions per wave in whole
  // tiles, in pieces LN_STEP by all waves at a time, so that a piece is the first iterations
  auto ln_position = [&](bool in_piece, int it) {
    return in_piece ? it * LN_STEP + wave * PPI + ln_pp : wave * (TP / NW) + it * PPI + ln_pp;
  };
  uint32_t* xt32 = reinterpret_cast<uint32_t*>(xtile);

  // The loads of a tile (z row-wise for the gate, x channel-major) are issued one tile ahead,
  // right after the previous tile's values have gone into LDS, and travel under its MFMA phase.
  u32x4_t zraw[LN_ITERS];
  u32x4_t xa[XROUNDS], xb[XROUNDS];
  auto load_tile = [&](int item) {
    const TilePiece piece = tile_piece<PART, TP>(item, whole_tiles);
    int b, i0, j0, shift_rt;
    tile_origin(piece.tile, b, i0, j0, shift_rt);
    const int shift = RAGGED ? shift_rt : WHOLE;  // a constant without ragged pieces: di below folds to 0
    const int jmask = (1 << shift) - 1;
    const bf16_t* zrow = p.z + b * p.z_view.stride_b + i0 * p.z_view.stride_r;  // the tile's first row (scalar)
#pragma unroll
    for (int it = 0; it < LN_ITERS; ++it) {
      int in_item = ln_position(piece.count < TP, it);
      if (ROWS && PART < TP) in_item = in_item < piece.count ? in_item : piece.count - 1;
      const int pos = piece.first + in_item;
      int di = RAGGED ? pos >> shift : 0, j = j0 + (RAGGED ? pos & jmask : pos);  // di = 0 in the whole-row pieces
      if (ROWS) {
        if (RAGGED) di = i0 + di < N ? di : N - 1 - i0, j = j < N ? j : N - 1;
        zraw[it] = *reinterpret_cast<const u32x4_t*>(zrow + di * p.z_view.stride_r + j * p.z_view.stride_k + 8 * ln_chunk);
        continue;
      }
      u32x4_t v = {0u, 0u, 0u, 0u};
      if ((PART == TP || it * LN_STEP < piece.count) && (!RAGGED || i0 + di < N) && j < N) v = *reinterpret_cast<const u32x4_t*>(zrow + di * p.z_view.stride_r + j * p.z_view.stride_k + 8 * ln_chunk);
      zraw[it] = v;
    }
#pragma unroll
    for (int rr = 0; rr < XROUNDS; ++rr) {
      const int item = rr * NTH + tid;
      // channels 2cp, 2cp+1; positions 8pg..8pg+7: one row, as the width is >= 8
      int cp = item >> piece.group_bits;
      const int pg = (piece.first >> 3) + (item & ((1 << piece.group_bits) - 1));
      if (PART < TP && ROWS) cp = cp < CH / 2 ? cp : CH / 2 - 1;
      else if (PART < TP && cp >= CH / 2) break;
      int i = i0 + (RAGGED ? (8 * pg) >> shift : 0);
      const int j = j0 + (RAGGED ? (8 * pg) & jmask : 8 * pg);  // < Np: the planes are padded to whole 128-wide pieces
      if (RAGGED) i = i < Np ? i : Np - 1;    // rows of a last piece past the end of the plane: any row, never used
      const bf16_t* src = p.x + (((size_t)b * CH + 2 * cp) * Np + i) * Np + j;
      xa[rr] = *reinterpret_cast<const u32x4_t*>(src);
      xb[rr] = *reinterpret_cast<const u32x4_t*>(src + (size_t)Np * Np);
    }
  };
  if ((int)blockIdx.x >= total_items) return;
  load_tile(blockIdx.x);
  if (ROWS) {  // the weights count as used here: no wait for them, which would be one for the next tile's loads, inside the loop
#pragma unroll
    for (int s = 0; s < KS; ++s) __asm__ volatile("" : "+v"(wz[s]), "+v"(wgt[s]));
  }

  auto do_tile = [&](auto positions, int item) {
    constexpr int P = decltype(positions)::value;
    constexpr int GROUPS = P / 8, XR = (CH / 2) * GROUPS > NTH ? (CH / 2) * GROUPS / NTH : 1;
    constexpr int T = P / 32 >= WPG ? P / 32 / WPG : 1;  // position tiles per wave
    const TilePiece piece = tile_piece<PART, TP>(item, whole_tiles);
    const int first = P == TP ? 0 : piece.first;
    int b, i0, j0, shift_rt;
    tile_origin(piece.tile, b, i0, j0, shift_rt);
    const int shift = RAGGED ? shift_rt : WHOLE;
    const int jmask = (1 << shift) - 1;
    bf16_t* orow0 = p.out + b * p.z_view.stride_b + i0 * p.z_view.stride_r;  // the tile's first row (scalar)
    if (ROWS && P < TP) __syncthreads();  // a whole tile's rows have left before other lanes write their places

    // x: transpose into xtile[pos][c] with 4-byte (channel pair) writes
#pragma unroll
    for (int rr = 0; rr < XR; ++rr) {
      const int item = rr * NTH + tid;
      const int cp = item / GROUPS, pg = (first >> 3) + item % GROUPS;
      if ((CH / 2) * GROUPS < NTH && cp >= CH / 2) break;
      const int chunk = (2 * cp) >> 3, within = (2 * cp) & 7;  // `within` is even
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const uint32_t ua = xa[rr][e >> 1], ub = xb[rr][e >> 1];
        const uint32_t w = __builtin_amdgcn_perm(ub, ua, (e & 1) ? 0x07060302u : 0x05040100u);
        const int pos = 8 * pg + e;
        xt32[tile_slot<NCH, 0>(pos, chunk) * 4 + (within >> 1)] = w;
      }
    }
    // z: LayerNorm_in -> ztile
#pragma unroll
    for (int it = 0; it < LN_ITERS; ++it) {
      const int pos = first + ln_position(P < TP, it);
      if (P < TP && pos >= first + P) break;
      ztile[tile_slot<NCH, 0>(pos, ln_chunk)] = layer_norm_chunk<C>(zraw[it], iw, ib);
      rtile[tile_slot<NCH, 0>(pos, ln_chunk)] = zraw[it];
    }
    __syncthreads();
    if (P == TP && item + (int)gridDim.x < total_items) load_tile(item + gridDim.x);

    // x: LayerNorm_out in place (lane owns one 16-byte chunk of one position)
#pragma unroll
    for (int it = 0; it < LN_ITERS; ++it) {
      const int pos = first + ln_position(P < TP, it);
      if (P < TP && pos >= first + P) break;
      const int slot = tile_slot<NCH, 0>(pos, ln_chunk);
      xtile[slot] = layer_norm_chunk<CH>(xtile[slot], ow, ob);
    }
    __syncthreads();

    // ---- matrix phase
    if (P < TP && wave / NOT * T >= P / 32) return;  // nothing comes after a piece
#pragma unroll
    for (int tt = 0; tt < T; ++tt) {
      const int pos = first + 32 * (wave / NOT * T + tt) + l32;
      f32x16_t accu = zero16(), accg = zero16();
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const u32x4_t bx = xtile[tile_slot<NCH, 0>(pos, 2 * s + lh)];
        const u32x4_t bz = ztile[tile_slot<NCH, 0>(pos, 2 * s + lh)];
        accu = mfma_32x32x16(wz[s], bx, accu);
        accg = mfma_32x32x16(wgt[s], bz, accg);
      }
      const int di = RAGGED ? pos >> shift : 0, j = j0 + (RAGGED ? pos & jmask : pos);
      if ((ROWS && P == TP) || ((!RAGGED || i0 + di < N) && j < N)) {
        bf16_t* orow = orow0;
        const int64_t off = di * p.z_view.stride_r + j * p.z_view.stride_k + 32 * ot + 16 * lh;
        float res[16];
#pragma unroll
        for (int v = 0; v < 16; ++v) res[v] = accu[v] * sigmoid_from_scaled(accg[v]);
        if (p.add_residual) {
          const u32x4_t r0 = rtile[tile_slot<NCH, 0>(pos, 4 * ot + 2 * lh)];
          const u32x4_t r1 = rtile[tile_slot<NCH, 0>(pos, 4 * ot + 2 * lh + 1)];
          float zr[8];
          unpack8(r0, zr);
#pragma unroll
          for (int v = 0; v < 8; ++v) res[v] += zr[v];
          unpack8(r1, zr);
#pragma unroll
          for (int v = 0; v < 8; ++v) res[8 + v] += zr[v];
        }
        u32x4_t o0, o1;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          o0[q] = pack_bf16(res[2 * q], res[2 * q + 1]);
          o1[q] = pack_bf16(res[8 + 2 * q], res[8 + 2 * q + 1]);
        }
        if (ROWS && P == TP) {
          rtile[tile_slot<NCH, 0>(pos, 4 * ot + 2 * lh)] = o0;
          rtile[tile_slot<NCH, 0>(pos, 4 * ot + 2 * lh + 1)] = o1;
        } else {
          *reinterpret_cast<u32x4_t*>(orow + off) = o0;
          *reinterpret_cast<u32x4_t*>(orow + off + 8) = o1;
        }
      }
    }
    if (P == TP) __syncthreads();  // both tiles are rewritten by the next iteration
    if (ROWS && P == TP) {
      const __amdgpu_buffer_rsrc_t rows = buffer_rsrc(orow0 + j0 * p.z_view.stride_k, 0x7fffffffu);
      const int sr = (int)p.z_view.stride_r, sk = (int)p.z_view.stride_k;  // a tile's offsets fit 31 bits (trimul_out_launch)
#pragma unroll
      for (int it = 0; it < LN_ITERS; ++it) {
        const int pos = ln_position(false, it), di = RAGGED ? pos >> shift : 0, dj = RAGGED ? pos & jmask : pos;
        const bool there = !RAGGED || (i0 + di < N && j0 + dj < N);
        const uint32_t off = there ? (uint32_t)(di * sr + dj * sk + 8 * ln_chunk) * 2u : 0x80000000u;
        __builtin_amdgcn_raw_buffer_store_b128(rtile[tile_slot<NCH, 0>(pos, ln_chunk)], rows, off, 0, 0);
      }
    }
  };
  typedef std::integral_constant<int, TP> Whole;
  int item = blockIdx.x;
  if constexpr (ROWS) {
    if (item < whole_tiles) {  // peeled: the loop proper is only entered with a tile's stores in flight
      do_tile(Whole{}, item);
      for (item += gridDim.x; item < whole_tiles; item += gridDim.x) do_tile(Whole{}, item);
    }
  } else {
    for (; item < whole_tiles; item += gridDim.x) do_tile(Whole{}, item);
  }
  if constexpr (PART < TP) {
    if (item < total_items) do_tile(std::integral_constant<int, PART>{}, item);  // one piece: the last round
  }
}

template <int C, int CH, bool RAGGED, int TP>
hipError_t launch(const TrimulOutArgs& a, hipStream_t stream) {
  static int cache[kMaxDevices];
  int grid_cap = 0;
  hipError_t e =
      per_device(cache, [&](int dev, int* v) { return resident_blocks(trimul_out_kernel<C, CH, RAGGED, TP, TP>, 4 * TP, dev, v); }, &grid_cap);
  if (e != hipSuccess) return e;
  const RaggedTiles t = ragged_tiles<TP>(a.N);
  const long total = (long)a.B * t.per_batch;
  if (total > 0x7fffffffL) return hipErrorInvalidValue;
  LastRound r = {(int)total, (int)total, TP};
  if (TP == 64) r = last_round<TP>(total, grid_cap);  // tiles of 128: dozens of rounds
  const int grid = r.items < grid_cap ? r.items : grid_cap;
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(grid), dim3(4 * TP), 0, stream, a, t.full_per_row, t.tail_shift, t.per_batch, r.whole, r.items);
  };
  if (r.piece == TP) go(trimul_out_kernel<C, CH, RAGGED, TP, TP>);
  else if constexpr (TP == 64) go(trimul_out_kernel<C, CH, RAGGED, 32, TP>);
  return hipGetLastError();
}
template <int C, int TP>
hipError_t launch_tiles(const TrimulOutArgs& a, hipStream_t stream) {
  return a.N % TP != 0 ? launch<C, C, true, TP>(a, stream) : launch<C, C, false, TP>(a, stream);
}

}  // namespace

hipError_t trimul_out_launch(const TrimulOutArgs& args, int C, int CH, hipStream_t stream) {
  if ((C != 128 && C != 64) || CH != C) return hipErrorInvalidValue;
  // Short sequences on 32-position tiles, up to two of them per CU (C = 128, us per pass with packed weights, 128- against
  // 32-position tiles: N = 40 8.3 / 5.4, 64 8.5 / 5.8, 96 9.0 / 7.6, 128 9.4 / 8.6, 160 9.9 / 10.4), one at 64 channels
  // (B = 2: N = 64 5.2 / 4.8, 80 5.4 / 5.9).
  bool small = false;
  const hipError_t e = small_pass(args.B, args.N, C == 128 ? 2 : 1, &small);
  if (e != hipSuccess) return e;
  if (small) return trimul_out_panels_launch(args, C, stream);
  // at 64 channels the stores of a tile of 64 have 32-bit offsets from its first position: 8 rows, 64 columns
  const bool fits = C != 64 || 8 * args.z_view.stride_r + 64 * args.z_view.stride_k + C < (1l << 30);
  const bool half = fits && out_tile_positions(args.N, true) == 64;
  if (C == 128) return half ? launch_tiles<128, 64>(args, stream) : launch_tiles<128, 128>(args, stream);
  return half ? launch_tiles<64, 64>(args, stream) : launch_tiles<64, 128>(args, stream);
}

}  // namespace of3
