// Triangle-attention input pass: xn = LayerNorm(x), then
//     q = (xn Wq^T) * log2(e)/sqrt(D),  k = xn Wk^T,  v = xn Wv^T     (attention.py:265-286)
//     triangle bias tb[h][q][k] = log2(e) * (xn[q][k] . Wb[h])          (tri_att.py:137-140)
//     mask bias     mb[i][k]    = log2(e) * inf * (mask[i][k] - 1)      (tri_att.py:134)
// written in the layouts the flash kernel consumes: q, k as [b][i][h][j][d]; v transposed
// in panels of 32 keys as [b][i][h][j/32][d][j%32] (one key tile of one head = 2 KB
// contiguous); tb as [b][h][i][j] and mb as [b][i][j] in fp32.  log2(e) is folded
// in so the softmax can use the hardware base-2 exponential.  The PairView makes (i, j)
// walk either the tensor itself (starting node) or its transpose (ending node).
//
// Reads x once, writes q, k, v once; at N = 768 (128 channels) 4.7 to 5.4 TB/s, a large copy's rate.  Same structure as the
// triangle-multiplication input pass: 8 waves per work-group, weights resident in registers
// as MFMA A operands, 128-position tiles normalised in registers and staged once in a
// double-buffered LDS tile (one barrier per tile).
//
// Tiles: the whole 128-wide pieces of every row; when N is not a multiple of 128 (RAGGED), the remaining
// columns come in pieces of 32, 64 or 128 columns x 4, 2 or 1 consecutive rows, so that the ragged end
// of the rows costs a tile per four (two) rows instead of one per row.  The last such piece of a batch
// element is moved up to end at the last row (rows computed twice are written twice with the same values).
// Columns are written up to the end of the 32-wide panel that holds the last token, which is as far as
// the attention core reads.
#include "of3_device.h"
#include "of3_kernels.h"
#include "of3_launch.h"
#include "of3_pass_bf16.h"

#include <type_traits>

// Waves per work-group of the C = 128 kernel: 8 (two per SIMD, 248 registers) or 16 (four per SIMD,
// 118 registers, one matrix per wave).  Measured at N = 768 inside the block: 126 us against 128 us,
// stand-alone 150 against 158: more waves in flight do not help this pass, the shipped form is 8.
#ifndef OF3_TP_WAVES
#define OF3_TP_WAVES 8
#endif

namespace of3 {

namespace {

// [position][channel] LDS tile.  Readers take, per 8 lanes, either 8 consecutive positions
// (q, k, bias: natural order, so that their stores walk consecutive rows) or the positions
// {x..x+3, x+16..x+19} (v: rowperm16 order).  The key (pos ^ (pos >> 2)) & 7 is distinct
// within 8 lanes for both patterns.
template <int NCH>
__device__ __forceinline__ int proj_slot(int pos, int chunk) {
  const int key = (pos ^ (pos >> 2)) & 7 & (NCH - 1);
  return pos * NCH + (chunk ^ key);
}

// PART: positions of the pieces that the tiles of the last round are dealt in (last_round in of3_tiles.h), 128: whole tiles only.  PER_CU: work-groups
template <int C, int D, int NW, bool RAGGED, int PART, int PER_CU>
__global__ __launch_bounds__(64 * NW, PER_CU == 2 ? NW / 2 : 1) void triattn_proj_kernel(TriattnProjArgs p, int full_per_row, int tail_shift,
                                                               int tiles_per_batch, int whole_tiles, int total_items) {
  constexpr int H = 4;
  constexpr int HD = H * D;
  constexpr int NCH = C / 8;
  constexpr int LPP = NCH;
  constexpr int PPI = 64 / LPP;
  constexpr int TP = 128;
  constexpr int LN_ITERS = (TP / NW) / PPI;
  constexpr int KS = C / 16;
  constexpr int NT = HD / 32;          // 32-row output tiles per matrix (4 or 2)
  constexpr bool WIDE = (NT == 4);
  constexpr bool W16 = (NW == 16);
  // WIDE (H*D = 128), 8 waves: waves 0..3 own output tile w of q and of k, waves 4..7 own tile
  //   w-4 of v plus the bias of position tile w-4; waves w and w+4 share a SIMD, so every SIMD
  //   carries the same MFMA load.
  // WIDE, 16 waves (four per SIMD at 128 registers): waves 0..3 own tile w of q, 4..7 of k, 8..11
  //   of v, 12..15 the bias of position tile w-12; waves w, w+4, w+8, w+12 share a SIMD.
  // else (H*D = 64): waves 0..5 own one (matrix, tile) job, waves 6 and 7 do the bias of two
  //   position tiles each.
  static_assert(!W16 || WIDE, "the sixteen-wave form is built for H*D = 128");
  constexpr int LN_STEP = NW * PPI;    // positions that the waves normalise at a time, PPI consecutive ones each
  static_assert(NT == 4 || NT == 2, "H*D must be 128 or 64");

  __shared__ u32x4_t tile[2][TP * NCH];
  __shared__ u32x4_t wb_lds[KS * 64];  // triangle-bias weights in MFMA A-operand order (rows >= H are zero)

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, l32 = lane & 31, lh = lane >> 5;
  const int ln_chunk = lane % LPP, ln_pp = lane / LPP;

  // affine parameters of this lane's 8 channels, kept packed (8 registers instead of 16) and unpacked once per tile
  const u32x4_t lw_pk = *reinterpret_cast<const u32x4_t*>(p.ln_w + 8 * ln_chunk);
  const u32x4_t lb_pk = *reinterpret_cast<const u32x4_t*>(p.ln_b + 8 * ln_chunk);

  if (wave == 0) {
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      u32x4_t w = {0u, 0u, 0u, 0u};
      if (l32 < H) w = *reinterpret_cast<const u32x4_t*>(p.w_b + l32 * C + 16 * s + 8 * lh);
      wb_lds[s * 64 + lane] = w;
    }
  }  // published by the first tile's barrier
  const float qscale = kLog2e * __builtin_amdgcn_rsqf((float)D);

  const int N = p.N, Jp = p.Jp;
  // tile -> batch element, first row, first column, log2 of the width (wave-uniform); the last ragged piece
  // is moved up to end at the last row, so every row of a tile exists (the launcher makes sure that N >= 4)
  auto tile_origin = [&](int tile_id, int& b, int& i0, int& j0, int& shift) {
    const TilePlace t = tile_place<RAGGED>(tile_id, N, full_per_row, tail_shift, tiles_per_batch, true);
    b = t.b, i0 = t.i0, j0 = t.j0, shift = t.shift;
  };

  u32x4_t raw[LN_ITERS];
  float mraw[LN_ITERS];  // mask of the same positions (used by the lane with ln_chunk == 0)
  // LayerNorm-phase position `it` of this lane, from the item's first one: TP / NW consecutive positions per wave in whole
  // tiles, in pieces LN_STEP by all waves at a time, so that a piece is the first iterations
  auto ln_position = [&](bool in_piece, int it) {
    return in_piece ? it * LN_STEP + wave * PPI + ln_pp : wave * (TP / NW) + it * PPI + ln_pp;
  };
  auto load_tile = [&](int item) {
    const TilePiece piece = tile_piece<PART>(item, whole_tiles);
    int b, i0, j0, shift_rt;
    tile_origin(piece.tile, b, i0, j0, shift_rt);
    const int shift = RAGGED ? shift_rt : 7, jmask = (1 << shift) - 1;
    const bf16_t* xrow = p.x + b * p.x_view.stride_b + i0 * p.x_view.stride_r;  // the tile's first row
    const float* mrow = p.mask ? p.mask + b * p.mask_view.stride_b + i0 * p.mask_view.stride_r : nullptr;
#pragma unroll
    for (int it = 0; it < LN_ITERS; ++it) {
      const int in_item = ln_position(piece.count < TP, it), pos = piece.first + in_item;
      const int di = RAGGED ? pos >> shift : 0, j = j0 + (RAGGED ? pos & jmask : pos);  // every row i0 + di exists
      u32x4_t v = {0u, 0u, 0u, 0u};
      float m = 1.f;
      if ((PART == TP || in_item < piece.count) && j < N) {
        v = *reinterpret_cast<const u32x4_t*>(xrow + di * p.x_view.stride_r + j * p.x_view.stride_k + 8 * ln_chunk);
        if (mrow && ln_chunk == 0) m = mrow[di * p.mask_view.stride_r + j * p.mask_view.stride_k];
      }
      raw[it] = v;
      mraw[it] = m;
    }
  };

  // Every job takes the positions in natural order: position 32*tt + l32 is column l32 of
  // position tile tt (q, k, bias: activations are the MFMA B operand) or, for v, row
  // rowperm16(l32) of it (activations are the A operand, so that a lane ends up with 16
  // consecutive keys of one channel: 32 contiguous bytes of the V^T panel).
  const int krow = rowperm16(l32);

  // A wave's role is fixed for the kernel, and each role runs its own copy of the tile loop:
  //   role 0  q and k of output tile w (H*D = 128), or one of them (H*D = 64: waves 0..3)
  //   role 1  v of output tile w-4 plus the bias of position tile w-4 (H*D = 128), or v alone
  //   role 2  bias of two position tiles (H*D = 64: waves 6, 7)
  // Inside a role every tile issues the same sequence of loads and stores.  Together with the
  // peeled first tile this lets the wait for the values loaded one tile ahead leave the
  // previous tile's stores in flight (the compiler counts them; it cannot when the number
  // depends on a branch).
  auto run = [&](auto role_tag) {
    constexpr int ROLE = decltype(role_tag)::value;
    constexpr int NJ = (ROLE == 0 && WIDE && !W16) ? 2 : (ROLE == 2 ? 0 : 1);
    const int ot = WIDE ? wave % 4 : wave % 2;
    const int m0 = ROLE == 1 ? 2 : (WIDE ? (W16 ? wave / 4 : 0) : wave / 2);  // matrix of job 0: 0 q, 1 k, 2 v

    u32x4_t wj[NJ > 0 ? NJ : 1][KS];
#pragma unroll
    for (int jj = 0; jj < NJ; ++jj) {
      const int m = m0 + jj;
      const bf16_t* W = (m == 0) ? p.w_q : (m == 1 ? p.w_k : p.w_v);
      // q, k (A operands): lane owns 16 consecutive channels (rowperm16); v (B operand): natural rows
      pass_bf16::load_unit<C>(W, ot, (ROLE == 1) ? l32 : rowperm16(l32), lh, p.packed, wj[jj]);
    }

    auto do_tile = [&](auto positions, int item, int buf) {
      constexpr int P = decltype(positions)::value;
      const TilePiece piece = tile_piece<PART>(item, whole_tiles);
      const int first = P == TP ? 0 : piece.first, tt0 = first / 32;
      int b, i0, j0, shift_rt;
      tile_origin(piece.tile, b, i0, j0, shift_rt);
      const int shift = RAGGED ? shift_rt : 7, jmask = (1 << shift) - 1;
      // row and first column of the 32-position tile tt (wave-uniform): one row, one 32-key panel
      auto tile_row = [&](int tt) { return RAGGED ? i0 + ((32 * tt) >> shift) : i0; };
      auto tile_col = [&](int tt) { return RAGGED ? j0 + ((32 * tt) & jmask) : j0 + 32 * tt; };

      // ---- LayerNorm phase (+ mask bias, one lane per position)
      float lw[8], lb[8];
      {
        u32x4_t tw = lw_pk, tb = lb_pk;
        if (WIDE && (RAGGED || PART < TP)) __asm__ volatile("" : "+v"(tw), "+v"(tb));  // keeps the unpacked copies from being hoisted out of the loop
        unpack8(tw, lw);
        unpack8(tb, lb);
      }
#pragma unroll
      for (int it = 0; it < LN_ITERS; ++it) {
        const int pos = first + ln_position(P < TP, it);
        if (P < TP && pos >= first + P) break;
        tile[buf][proj_slot<NCH>(pos, ln_chunk)] = layer_norm_chunk<C>(raw[it], lw, lb);
        if (ln_chunk == 0) {
          const int i = RAGGED ? i0 + (pos >> shift) : i0, j = j0 + (RAGGED ? pos & jmask : pos);
          float mb = -__builtin_inff();
          if (j < N) mb = kLog2e * (p.inf * (mraw[it] - 1.f));
          p.mbias[((size_t)b * N + i) * Jp + j] = mb;
        }
      }
      if (P == TP && item + (int)gridDim.x < total_items) load_tile(item + gridDim.x);
      __syncthreads();  // the only barrier per tile (the LDS tile is double buffered)

      // ---- projection phase
      auto bias_tile = [&](int tt) {  // triangle bias of position tile tt (wave-uniform, may be a run-time value)
        const int pos = 32 * tt + l32, i = tile_row(tt), j0 = tile_col(tt), j = j0 + l32;
        f32x16_t acc = zero16();
#pragma unroll
        for (int s = 0; s < KS; ++s)
          acc = mfma_32x32x16(wb_lds[s * 64 + lane], tile[buf][proj_slot<NCH>(pos, 2 * s + lh)], acc);
        // rows 0..3 of the result sit in registers 0..3 of lanes 0..31
        if constexpr (ROLE == 2) {
          // Lanes 32..63 store past the end of their buffer: with the stores under a condition, and no others in this role, the compiler waits for all of
          // them at the top of the loop (three templates of 300 34.2 / 32.9 us, four of 512 116.8 / 114.8; at 128 channels, where v's come after, no
          // difference).
#pragma unroll
          for (int h = 0; h < H; ++h) {
            const __amdgpu_buffer_rsrc_t row = buffer_rsrc(p.tbias + (((size_t)b * H + h) * N + i) * Jp + j0, 32 * sizeof(float));
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(j < N ? acc[h] * kLog2e : 0.f), row, 4 * l32 + 128 * lh, 0, 0);
          }
        } else if (lh == 0) {
#pragma unroll
          for (int h = 0; h < H; ++h) p.tbias[(((size_t)b * H + h) * N + i) * Jp + j] = (j < N) ? acc[h] * kLog2e : 0.f;
        }
      };
      auto holds = [&](int tt) { return P == TP || (tt >= tt0 && tt < tt0 + P / 32); };
      if (ROLE == 2) {
        if (W16) {
          if (holds(wave - 12)) bias_tile(wave - 12);
        } else {
          if (holds(2 * (wave - 6))) bias_tile(2 * (wave - 6));
          if (holds(2 * (wave - 6) + 1)) bias_tile(2 * (wave - 6) + 1);
        }
        return;
      }
#pragma unroll
      for (int u = 0; u < P / 32; ++u) {  // every wave visits all position tiles
        const int tt = tt0 + u;
        if (!RAGGED && WIDE && PART < TP) __builtin_amdgcn_sched_barrier(0);  // operands of the next position tile held early cost spills
        const size_t bi = (size_t)b * N + tile_row(tt);
        const int jt = tile_col(tt);
#pragma unroll
        for (int jj = 0; jj < NJ; ++jj) {
          f32x16_t acc = zero16();
          u32x4_t o0, o1;
          bf16_t* dst;
          if (ROLE == 1) {
            // V^T panel of this position tile: rows = keys (A), columns = channels (B)
            const int kpos = 32 * tt + krow;
#pragma unroll
            for (int s = 0; s < KS; ++s)
              acc = mfma_32x32x16(tile[buf][proj_slot<NCH>(kpos, 2 * s + lh)], wj[jj][s], acc);
            // lane: channel 32*ot + l32 = head*D + d, keys 16*lh + (0..15) of the panel
            const int ch = 32 * ot + l32;
            const int head = ch / D, d = ch % D;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              o0[q] = pack_bf16(acc[2 * q], acc[2 * q + 1]);
              o1[q] = pack_bf16(acc[8 + 2 * q], acc[8 + 2 * q + 1]);
            }
            dst = p.vt + (bi * H + head) * D * Jp + (size_t)(jt >> 5) * (D * 32) + d * 32 + 16 * lh;
          } else {
            // the activation operand is re-read from LDS by every job: cheaper than holding it in
            // 32 registers across the jobs
            const int pos = 32 * tt + l32;
#pragma unroll
            for (int s = 0; s < KS; ++s)
              acc = mfma_32x32x16(wj[jj][s], tile[buf][proj_slot<NCH>(pos, 2 * s + lh)], acc);
            // lane owns channels 32*ot + 16*lh + v  ->  head, d0 .. d0+15
            const int ch0 = 32 * ot + 16 * lh;
            const int head = ch0 / D, d0 = ch0 % D;
            const bool is_q = (m0 + jj) == 0;
            const float sc = is_q ? qscale : 1.f;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              o0[q] = pack_bf16(acc[2 * q] * sc, acc[2 * q + 1] * sc);
              o1[q] = pack_bf16(acc[8 + 2 * q] * sc, acc[8 + 2 * q + 1] * sc);
            }
            dst = (is_q ? p.q : p.k) + ((bi * H + head) * Jp + jt + l32) * D + d0;
          }
          *reinterpret_cast<u32x4_t*>(dst) = o0;
          *reinterpret_cast<u32x4_t*>(dst + 8) = o1;
        }
      }
      if (ROLE == 1 && WIDE && !W16 && holds(wave - 4)) bias_tile(wave - 4);
    };

    typedef std::integral_constant<int, TP> Whole;
    int item = blockIdx.x;
    int buf = 0;
    if (item >= total_items) return;
    load_tile(item);
    if (PART == TP || item < whole_tiles) {
      do_tile(Whole{}, item, buf);
      item += gridDim.x;
      buf ^= 1;
    }
    for (; item < whole_tiles; item += gridDim.x, buf ^= 1) do_tile(Whole{}, item, buf);
    if constexpr (PART < TP) {
      if (item < total_items) do_tile(std::integral_constant<int, PART>{}, item, buf);  // one piece: the last round
    }
  };

  if (W16) {
    if (wave < 8) run(std::integral_constant<int, 0>{});
    else if (wave < 12) run(std::integral_constant<int, 1>{});
    else run(std::integral_constant<int, 2>{});
  } else if (WIDE) {
    if (wave < 4) run(std::integral_constant<int, 0>{});
    else run(std::integral_constant<int, 1>{});
  } else {
    if (wave < 4) run(std::integral_constant<int, 0>{});
    else if (wave < 6) run(std::integral_constant<int, 1>{});
    else run(std::integral_constant<int, 2>{});
  }
}

template <int C, int D, int NW, bool RAGGED, int PER_CU>
hipError_t launch(const TriattnProjArgs& a, const RaggedTiles& t, long total, hipStream_t stream) {
  static int cache[kMaxDevices];
  int grid_cap = 0;
  hipError_t e = per_device(
      cache, [&](int dev, int* v) { return C == 64 ? cu_count(dev, v) : resident_blocks(triattn_proj_kernel<C, D, NW, RAGGED, 128, PER_CU>, 64 * NW, dev, v); },
      &grid_cap);
  if (e != hipSuccess) return e;
  if (C == 64) grid_cap *= PER_CU;
  const LastRound r = last_round(total, grid_cap);
  const int grid = r.items < grid_cap ? r.items : grid_cap;
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(grid), dim3(64 * NW), 0, stream, a, t.full_per_row, t.tail_shift, t.per_batch, r.whole, r.items);
  };
  if (r.piece == 32) go(triattn_proj_kernel<C, D, NW, RAGGED, 32, PER_CU>);
  else if (r.piece == 64) go(triattn_proj_kernel<C, D, NW, RAGGED, 64, PER_CU>);
  else go(triattn_proj_kernel<C, D, NW, RAGGED, 128, PER_CU>);
  return hipGetLastError();
}
template <int C, int D, int NW, bool RAGGED>
hipError_t launch_tiles(const TriattnProjArgs& a, hipStream_t stream) {
  RaggedTiles t = {a.Jp / 128, 7, a.N * (a.Jp / 128)};  // whole (padded) rows in 128-wide pieces
  if (RAGGED) t = ragged_tiles(a.N, 5);                 // pieces of whole 32-key panels
  const long total = (long)a.B * t.per_batch;
  if (total > 0x7fffffffL) return hipErrorInvalidValue;
  if constexpr (C == 64) {
    // Two work-groups to a CU, whose barriers do not coincide, from more than one tile per CU up to sixteen; us a launch, one / two: templates 2 x 300 24.9 /
    // 23.3, 4 x 300 43.3 / 40.5, 3 x 400 58.6 / 56.2, 1 x 512 31.0 / 29.8, 2 x 384 34.0 / 33.6; beyond, where the passes move 5 TB/s, 4 x 384 64.4 / 64.2, 3 x 500
    // 93.9 / 95.6, 4 x 450 101.2 / 104.6.  Launches one after another prefer one earlier (2 x 450 47.1 / 48.9, 3 x 360 43.8 / 46.2), whole passes do not: 2 x 390
    // 1120 / 1109, 2 x 450 1441 / 1433, 3 x 360 1303 / 1288, 3 x 430 2008 / 1990, 2 x 512 1769 / 1772, 4 x 256 773 / 776; beyond, 3 x 512 2695 / 2712, 4 x 512 3489 /
    // 3517.  (Whole rows in 128 registers spill 10, which costs long launches 3 %.)
    static int cache[kMaxDevices];
    int cus = 0;
    const hipError_t e = per_device(cache, [](int dev, int* v) { return cu_count(dev, v); }, &cus);
    if (e != hipSuccess) return e;
    if (total > cus && total <= 16L * cus) return launch<C, D, NW, RAGGED, 2>(a, t, total, stream);
  }
  return launch<C, D, NW, RAGGED, 1>(a, t, total, stream);
}

}  // namespace

hipError_t triattn_proj_launch(const TriattnProjArgs& args, int C, int D, hipStream_t stream) {
  if (args.H != 4 || (C != 128 && C != 64) || 4 * D != C) return hipErrorInvalidValue;
  // Short sequences on 32-position tiles, under the rule of the triangle multiplication's input pass (C = 128, packed, us,
  // 128- against 32-position tiles: N = 40 8.1 / 6.0, 64 8.6 / 6.8, 80 10.5 / 8.7, 96 11.1 / 9.6, 128 12.1 / 13.0).
  bool small = false;
  const hipError_t e = small_pass(args.B, args.N, 1, &small);
  if (e != hipSuccess) return e;
  if (small) return triattn_proj_panels_launch(args, C, stream);
  // ragged pieces hold up to four rows, all of which must exist
  const bool ragged = args.N % 128 != 0 && args.N >= 4;
  if (C == 128) return ragged ? launch_tiles<128, 32, OF3_TP_WAVES, true>(args, stream) : launch_tiles<128, 32, OF3_TP_WAVES, false>(args, stream);
  return ragged ? launch_tiles<64, 16, 8, true>(args, stream) : launch_tiles<64, 16, 8, false>(args, stream);
}

}  // namespace of3
