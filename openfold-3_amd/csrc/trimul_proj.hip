// Triangle-multiplication input pass: LayerNorm(z) and the four gated projections
//     a = mask * sigmoid(zn Wag^T) * (zn Wap^T),   b = mask * sigmoid(zn Wbg^T) * (zn Wbp^T)
// (triangular_multiplicative_update.py:485-493), written channel-major in the k-panel
// layout a[b][c][k/32][r][k%32] the contraction kernel streams from, so that the
// contraction is a plain "row times row" product for both directions: the caller's PairView
// makes (r, k) = (i, k) for the outgoing update and (r, k) = (i, k) of the transposed tensor
// for the incoming one.
//
// Persistent work-groups of 8 waves (at 64 channels also of 4), two per SIMD, so that
// one wave's MFMAs overlap the other's VALU work, keep the four weight
// matrices in registers as MFMA A operands, one 32-row slice pair per wave; each tile of
// 128 positions is normalised in registers (statistics by DPP lane permutations), staged
// once in LDS as bf16 and consumed as the MFMA B operand by all waves.  The LDS tile is
// double buffered, which leaves a single barrier per tile.  Positions are dealt to MFMA
// columns so that a lane finishes 4 consecutive k of one row and channel and stores them as
// one 8-byte vector.  A tile is 4 consecutive rows r of one 32-wide k-panel: in the k-panel
// layout these are 256 contiguous bytes per channel, so 32 lanes write whole 128-byte lines.
// Only the panels that hold a k below N are written (the last one with zeros from N on), and only
// the rows up to N rounded up to 4: the contraction sums over no other panel, and what it makes of
// the other rows lands in rows and columns of x that nobody reads.
#include "of3_device.h"
#include "of3_kernels.h"
#include "of3_launch.h"
#include "of3_pass_bf16.h"

#include <type_traits>

namespace of3 {

namespace {

int panels_of(const TrimulProjArgs& a) { return (a.N + 31) / 32; }  // the panels that hold a k below N; the contraction reads no others

// PART: positions of the pieces that the tiles of the last round are dealt in (last_round in of3_tiles.h), 128: whole tiles only.
// NW: waves per work-group
template <int C, int CH, int PART, int NW>
__global__ __launch_bounds__(64 * NW, 2) void trimul_proj_kernel(TrimulProjArgs p, int panels, int whole_tiles, int total_items) {
  constexpr int NCH = C / 8;        // 16-byte chunks per position
  constexpr int LPP = NCH;          // lanes sharing one position in the LayerNorm phase
  constexpr int PPI = 64 / LPP;     // positions per wave instruction
  constexpr int TP = 128;           // positions per tile: TR rows x one 32-wide k-panel
  constexpr int TR = TP / 32;
  constexpr int LN_ITERS = (TP / NW) / PPI;
  constexpr int LN_STEP = NW * PPI; // positions that the waves normalise at a time where they share a row
  constexpr int KS = C / 16;        // MFMA k-steps
  constexpr int OT = CH / 32;       // 32-row output tiles per matrix
  constexpr int NJOBS = 2 * OT;     // (a|b, output tile) jobs: 8 or 4
  constexpr int WPJ = NW / NJOBS;   // waves sharing a job: 1 or 2, each takes 4/WPJ position tiles
  constexpr int TPW = 4 / WPJ;      // position tiles per wave: 4 or 2
  static_assert(NJOBS == 8 || NJOBS == 4, "CH must be 128 or 64");

  // two tiles: LayerNorm of tile n+1 is written while other waves still read tile n
  __shared__ u32x4_t tile[2][TP * NCH];

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, l32 = lane & 31, lh = lane >> 5;
  const int ln_chunk = lane % LPP, ln_pp = lane / LPP;

  // LayerNorm affine parameters of this lane's 8 channels, kept packed (8 registers instead
  // of 16) and unpacked once per tile
  u32x4_t lw_pk = *reinterpret_cast<const u32x4_t*>(p.ln_w + 8 * ln_chunk);
  u32x4_t lb_pk = *reinterpret_cast<const u32x4_t*>(p.ln_b + 8 * ln_chunk);
  __asm__ volatile("" : "+v"(lw_pk), "+v"(lb_pk));  // waited for here, once

  // this wave's job: gate and projection rows 32*ot .. +31 of a (pair 0) or b (pair 1),
  // resident in registers as MFMA A operands for the whole kernel
  const int job = wave % NJOBS, tgroup = wave / NJOBS;
  const int pair = job / OT, ot = job % OT;
  u32x4_t wg[KS], wp[KS];
  {
    const bf16_t* Wg = pair ? p.w_bg : p.w_ag;
    const bf16_t* Wp = pair ? p.w_bp : p.w_ap;
    pass_bf16::load_unit<C>(Wg, ot, l32, lh, p.packed, wg);
    pass_bf16::load_unit<C>(Wp, ot, l32, lh, p.packed, wp);
    // the weights count as used here: the compiler waits for them once, before the tile loop,
    // instead of carrying "may still be in flight" into every iteration (where its wait for
    // them would also be a wait for the tile's prefetch and the previous tile's stores)
#pragma unroll
    for (int s = 0; s < KS; ++s) __asm__ volatile("" : "+v"(wg[s]), "+v"(wp[s]));
  }
  bf16_t* const out = pair ? p.b : p.a;

  const int N = p.N, Np = p.Np;
  const int tiles_per_batch = ((N + TR - 1) / TR) * panels;

  // LayerNorm-phase position `it` of this lane: a wave takes PPI consecutive ones per instruction.  Whole tiles of 128
  // channels: TP / NW consecutive positions per wave (N = 768: 112 against 115 us); pieces, and 64 channels (4 x 512^2: 91 against 101): LN_STEP
  // positions by all waves at a time, so that a piece is the first iterations.
  constexpr bool RUNS = C == 128;
  auto ln_first = [&](bool piece, int it) {  // of the wave's PPI positions, which share a row
    return RUNS && !piece ? wave * (TP / NW) + it * PPI : it * LN_STEP + wave * PPI;
  };
  // Everything a tile reads from global memory (its z values and this lane's mask values) is
  // requested one tile ahead by a fixed number of unconditional loads (positions past the end
  // are clamped to the last one and zeroed through the mask value), and every tile issues the
  // same 16 stores (the padding rows of a and b are written too, with zeros).  With fixed
  // counts the compiler's wait for the prefetched values can leave the previous tile's stores
  // in flight; with a load or store under a condition it cannot, and waits for all of them.
  u32x4_t raw[LN_ITERS];
  float mraw[TPW];
  const float* const mask_base = p.mask ? p.mask : reinterpret_cast<const float*>(p.ln_w);  // dummy when absent
  const int64_t msb = p.mask ? p.mask_view.stride_b : 0, msr = p.mask ? p.mask_view.stride_r : 0,
                msk = p.mask ? p.mask_view.stride_k : 0;
  // Positions of a tile, or of a piece of P positions, are dealt to MFMA columns so that a lane finishes
  // T = min(P / (32 WPJ), 1) consecutive ones: position  32*T*tgroup + T*l32 + tt  is column l32 of this wave's tile tt.
  struct Place {
    int b, r0, k0;  // batch element, first row, first k
  };
  auto place = [&](int item) {
    const TilePiece piece = tile_piece<PART>(item, whole_tiles);
    Place t;
    t.b = piece.tile / tiles_per_batch;
    const int rem = piece.tile - t.b * tiles_per_batch, rg = rem / panels;
    t.r0 = rg * TR + piece.first / 32;
    t.k0 = (rem - rg * panels) * 32;
    return t;
  };
  auto load_tile = [&](int item) {
    const Place t = place(item);
    const bool piece = PART < TP && item >= whole_tiles;
    // a piece issues the loads of a whole tile, the ones it has no use for from its last row again
    const int rows = piece ? PART / 32 : TR, per_lane = piece ? (PART / 32 + WPJ - 1) / WPJ : TPW;
    const int last = t.r0 + rows - 1 < N ? t.r0 + rows - 1 : N - 1;
    const bf16_t* base = p.z + t.b * p.z_view.stride_b + 8 * ln_chunk;
#pragma unroll
    for (int it = 0; it < LN_ITERS; ++it) {
      const int pos = ln_first(piece, it);
      int row = t.r0 + (pos >> 5), k = t.k0 + (pos & 31) + ln_pp;
      row = row < last ? row : last;
      k = k < N ? k : N - 1;
      raw[it] = *reinterpret_cast<const u32x4_t*>(base + row * p.z_view.stride_r + k * p.z_view.stride_k);
    }
    const int pos0 = per_lane * (32 * tgroup + l32);
    int mr = t.r0 + (pos0 >> 5);
    mr = mr < last ? mr : last;
    const float* mrow = mask_base + t.b * msb + mr * msr;
#pragma unroll
    for (int tt = 0; tt < TPW; ++tt) {
      int km = t.k0 + (pos0 & 31) + tt;
      km = km < N ? km : N - 1;
      mraw[tt] = mrow[km * msk];
    }
  };

  auto do_tile = [&](auto positions, int item, int buf) {
    constexpr int P = decltype(positions)::value;
    constexpr int T = P / 32 >= WPJ ? P / 32 / WPJ : 1;  // positions per lane
    constexpr int KSH = T == 4 ? 2 : T == 2 ? 1 : 0;     // swizzle key from pos / T: distinct for the 8 lanes of a read group
    const Place t = place(item);
    const int pos0 = 32 * T * tgroup + T * l32;
    const int b = t.b, r = t.r0 + (pos0 >> 5);  // this lane's row and first k
    const int kfirst = t.k0 + (pos0 & 31);

    float mval[T];
#pragma unroll
    for (int tt = 0; tt < T; ++tt) mval[tt] = (kfirst + tt < N && r < N) ? (p.mask ? mraw[tt] : 1.f) : 0.f;
    bool not_one = false;
#pragma unroll
    for (int tt = 0; tt < T; ++tt) not_one |= mval[tt] != 1.f;
    const bool masked = __builtin_amdgcn_ballot_w64(not_one) != 0;  // wave-uniform

    // ---- LayerNorm phase
    float lw[8], lb[8];
    {
      u32x4_t tw = lw_pk, tb = lb_pk;
      __asm__ volatile("" : "+v"(tw), "+v"(tb));  // keeps the unpacked copies from being hoisted out of the loop
      unpack8(tw, lw);
      unpack8(tb, lb);
    }
#pragma unroll
    for (int it = 0; it < LN_ITERS; ++it) {
      const int pos = ln_first(P < TP, it) + ln_pp;
      if (P < TP && pos >= P) break;
      tile[buf][tile_slot<NCH, KSH>(pos, ln_chunk)] = layer_norm_chunk<C>(raw[it], lw, lb);
    }
    // next tile's z travels while this tile's matrix phase runs
    if (P == TP && item + (int)gridDim.x < total_items) load_tile(item + gridDim.x);
    // One barrier per tile: it publishes this tile, and since every wave has finished the
    // previous tile's matrix phase before arriving, the other buffer may be overwritten by
    // the next LayerNorm phase.
    __syncthreads();
    if (P < TP && 32 * T * tgroup >= P) return;  // of a whole tile every wave has a part, which the compiler cannot tell: it would count no stores

    // ---- projection phase
    float res[T][16];
#pragma unroll
    for (int tt = 0; tt < T; ++tt) {
      f32x16_t accg = zero16(), accp = zero16();
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const u32x4_t bop = tile[buf][tile_slot<NCH, KSH>(pos0 + tt, 2 * s + lh)];
        accg = mfma_32x32x16(wg[s], bop, accg);
        accp = mfma_32x32x16(wp[s], bop, accp);
      }
      // mask * sigmoid(gate) * projection; a wave whose positions all carry mask 1 (the usual tile)
      // skips the multiplication by 1
      if (masked) {
#pragma unroll
        for (int v = 0; v < 16; ++v) res[tt][v] = (mval[tt] * sigmoidf_fast(accg[v])) * accp[v];
      } else {
#pragma unroll
        for (int v = 0; v < 16; ++v) res[tt][v] = sigmoidf_fast(accg[v]) * accp[v];
      }
    }
    // stores: register v of a lane is channel 32*ot + 8*(v/4) + 4*lh + v%4; k-panel layout
    // plane[k / 32][row][k % 32].  r < Np always (Np is a multiple of 128): rows between N and
    // Np receive zeros
    {
      // lane base: channel 32*ot + 4*lh of this batch element, row r, first k of the lane;
      // the 16 registers add wave-uniform channel offsets
      const size_t plane = (size_t)Np * Np;
      bf16_t* dst0 = out + ((size_t)b * CH + 32 * ot + 4 * lh) * plane + (size_t)(kfirst >> 5) * (Np * 32) + r * 32 +
                     (kfirst & 31);
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        bf16_t* dst = dst0 + (size_t)(8 * (v >> 2) + (v & 3)) * plane;
        if constexpr (T == 4) {
          u32x2_t w2 = {pack_bf16(res[0][v], res[1][v]), pack_bf16(res[2][v], res[3][v])};
          *reinterpret_cast<u32x2_t*>(dst) = w2;
        } else if constexpr (T == 2) {
          *reinterpret_cast<uint32_t*>(dst) = pack_bf16(res[0][v], res[1][v]);
        } else {
          *dst = to_bf16(res[0][v]);
        }
      }
    }
  };

  // the first tile is peeled: the loop proper is only entered with a tile's stores in flight
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
}

template <int C, int CH, int NW>
hipError_t launch(const TrimulProjArgs& a, long tiles, hipStream_t stream) {
  static int cache[kMaxDevices];
  int grid_cap = 0;
  hipError_t e = per_device(cache, [&](int dev, int* v) { return resident_blocks(trimul_proj_kernel<C, CH, 128, NW>, 64 * NW, dev, v); }, &grid_cap);
  if (e != hipSuccess) return e;
  const LastRound r = last_round(tiles, grid_cap);
  const int grid = r.items < grid_cap ? r.items : grid_cap;
  auto go = [&](auto kern) { hipLaunchKernelGGL(kern, dim3(grid), dim3(64 * NW), 0, stream, a, panels_of(a), r.whole, r.items); };
  if (r.piece == 32) go(trimul_proj_kernel<C, CH, 32, NW>);
  else if (r.piece == 64) go(trimul_proj_kernel<C, CH, 64, NW>);
  else go(trimul_proj_kernel<C, CH, 128, NW>);
  return hipGetLastError();
}

}  // namespace

hipError_t trimul_proj_launch(const TrimulProjArgs& args, int C, int CH, hipStream_t stream) {
  if ((C != 128 && C != 64) || CH != C) return hipErrorInvalidValue;
  // Short sequences on 32-position tiles.  256 CUs, C = 128, us per pass, packed weights, 128- against 32-position tiles:
  // N = 40 8.3 / 6.3, 64 8.9 / 6.8, 80 9.8 / 7.8, 96 10.6 / 10.5, 160 11.4 / 13.8 (row-major weights 10.9 / 12.5 at 96): the
  // line lies at one tile per CU.  At 64 channels (B = 2) 5.6 / 4.4 at N = 64, even at 80.
  bool small = false;
  const hipError_t e = small_pass(args.B, args.N, 1, &small);
  if (e != hipSuccess) return e;
  if (small) return trimul_proj_panels_launch(args, C, stream);
  const long tiles = (long)args.B * ((args.N + 3) / 4) * panels_of(args);
  if (C == 128) return launch<128, 128, 8>(args, tiles, stream);
  // 64 channels: from more than two tiles per CU on two work-groups of four waves to a CU, whose LayerNorms and products do not coincide, in the
  // place of one of eight in which two waves share a tile's positions.  us a launch, eight / four waves: 350 tiles (200 tokens) 9.9 / 10.4, 360 10.4 / 10.6,
  // 564 (two templates of 187) 13.4 / 12.4, three templates of 300 31.0 / 29.2, four of 512 103.4 / 93.2; three to a CU, at 168 registers, 21 of
  // them spilled, 122.7 for the last.  128 channels have twice the matrices: two pairs to a wave, on tiles of 64 positions, spill too and store 4 bytes a
  // lane (N = 384 38.2 / 39.5, 768 124 / 158).
  static int cache[kMaxDevices];
  int cus = 0;
  const hipError_t s = per_device(cache, [](int dev, int* v) { return cu_count(dev, v); }, &cus);
  if (s != hipSuccess) return s;
  return tiles > 2L * cus ? launch<64, 64, 4>(args, tiles, stream) : launch<64, 64, 8>(args, tiles, stream);
}

}  // namespace of3
