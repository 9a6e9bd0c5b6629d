// fp32 pair transition (transition.py:225-271, activations.py:33-61) at 64 and 128 channels with a hidden width in
// multiples of 128, products on the fp16 matrix instructions with operands split into two fp16 terms:
//     out = [x +] ((silu(LN(x) Wa^T) * (LN(x) Wb^T)) Wout^T) * mask
// pair_f32.hip has the kernels for every other shape.
//
// 18 flops per channel and hidden channel in fp16 products: 0.17 Tflop for N = 384 at n = 4, 145 us at the 1.2 PFLOP/s of a large bf16
// product, 207.5 taken (0.84).  The split weights (393 KB at C = 128, n = 4) do not fit a CU and stream from L2.
// One wave per tile of 32 hidden channels and all of the tile's positions: a work-group of eight waves takes the
// hidden dimension in slices of 32 S channels (S = 8, or 4 with a wave per position tile), so that an operand of Wa
// and Wb is read once for 64 positions and a slice of 256 hidden channels costs two barriers, against 32 positions
// and slices of 128 in pair_f32.hip's kernel.  Many tiles: work-groups of four waves with slices of 128, two to a CU (NW).  The operands of a k-step are requested one to four steps ahead, those of
// the other product before the barrier between them.  Below two tiles of 64 positions per CU, tiles of 32 positions (two
// waves then share the sum of the second product).
#include "of3_pass_f32.h"
#include "of3_weight_split.h"

namespace of3 {

namespace {

using namespace pass_f32;

struct TransitionPass {
  const float *x, *mask;
  PairView xv, mv;
  const float *ln_w, *ln_b;
  WeightX3 s_a, s_b, s_out;
  float* out;
  int R, L;     // rows per batch element, positions per row
  int panels;   // 32-position panels per row
  int total;    // panels in all
  int HID, add_residual;
  // the attention before it (AFTER)
  const float *att_o, *att_ln_w, *att_ln_b;
  WeightX3 att_g, att_out;
  int N;
  // the pair bias of the result (BIAS)
  const float *pb_w, *pb_ln_w, *pb_ln_b;
  float* pb_out;
  int pb_H;
};

constexpr int kRowLd = 4;  // floats between the rows of the updated tile, beside their channels
template <int C, int S, int NPT, bool AFTER, bool BIAS>
constexpr size_t transition_lds() {
  return (size_t)NPT * (HalfTile<C>::SLOTS + HalfTile<32 * S>::SLOTS) * 16 + 2 * C * sizeof(float) +
         (AFTER ? (2 * C + 32 * (C + kRowLd)) * sizeof(float) : 0) + (BIAS ? PassTile<C>::SLOTS * 16 : 0);
}

// AFTER: the tile begins with the output pass of the ending node's triangle attention (triattn_out_pass: same steps, same bits), its gates in
// the first four waves and its output projection in the others; the updated rows stay in LDS.
// BIAS: and ends with the pair bias of the block's attention over s (pair_bias_pass: same steps, same bits), from the rows that it has just finished. Four
// trunk blocks at N = 24 / 45 / 64 / 80 / 90 527 / 579 / 587 / 696 / 758 us, so 502 / 554 / 565 / 671 / 736 (a launch, and z read once more).
// KEEP: the hidden dimension is one slice, a wave's operands of all three matrices stay in registers (96 of 208).  Three templates of 200, 64
// channels, n = 2, two transitions of 2100 tiles: the operands fetched again for every tile 107 us, so 90.
// NW: waves of the work-group.  With four, each has a hidden tile and an output tile for all of the tile's positions, and two work-groups share a
// CU: their barriers, LayerNorms and SiLUs do not coincide, and at 128 channels an operand of Wout serves both position tiles.  One of eight waves /
// two of four, us: 128 channels, n = 4, N = 384 211.5 / 207.5 (matrix pipe 43 % busy, vector pipe 32 %; 196 with every weight in
// the L1, so no wait for those), 64 channels, KEEP, 44.2 / 40.6.  Same bits.
template <int C, int S, int NPT, bool AFTER, bool BIAS, bool KEEP, int NW>
__global__ __launch_bounds__(64 * NW, 2) void transition_pass(TransitionPass p) {
  static_assert(AFTER || !BIAS, "one tile per work-group");
  static_assert(!AFTER || (C == 128 && NPT == 1), "eight waves: a gate and an output tile for each 32 channels");
  static_assert(S == NW || (S == 4 && NW == 8 && NPT == 2), "the waves share the hidden tiles of a slice");
  typedef HalfTile<C> XTile;
  typedef HalfTile<32 * S> HTile;
  constexpr int KS = C / 16, OT = C / 32, RG = 8 / NW;  // RG: rows of a position tile that a lane has a part of
  constexpr int XT = S == NW ? NPT : 1;                 // position tiles of a wave in the first product
  constexpr int OP = OT * NPT > NW ? OT * NPT / NW : 1;  // ... in the second
  constexpr int KSPLIT = NW * OP / (OT * NPT);          // waves sharing an output tile's sum in the second
  static_assert(OP == 1 || OP == NPT, "");
  constexpr int OSTEPS = 2 * S / KSPLIT;           // its k-steps per slice and wave
  // steps that an operand is requested ahead: an L2 read takes about as long as 24 MFMAs of two waves per SIMD
  constexpr int DA = KEEP ? KS : XT == 1 ? 2 : 1, DO = KEEP ? OSTEPS : 4 / OP;
  static_assert(OSTEPS >= DO && KS >= DA, "");
  // the residual before the next tile's rows, a slice's scales before its operands and Wout's first operands before the hidden values; there
  // they would spill (four templates of 200, 64 channels, n = 4: with 4 registers spilled 1242 us a pass, so 1238; two of 300 1453, 1446)
  constexpr bool kEarly = !(C == 64 && S == 8 && NPT == 2), kEarlyRes = kEarly && OP == 1;
  extern __shared__ u32x4_t lds[];
  u32x4_t* const hid = lds + NPT * XTile::SLOTS;
  float* ln = reinterpret_cast<float*>(hid + NPT * HTile::SLOTS);  // [2][C]
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ht = S == NW ? wave : wave & 3, pt_a = S == NW ? 0 : wave >> 2;
  const int ot = wave % OT, pt_b = OP > 1 ? 0 : (wave / OT) % NPT, kh = wave / (OT * NPT);
  const int L = p.L, slices = KEEP ? 1 : p.HID / (32 * S);
  // The activations' scale is in ln, those of the hidden channels are in the rows of Wb, their inverses in the columns of Wout
  const float x_scale = p.s_a.scales()[0].input;
  ColumnScales so(p.s_out, p.HID / 32);
  for (int c = tid; c < C; c += 64 * NW) ln[c] = p.ln_w[c] * x_scale, ln[C + c] = p.ln_b[c] * x_scale;

  const int lane0 = tid & 63, src_lane = rowperm16(lane0 & 31) + (lane0 & 32);  // outputs dealt by rowperm16
  const u32x4_t* wa = reinterpret_cast<const u32x4_t*>(p.s_a.h) + src_lane;
  const u32x4_t* wb = reinterpret_cast<const u32x4_t*>(p.s_b.h) + src_lane;
  const u32x4_t* wo = reinterpret_cast<const u32x4_t*>(p.s_out.h) + (size_t)(ot * (p.HID / 16) + kh * OSTEPS) * 64 + src_lane;
  const long pa = p.s_a.plane / 8, po = p.s_out.plane / 8;

  auto row_of = [&](int pn, int& j0) {  // element offsets of the panel's row in x and in the mask
    const int r = pn / p.panels;
    j0 = 32 * (pn - r * p.panels);
    return r;
  };
  RowRegs<C> raw[NPT][RG];
  auto load_tile = [&](int tile) {
    const Lane here = lane_here();
#pragma unroll
    for (int t = 0; t < NPT; ++t) {
      int pn = NPT * tile + t, j0;
      pn = pn < p.total ? pn : p.total - 1;
      const int r = row_of(pn, j0), b = r / p.R, i = r - b * p.R;
#pragma unroll
      for (int g = 0; g < RG; ++g) {
        int j = j0 + 4 * (NW * g + wave) + here.lg;
        j = j < L ? j : L - 1;
        load_row<C>(p.x + b * p.xv.stride_b + i * p.xv.stride_r + (int64_t)j * p.xv.stride_k, here.li, raw[t][g]);
      }
    }
  };
  u32x4_t na[DA][2], nb[DA][2], no[DO][2];  // operands of the next steps
  auto fetch_ab = [&](int slice, int s) {
    const size_t at = ((size_t)(slice * S + ht) * KS + s) * 64;
#pragma unroll
    for (int pl = 0; pl < 2; ++pl) na[s % DA][pl] = wa[pl * pa + at], nb[s % DA][pl] = wb[pl * pa + at];
  };
  auto fetch_o = [&](int slice, int s) {
    const size_t at = (size_t)(slice * 2 * S + s) * 64;
#pragma unroll
    for (int pl = 0; pl < 2; ++pl) no[s % DO][pl] = wo[pl * po + at];
  };

  if constexpr (KEEP) {
#pragma unroll
    for (int s = 0; s < KS; ++s) fetch_ab(0, s);
#pragma unroll
    for (int s = 0; s < OSTEPS; ++s) fetch_o(0, s);
    wait_vmcnt<0>();  // no wait for them, and with it for the rows in flight, inside the loop
  }
  const int tiles = (p.total + NPT - 1) / NPT;
  int tile = grid_slot();
  if (tile < tiles) load_tile(tile);
  float* const att_ln = ln + 2 * C;         // [2][C]
  float* const rows = att_ln + 2 * C;       // [32][C + kRowLd]
  if (AFTER)
    for (int c = tid; c < C; c += 64 * NW) {
      const float s = p.att_g.scales()[0].input;
      att_ln[c] = p.att_ln_w[c] * s, att_ln[C + c] = p.att_ln_b[c] * s;
    }
  so.finish();
  auto scales_of = [&](int slice, float& ua, float& ub) {
    ua = p.s_a.scales()[slice * S + ht].unscale, ub = ua * p.s_b.scales()[slice * S + ht].store * so.at(slice * S + ht);
  };
  // KEEP: the scales of the only slice once for all tiles, the first rows waited for here, and all waves on the way of the stores, so that the compiler's wait for
  // a tile's rows inside the loop counts the stores of the tile before and leaves them in flight.  us a launch, before / now: templates 2 x 100 12.8 / 12.1, 3 x
  // 200 42.5 / 39.2, 2 x 300 57.6 / 51.6, 4 x 384 158 / 146, 2 x 512 142 / 130
  float kept_a = 0.f, kept_b = 0.f;
  if constexpr (KEEP) {
    scales_of(0, kept_a, kept_b);
    wait_vmcnt<0>();
  }
  __syncthreads();
  for (; tile < tiles; tile += gridDim.x) {
    if constexpr (AFTER) {
      const XTile xn = {lds}, gated = {hid};
      u32x4_t w[KS][2];
      load_unit<C, 2>(kh == 0 ? p.att_g : p.att_out, ot, src_lane, w);
      ColumnScales att_so(p.att_out, OT);
      const float att_tile = p.att_out.scales()[ot].unscale, att_g_unscale = p.att_g.scales()[ot].unscale;
      int j0;
      const int b = row_of(tile, j0);  // one row per batch element
      const Lane here = lane_here();
      float4 o[4];
      if (kh == 0) {
        const int f = j0 + here.l32 < L ? j0 + here.l32 : L - 1, r = f / p.N, k = f - r * p.N;
        const float* src = p.att_o + (((size_t)b * p.N + k) * p.N + r) * C + 32 * ot + 16 * here.lh;
#pragma unroll
        for (int a = 0; a < 4; ++a) o[a] = *reinterpret_cast<const float4*>(src + 4 * a);
      }
      // the operands of a step are read one step ahead, no further: all of them do not fit the registers
      auto product = [&](const XTile& t) {
        HalfSum<C, true> sum;
        u32x4_t nxt[2];
        const Lane at = lane_here();
        auto read = [&](int s) {
          const u32x4_t* x = t.s + XTile::slot(at.l32, 2 * s + at.lh);
          nxt[0] = x[0], nxt[1] = x[XTile::PLANE];
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
      const int pos = 4 * wave + here.lg;
      float4 y[C / 64];
      norm_row<C>(raw[0][0], att_ln, here.li, y);
#pragma unroll
      for (int e = 0; e < C / 64; ++e) {
        xn.store4(pos, here.li + 16 * e, y[e]);
        *reinterpret_cast<float4*>(rows + pos * (C + kRowLd) + 64 * e + 4 * here.li) = raw[0][0].v[e];
      }
      att_so.finish();
      const float o_scale = att_so.of(att_tile), att_unscale = kh == 0 ? att_g_unscale : att_so.total;
      __syncthreads();
      if (kh == 0) {
        const f32x16_t gate = product(xn);
        const Lane mid = lane_here();
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) {
          const float4 o0 = o[2 * hf], o1 = o[2 * hf + 1];
          const float ov[8] = {o0.x, o0.y, o0.z, o0.w, o1.x, o1.y, o1.z, o1.w};
          float g[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) g[e] = ov[e] * o_scale * sigmoid_hw_f32(gate[8 * hf + e], att_unscale);
          gated.store8(mid.l32, 4 * ot + 2 * mid.lh + hf, g);
        }
      }
      __syncthreads();
      if (kh > 0) {
        f32x16_t acc = product(gated);
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[v] *= att_unscale;
        const Lane mid = lane_here();
        float* row = rows + mid.l32 * (C + kRowLd) + 32 * ot + 16 * mid.lh;
        store_row16(row, row, acc, 1);
      }
      __syncthreads();
#pragma unroll
      for (int e = 0; e < C / 64; ++e) raw[0][0].v[e] = *reinterpret_cast<const float4*>(rows + pos * (C + kRowLd) + 64 * e + 4 * here.li);
    }
    {
      const Lane here = lane_here();
#pragma unroll
      for (int t = 0; t < NPT; ++t) {
        int j0;
        const int pn = NPT * tile + t;
        row_of(pn, j0);
        const XTile xn = {lds + t * XTile::SLOTS};
#pragma unroll
        for (int g = 0; g < RG; ++g) {
          const int pos = 4 * (NW * g + wave) + here.lg;
          float4 y[C / 64];
          norm_row<C>(raw[t][g], ln, here.li, y);
#pragma unroll
          for (int e = 0; e < C / 64; ++e) xn.store4(pos, here.li + 16 * e, y[e]);
        }
      }
    }
    // this wave's rows of the result, of one position tile or of all
    struct Rows {
      int r, bb, i, j0;
      int64_t row0;
    };
    auto rows_of = [&](int o) {
      const int pn = NPT * tile + pt_b + o;
      Rows w;
      w.r = row_of(pn < p.total ? pn : p.total - 1, w.j0), w.bb = w.r / p.R, w.i = w.r - w.bb * p.R;
      w.row0 = w.bb * p.xv.stride_b + w.i * p.xv.stride_r + (int64_t)w.j0 * p.xv.stride_k;
      return w;
    };
    Row16 res[OP];
    float m[OP];
    auto global_rows = [&](const Rows& w) { return GlobalRows(p.x, p.out, AFTER ? 0 : w.row0, p.add_residual && kh == 0); };
    auto offset_of = [&](int o, const Rows& w) {
      return global_rows(w).offset(w.j0, NPT * tile + pt_b + o < p.total && kh == 0 ? L : 0, p.xv.stride_k, 32 * ot);
    };
    // before the next tile's rows, so that a wait for these leaves those in flight
    auto load_residual = [&] {
#pragma unroll
      for (int o = 0; o < OP; ++o) {
        const Rows w = rows_of(o);
        const int j = w.j0 + lane_here().l32 < L ? w.j0 + lane_here().l32 : L - 1;
        m[o] = p.mask ? p.mask[w.bb * p.mv.stride_b + w.i * p.mv.stride_r + (int64_t)j * p.mv.stride_k] : 1.f;
        if (!AFTER) res[o] = global_rows(w).load(offset_of(o, w));
      }
    };
    if constexpr (!KEEP) {
#pragma unroll
      for (int s = 0; s < DA; ++s) fetch_ab(0, s);
    }
    HalfSum<128, true> osum[OP];
    for (int slice = 0; slice < slices; ++slice) {
      // requested ahead of the operands (where the registers allow it): behind them they wait for every operand in flight
      float ua = kept_a, ub = kept_b;
      if (!KEEP && kEarly) scales_of(slice, ua, ub);
      __syncthreads();  // the activations (first slice), or: everybody has read the slice before
      f32x16_t a[XT], b[XT];
      HalfSum<C, true> sum_a[XT], sum_b[XT];
      {
        const Lane at = lane_here();
        u32x4_t nx[XT][2];
        auto read_x = [&](int s) {
#pragma unroll
          for (int t = 0; t < XT; ++t) {
            const u32x4_t* x = lds + (pt_a + t) * XTile::SLOTS + XTile::slot(at.l32, 2 * s + at.lh);
            nx[t][0] = x[0], nx[t][1] = x[XTile::PLANE];
          }
        };
        read_x(0);
#pragma unroll
        for (int s = 0; s < KS; ++s) {
          u32x4_t x[XT][2], ca[2], cb[2];
#pragma unroll
          for (int pl = 0; pl < 2; ++pl) {
            ca[pl] = na[s % DA][pl], cb[pl] = nb[s % DA][pl];
#pragma unroll
            for (int t = 0; t < XT; ++t) x[t][pl] = nx[t][pl];
          }
          if (s + 1 < KS) read_x(s + 1);
          if (s + DA < KS) fetch_ab(slice, s + DA);
          if (!KEEP && kEarly && s + 1 == KS) {
#pragma unroll
            for (int q = 0; q < DO; ++q) fetch_o(slice, q);
          }
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int term = 0; term < 3; ++term) {  // chains of dependent products in turn (211 / 207.5 us at N = 384)
#pragma unroll
            for (int t = 0; t < XT; ++t) sum_a[t].term(term, ca, x[t]), sum_b[t].term(term, cb, x[t]);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int t = 0; t < XT; ++t) a[t] = sum_a[t].total(), b[t] = sum_b[t].total();
      }
      if (!kEarly) {
        scales_of(slice, ua, ub);
#pragma unroll
        for (int q = 0; q < DO; ++q) fetch_o(slice, q);
      }
      {
        const Lane at = lane_here();
#pragma unroll
        for (int t = 0; t < XT; ++t) {
          const HTile h = {hid + (pt_a + t) * HTile::SLOTS};
#pragma unroll
          for (int hf = 0; hf < 2; ++hf) {  // lane (position, half lh): hidden channels 32 ht + 16 lh + 8 hf + e
            float y[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) y[e] = (a[t][8 * hf + e] * sigmoid_hw_f32(a[t][8 * hf + e], ua)) * (b[t][8 * hf + e] * ub);
            h.store8(at.l32, 4 * ht + 2 * at.lh + hf, y);
          }
        }
      }
      __syncthreads();  // the slice's hidden activations are complete
      const bool last = slice + 1 == slices;
      {
        const Lane at = lane_here();
        const u32x4_t* ht0 = hid + pt_b * HTile::SLOTS;
        u32x4_t nx[OP][2];
        auto read_h = [&](int s) {
#pragma unroll
          for (int o = 0; o < OP; ++o) {
            const u32x4_t* x = ht0 + o * HTile::SLOTS + HTile::slot(at.l32, 2 * (kh * OSTEPS + s) + at.lh);
            nx[o][0] = x[0], nx[o][1] = x[HTile::PLANE];
          }
        };
        read_h(0);
#pragma unroll
        for (int s = 0; s < OSTEPS; ++s) {
          const u32x4_t co[2] = {no[s % DO][0], no[s % DO][1]};
          u32x4_t x[OP][2];
#pragma unroll
          for (int o = 0; o < OP; ++o) x[o][0] = nx[o][0], x[o][1] = nx[o][1];
          if (s + 1 < OSTEPS) read_h(s + 1);
          if (s + DO < OSTEPS) fetch_o(slice, s + DO);
          if (s + DO == OSTEPS) {  // after the last weights: loads return in order
            if (KEEP || last) {
              if (kEarlyRes) load_residual();
              if (!AFTER) load_tile(tile + (int)gridDim.x < tiles ? tile + gridDim.x : tile);
            } else
#pragma unroll
              for (int q = 0; q < DA; ++q) fetch_ab(slice + 1, q);
          }
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int term = 0; term < 3; ++term) {
#pragma unroll
            for (int o = 0; o < OP; ++o) osum[o].term(term, co, x[o]);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
    if (!kEarlyRes) load_residual();
    if constexpr (OP > 1) {
#pragma unroll
      for (int o = 0; o < OP; ++o) {
        const Rows w = rows_of(o);
        f32x16_t v = osum[o].total();
#pragma unroll
        for (int e = 0; e < 16; ++e) v[e] *= so.total;
        if (p.mask) {
#pragma unroll
          for (int e = 0; e < 16; ++e) v[e] *= m[o];
        }
        global_rows(w).store(offset_of(o, w), v, res[o]);
      }
      continue;
    }
    f32x16_t oacc = osum[0].total();
    const Rows w = rows_of(0);
    const int j0 = w.j0, i = w.i, bb = w.bb;
    const Lane at = lane_here();
    if (KSPLIT > 1) {  // the waves of an output tile add up through the hidden tile's memory
      __syncthreads();
      float* red = reinterpret_cast<float*>(hid) + (wave % (OT * NPT)) * 1024 + at.l32 + 32 * at.lh;
      if (kh > 0) {
#pragma unroll
        for (int v = 0; v < 16; ++v) red[(kh - 1) * (OT * NPT * 1024) + 64 * v] = oacc[v];
      }
      __syncthreads();
      if (AFTER && !BIAS && kh > 0) return;
      if (!BIAS && !KEEP && kh > 0) continue;  // KEEP: what these waves store is past the end of their buffers
      if (!BIAS || kh == 0) {
#pragma unroll
        for (int q = 0; q < KSPLIT - 1; ++q)
#pragma unroll
          for (int v = 0; v < 16; ++v) oacc[v] += red[q * (OT * NPT * 1024) + 64 * v];
      }
    }
#pragma unroll
    for (int v = 0; v < 16; ++v) oacc[v] *= so.total;
    const int j = j0 + at.l32;
    if (p.mask) {
#pragma unroll
      for (int v = 0; v < 16; ++v) oacc[v] *= m[0];
    }
    if constexpr (BIAS) {
      float* row = rows + at.l32 * (C + kRowLd) + 32 * ot + 16 * at.lh;
      if (kh == 0) {
        store_row16(row, row, oacc, 1);
        if (j < L) {
          float4* dst = reinterpret_cast<float4*>(p.out + bb * p.xv.stride_b + i * p.xv.stride_r + (int64_t)j * p.xv.stride_k + 32 * ot + 16 * at.lh);
#pragma unroll
          for (int a = 0; a < 4; ++a) dst[a] = *reinterpret_cast<const float4*>(row + 4 * a);
        }
      }
      for (int c = tid; c < C; c += 64 * NW) att_ln[c] = p.pb_ln_w[c], att_ln[C + c] = p.pb_ln_b ? p.pb_ln_b[c] : 0.f;
      constexpr int SPW = KS / 4;  // four waves share the sum over the channels
      u32x4_t wp[SPW][3];
      if (wave < 4) {
        const int head = at.l32 < p.pb_H ? at.l32 : p.pb_H - 1;  // the rows from H on are dropped
#pragma unroll
        for (int s = 0; s < SPW; ++s) split_operand(p.pb_w + (size_t)head * C, SPW * wave + s, at.lh, wp[s]);
      }
      __syncthreads();  // the rows are complete, and everybody has read the partial sums
      const PassTile<C> xn = {reinterpret_cast<u32x4_t*>(rows + 32 * (C + kRowLd))};
      {
        const Lane here = lane_here();
        const int pos = 4 * wave + here.lg;
        float4 y[C / 64];
#pragma unroll
        for (int e = 0; e < C / 64; ++e) raw[0][0].v[e] = *reinterpret_cast<const float4*>(rows + pos * (C + kRowLd) + 64 * e + 4 * here.li);
        norm_row<C>(raw[0][0], att_ln, here.li, y);
#pragma unroll
        for (int e = 0; e < C / 64; ++e) xn.store4(pos, here.li + 16 * e, y[e]);
      }
      __syncthreads();
      float* part = reinterpret_cast<float*>(hid);  // [4][32 heads][kBiasLd]
      if (wave < 4) {
        f32x16_t acc = zero16();
#pragma unroll
        for (int s = 0; s < SPW; ++s) {
          const u32x4_t* x = xn.s + PassTile<C>::slot(at.l32, 2 * (SPW * wave + s) + at.lh);
          const u32x4_t op[3] = {x[0], x[PassTile<C>::PLANE], x[2 * PassTile<C>::PLANE]};
          acc = step6<true>(wp[s], op, acc);
        }
        float* mine = part + wave * (32 * kBiasLd) + at.l32;
#pragma unroll
        for (int v = 0; v < 16; ++v)
          if (8 * (v >> 2) < p.pb_H) mine[acc_row(v, at.lh) * kBiasLd] = acc[v];
      }
      __syncthreads();
      for (int h = tid >> 5; h < p.pb_H; h += 2 * NW) {
        const float* q = part + h * kBiasLd + (tid & 31);
        const float v = (q[0] + q[32 * kBiasLd]) + (q[2 * 32 * kBiasLd] + q[3 * 32 * kBiasLd]);
        const int f = j0 + (tid & 31);
        if (f < L) p.pb_out[((size_t)bb * p.pb_H + h) * L + f] = v;
      }
      return;
    }
    if constexpr (AFTER) {
      if (j < L) store_row16(rows + at.l32 * (C + kRowLd) + 32 * ot + 16 * at.lh, p.out + w.row0 + (int64_t)at.l32 * p.xv.stride_k + 32 * ot + 16 * at.lh, oacc, p.add_residual);
      return;
    } else {
      global_rows(w).store(offset_of(0, w), oacc, res[0]);
    }
  }
}

template <int C, int S, int NPT, bool AFTER = false, bool BIAS = false, bool KEEP = false, int NW = 8>
hipError_t launch(const TransitionPass& p, hipStream_t stream) {
  constexpr size_t lds = transition_lds<C, S, NPT, AFTER, BIAS>();
  unsigned grid = 0;
  hipError_t e = resident_grid<transition_pass<C, S, NPT, AFTER, BIAS, KEEP, NW>>(64 * NW, lds, (p.total + NPT - 1) / NPT, &grid);
  if (e != hipSuccess) return e;
  if (AFTER) grid = (unsigned)p.total;  // a tile each
  hipLaunchKernelGGL((transition_pass<C, S, NPT, AFTER, BIAS, KEEP, NW>), dim3(grid), dim3(64 * NW), lds, stream, p);
  return hipGetLastError();
}

hipError_t device_cus(int* cus) {
  static int cache[kMaxDevices];
  return per_device(cache, [](int dev, int* v) { return cu_count(dev, v); }, cus);
}
bool flat_rows(const TransitionF32Args& a) {
  return a.x_view.stride_r == a.N * a.x_view.stride_k && (!a.mask || a.mask_view.stride_r == a.N * a.mask_view.stride_k);
}

}  // namespace

bool transition_pass_serves(const TransitionF32Args& a) {
  return transition_half_shapes(a.B, a.N, a.C, a.HID) && rows_aligned(a.x, a.x_view) && rows_aligned(a.out, a.x_view);
}

// Wherever the transition by itself takes tiles of 32 positions (below four per CU).  Saves the launches, z's way to memory and back and the wait for
// the first tile: with the attention's output pass and the pair bias apart / in one, four trunk blocks at N = 64 / 80 / 90 / 128 / 180
// 597 / 705 / 780 / 1009 / 1913 us, so 565 / 671 / 736 / 977 / 1875, two at 140 744 / 728.
bool transition_pass_takes(const TransitionF32Args& a) {
  int cus = 0;
  return device_cus(&cus) == hipSuccess && a.C == 128 && a.HID % 256 == 0 && flat_rows(a) && a.end->C == 128 && a.end->s_o.terms == 2 && a.end->N == a.N &&
         a.end->B == a.B && a.end->add_residual && a.end->out == a.x && a.x == a.out && a.add_residual &&
         (long)a.B * (((long)a.N * a.N + 31) / 32) < 4l * cus;
}

hipError_t transition_pass_f32(const TransitionF32Args& a, const WeightX3& s_a, const WeightX3& s_b, const WeightX3& s_out,
                               hipStream_t stream) {
  TransitionPass p;
  p.x = a.x;
  p.mask = a.mask;
  p.xv = a.x_view;
  p.mv = a.mask_view;
  p.ln_w = a.ln_w;
  p.ln_b = a.ln_b;
  p.s_a = s_a;
  p.s_b = s_b;
  p.s_out = s_out;
  p.out = a.out;
  // a tensor (and mask) whose rows follow one another without gaps is one row of N * N positions
  const bool flat = flat_rows(a);
  p.R = flat ? 1 : a.N;
  p.L = flat ? a.N * a.N : a.N;
  p.panels = (p.L + 31) / 32;
  p.total = a.B * p.R * p.panels;
  p.HID = a.HID;
  p.add_residual = a.add_residual;
  int cus = 0;
  const hipError_t e = device_cus(&cus);
  if (e != hipSuccess) return e;
  if (a.end) {  // transition_pass_takes
    p.att_o = a.end->o;
    p.att_ln_w = a.end->ln_w;
    p.att_ln_b = a.end->ln_b;
    p.att_g = a.end->s_g;
    p.att_out = a.end->s_o;
    p.N = a.N;
    if (a.bias && pair_bias_pass_serves(*a.bias) && a.bias->C == 128 && a.bias->N == a.N && a.bias->B == a.B) {
      p.pb_w = a.bias->w;
      p.pb_ln_w = a.bias->ln_w;
      p.pb_ln_b = a.bias->ln_b;
      p.pb_out = a.bias->out;
      p.pb_H = a.bias->H;
      *a.bias_done = true;
      return launch<128, 8, 1, true, true>(p, stream);
    }
    return launch<128, 8, 1, true>(p, stream);
  }
  const bool large = p.total >= 4l * cus;  // two tiles of 64 positions for every CU
  if (a.HID % 256 != 0) {
    if (a.C == 128) return launch<128, 4, 2>(p, stream);
    return a.HID == 128 ? launch<64, 4, 1, false, false, true, 4>(p, stream) : launch<64, 4, 2>(p, stream);
  }
  if (a.C == 128) return large ? launch<128, 4, 2, false, false, false, 4>(p, stream) : launch<128, 8, 1>(p, stream);
  return large ? launch<64, 8, 2>(p, stream) : launch<64, 8, 1>(p, stream);
}

}  // namespace of3
