// fp32 triangle-attention core (attention.py:94-135 with the two biases of tri_att.py:134-140) on two fp16 terms
// (of3_split.h), head width 16 * STEPS (32 or 16), for the shapes whose projection pass delivers them
// (pair_pass_f32.hip); pair_f32.hip has the cores for every other shape.
//
// Work-group = 4 waves = 2 consecutive rows i x 2 halves of one (head, 128-query range), or 4 rows x one of 64 queries; a wave owns 64
// queries (two 32-query tiles) of one row.  Three work-groups share a CU (heads of 16: four), so that the products of one run under the exponentials and
// splits of the others.  Bound by matrix and vector time at the clock that both leave (N = 768, heads of 32: 901 us a launch, matrix
// pipe 48 %, vector pipe 63 %, 1.67 GHz; three bf16 terms 1446; heads of 16, three templates of 200: 54 us, 22 and 59 %; 88).
// A 32 x 32 tile is 98 vector instructions, 80 of them 16 each of exponentials, fused multiply-adds and additions and 32 of the splits (169 ns on a SIMD
// alone), the rest the loop's own, and 12 products (180, 300 with all CUs busy).
//   S^T = K Q^T  (rows = keys, columns = queries), three products per k-step, started from the triangle bias (the
//                accumulator is loaded with it).  Logits are in natural units times the scales of q and k, a power of
//                two that the bias and the mask bias carry too, and not pre-multiplied by log2(e): a row of masked keys
//                has to lose its logits against -1e9 at the reference's granularity, or it averages other keys than the
//                reference does.  The mask bias of a key tile rides on one more k-step, A = [hi, mid, lo, 0 ...] of the
//                key's bias split exactly into three bf16 terms, B = [1, 1, 1, 0 ...], taken only by tiles with a masked
//                or padded key
//   O^T = V^T P^T, the weights split in registers straight from the S^T accumulator into B operands, three products.
//                Width 16: the operand's free rows hold V^T's second terms, [vh; vl] p, added at the end: two products,
//                all four of the terms.
// Per 32-key tile the work-group brings in the bias slice of its query range (it does not depend on i: shared by its
// rows) and each row's K and V^T operands (shared by the row's waves) with direct-to-LDS buffer loads, one tile
// ahead, the bias into double buffers: no registers are held for data in flight, and the only wait for
// loads is one vmcnt(0) + barrier per key tile, a whole tile of arithmetic after they were issued.  The operands have one place, which (two
// waves to a row) a second barrier frees once they are in registers: with two, one work-group fewer fits (width 32, three / two, N = 768: 4596 / 4744 us a pass;
// width 16, four / three, us a launch: three templates of 150 34.2 / 36.4, of 250 83.8 / 88.0, two of 384 174 / 185, one of 150 16.9 / 16.6).
// The bias slice is XOR-swizzled on the global side (a lane picks which 16-byte chunk it fetches for its fixed LDS slot).
//
// Softmax weights as fp16 terms have to lie between 2^-13 (below it their second terms lose bits) and 2^16.  The first
// pass takes as a query's offset the largest logit of the first key tile that has an unmasked key, and lifts the weights by 2^kLift
// (any common offset gives the same softmax), so that a row sum is at least 2^kLift; a weight above 2^kHigh halves all that
// the query has summed as often as brings it down to 2^kLift (exact, and rare: the logit exceeds the first tile's largest by 8
// in natural units).  Key tiles whose keys are all masked or padded are left out; a row without any unmasked key ends with the sum 0, and
// its work-group runs the second pass, with running maxima.  Keys past N carry a mask bias of -inf.
#include <type_traits>

#include "of3_device.h"
#include "of3_launch.h"
#include "of3_pair_f32.h"
#include "of3_split.h"

namespace of3 {

namespace {

constexpr int kWaves = 4;
template <int STEPS>
constexpr int kPerCu = STEPS == 2 ? 3 : 4;  // work-groups
constexpr float kLift = 4.f, kHigh = 0x1p15f;
constexpr float kFloor = -3e38f;  // in place of -infinity as an offset
enum { kFirst, kTracked, kLevelled };  // what a pass over the keys does
template <int STEPS, int QW>
struct CoreH2 {
  static constexpr int kRows = kWaves / QW;
  static constexpr int kQueries = 64 * QW;
  static constexpr int kTb = kQueries * 8;           // bias slice [queries][32 keys] fp32 in 16-byte slots
  static constexpr int kTbI = kTb / (64 * kWaves);   // load instructions of a wave for it
  static constexpr int kKv = 2 * STEPS * 64;    // K (steps x terms), and as many of V^T (two steps x terms, or x 1 at width 16)
  static constexpr size_t kLds = (size_t)(2 * kTb + kRows * 2 * kKv) * 16;
};

// QW: waves of a row, 1 or 2 (kWaves / QW rows, 64 QW queries)
template <int STEPS, int QW>
__global__ __launch_bounds__(64 * kWaves, kPerCu<STEPS>) void triattn_core_h2_f32(TriattnF32 p, int n_qc, int n_rg, int total, int per_xcd) {
  typedef CoreH2<STEPS, QW> L;
  constexpr int kRows = L::kRows, kQueries = L::kQueries, kTb = L::kTb, kTbI = L::kTbI;
  constexpr int QT = 2, D = 16 * STEPS;
  extern __shared__ u32x4_t lds4[];
  u32x4_t* tb_lds = lds4;                 // [2][kTb]
  u32x4_t* kv_lds = lds4 + 2 * kTb;    // [kRows][K, V^T]
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int row = wave / QW, qh = wave % QW;
  const int lane = tid & 63, l32 = lane & 31, lh = lane >> 5;
  const int N = p.N, H = p.H, Jp = p.Jp, nt = Jp / 32;
  const int logical = xcd_logical_block(blockIdx.x, per_xcd);
  if (logical >= total) return;  // the whole work-group leaves together
  const int qc = logical % n_qc, rg = (logical / n_qc) % n_rg, bh = logical / (n_qc * n_rg);
  const int i_raw = rg * kRows + row;
  const bool row_valid = i_raw < N;  // wave-uniform; idle waves still take part in the loads and barriers
  const int i = row_valid ? i_raw : N - 1;
  const int b = bh / H, h = bh % H;
  const int q0 = qc * kQueries + 64 * qh;
  const size_t bih = ((size_t)b * N + i) * H + h;
  const long plane = p.qk_plane / 8;  // in 16-byte slots
  const u32x4_t* Q = reinterpret_cast<const u32x4_t*>(p.qs) + bih * nt * (64 * STEPS) + lane;
  const float* tbp = p.tb + ((size_t)b * H + h) * N * Jp;  // rows padded to Jp, zeros past N
  const int nkt = nt;

  // four keys of every row of the work-group (lane 4 r + c: key c of row r), read before anything else: below
  float sample = 0.f;
  {
    const int r = rg * kRows + ((lane >> 2) & (kRows - 1)), c = lane & 3;
    const int key = c == 0 ? r : c == 1 ? 0 : c == 2 ? N >> 1 : N - 1;
    if (p.mask && r < N) sample = p.inf * (p.mask[b * p.mv.stride_b + r * p.mv.stride_r + key * p.mv.stride_k] - 1.f);
  }
  const int wt = h * D / 32;  // the head's tile of 32 rows of its weights
  const float logit_scale = p.s_q.scales()[wt].output * p.s_k.scales()[wt].output;
  const float to_exp2 = 1.4426950408889634f / logit_scale;

  u32x4_t qop[QT][STEPS][2];
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    const int jt = q0 / 32 + qt < nt ? q0 / 32 + qt : nt - 1;  // tiles past the end: computed, not stored
#pragma unroll
    for (int st = 0; st < STEPS; ++st)
#pragma unroll
      for (int pl = 0; pl < 2; ++pl) qop[qt][st][pl] = Q[pl * plane + (jt * STEPS + st) * 64];
  }

  // bias slice: instruction n of wave w fills slots 64 (kTbI w + n) .. + 63; slot t holds chunk
  // (t & 7) ^ ((q >> 1) & 7) of query q = t >> 3 of the work-group's range
  uint32_t tb_off[4];  // kTbI of them: with the dependent size clang leaves the kernel out of the host code
  static_assert(kTbI <= 4, "");
#pragma unroll
  for (int n = 0; n < kTbI; ++n) {
    const int t = 64 * (kTbI * wave + n) + lane;
    const int qloc = t >> 3, chunk = (t & 7) ^ ((qloc >> 1) & 7);
    int qrow = qc * kQueries + qloc;
    qrow = qrow < N ? qrow : N - 1;
    tb_off[n] = (uint32_t)(((size_t)qrow * Jp + 4 * chunk) * sizeof(float));
  }
  // This wave's share of its row's tile: the K operands (first wave of the row) or the V^T operands, 2 STEPS instructions of
  // 1 KB, or (QW = 1) both.  Width 32: step n / 2, term n % 2, a descriptor per term (a plane can be larger than a descriptor's range);
  // width 16: the term n of K's step, or the step n of V^T's plane, which begins 1 KB further on
  const bool is_v = QW == 2 && qh;  // what its first 2 STEPS instructions bring
  const long kv_plane = STEPS == 2 ? (is_v ? p.v_plane : p.qk_plane) : (is_v ? 512 : p.qk_plane);
  const int kv_tile = STEPS == 2 || is_v ? 2048 : 1024;  // bytes of a key tile in a plane
  const bf16_t* kvp = (is_v ? p.vs : p.ks) + bih * nt * (kv_tile / 2);
  const size_t kv_bytes = (size_t)nt * kv_tile;
  const __amdgpu_buffer_rsrc_t kv_rsrc[2] = {buffer_rsrc(kvp, kv_bytes),
                                             buffer_rsrc(kvp + kv_plane, STEPS == 1 && is_v ? kv_bytes - 1024 : kv_bytes)};
  const bf16_t* vp = p.vs + bih * nt * 1024;
  const long v_plane = STEPS == 2 ? p.v_plane : 512;
  const __amdgpu_buffer_rsrc_t v_rsrc[2] = {buffer_rsrc(vp, (size_t)nt * 2048),  // QW = 1
                                            buffer_rsrc(vp + v_plane, (size_t)nt * 2048 - (STEPS == 1 ? 1024 : 0))};
  const __amdgpu_buffer_rsrc_t tb_rsrc = buffer_rsrc(tbp, (size_t)N * Jp * sizeof(float));
  const uint32_t lane_off = lane * 16;
  u32x4_t* kv_row = kv_lds + row * (2 * L::kKv);
  auto issue_bias = [&](int kt, int buf) {  // buf is a constant at every call site
    u32x4_t* tdst = tb_lds + buf * kTb + 64 * kTbI * wave;
#pragma unroll
    for (int n = 0; n < kTbI; ++n)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(tb_rsrc, (void OF3_LDS_AS*)(tdst + 64 * n), 16, tb_off[n],
                                               kt * (32 * (int)sizeof(float)), 0, 0);
  };
  auto issue_kv = [&](int kt) {
    u32x4_t* kdst = kv_row + qh * L::kKv;
#pragma unroll
    for (int n = 0; n < 2 * STEPS; ++n)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(kv_rsrc[n & 1], (void OF3_LDS_AS*)(kdst + 64 * n), 16, lane_off,
                                               kt * kv_tile + (n >> 1) * 1024, 0, 0);
    if (QW == 1) {
#pragma unroll
      for (int n = 0; n < 2 * STEPS; ++n)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(v_rsrc[n & 1], (void OF3_LDS_AS*)(kdst + L::kKv + 64 * n), 16, lane_off,
                                                 kt * 2048 + (n >> 1) * 1024, 0, 0);
    }
  };
  // mask value of key 32 kt + l32 (clamped to a real key; some bias value when there is no mask: not used)
  const float* mrow = p.mask ? p.mask + b * p.mv.stride_b + i * p.mv.stride_r : tbp;
  const long mstep = p.mask ? p.mv.stride_k : 1;
  auto load_mask = [&](int kt) {
    const int k = kt * 32 + l32 < N ? kt * 32 + l32 : N - 1;
    return mrow[k * mstep];
  };
  auto mask_bias = [&](int kt, float mv) {
    return kt * 32 + l32 < N ? (p.mask ? even_bias(p.inf * (mv - 1.f)) : 0.f) : -__builtin_inff();
  };
  // the mask-bias k-step on the 8-deep MFMA (two registers per operand): lanes 0..31 hold k = 0..3
  auto mask_step = [&](float mb, f32x16_t acc) {
    const bool lo = lh == 0;
    const uint32_t hi_bits = __float_as_uint(mb) & 0xffff0000u;
    const float r1 = __builtin_isinf(mb) ? 0.f : mb - __uint_as_float(hi_bits);  // exact
    const uint32_t mid_bits = __float_as_uint(r1) & 0xffff0000u;
    const float r2 = r1 - __uint_as_float(mid_bits);  // exact, at most 8 significant bits
    const u32x2_t a_op = {lo ? ((hi_bits >> 16) | mid_bits) : 0u, lo ? (__float_as_uint(r2) >> 16) : 0u};
    const u32x2_t b_op = {lo ? 0x3F803F80u : 0u, lo ? 0x3F80u : 0u};
    return mfma_32x32x8(a_op, b_op, acc);
  };

  f32x16_t oacc[QT];
  float m_run[QT], l_run[QT], l_tot[QT];  // m_run: first pass, what is subtracted before exp2; second, the largest logit
  bool fresh = true;                      // first pass: no offset yet
  const int tb_key = (l32 >> 1) & 7;

  // a wave of a row past the end, or whose queries all lie past the end, still takes part in the loads and
  // barriers of its work-group but leaves the arithmetic out; so does a 32-query tile past the end
  const bool wave_has_work = row_valid && q0 < N;
  auto largest = [&](const f32x16_t& s) {  // of the query's 32 keys
    float m = s[0];
#pragma unroll
    for (int v = 1; v < 16; ++v) m = fmaxf(m, s[v]);
    return fmaxf(m, __shfl_xor(m, 32, 64));
  };
  struct Operands {
    u32x4_t k[STEPS][2], v[2][STEPS];
  };
  auto read_operands = [&]() {
    const u32x4_t* kvb = kv_row + lane;
    Operands o;
#pragma unroll
    for (int st = 0; st < STEPS; ++st)
#pragma unroll
      for (int pl = 0; pl < 2; ++pl) o.k[st][pl] = kvb[(st * 2 + pl) * 64];
#pragma unroll
    for (int st = 0; st < 2; ++st)
#pragma unroll
      for (int pl = 0; pl < STEPS; ++pl) o.v[st][pl] = kvb[L::kKv + (st * STEPS + pl) * 64];
    return o;
  };
  uint32_t uneven[QT];  // level pass: bits in which a logit of the lane's query differed from level_at's
  uint32_t level_at = 0u;
  auto tile = [&](auto kind, int buf, float mb, const Operands& op, int keys_left) {
    constexpr bool kTrack = decltype(kind)::value == kTracked, kLevel = decltype(kind)::value == kLevelled;
    if (!wave_has_work) return;
    // first pass: a tile whose keys are all masked or padded adds exp(-1e9 + logit) = 0 exactly to every sum
    if (!kTrack && !kLevel && __builtin_amdgcn_ballot_w64(mb > -1e8f) == 0) return;
    const bool has_mb = __builtin_amdgcn_ballot_w64(mb != 0.f) != 0;
    const u32x4_t* tbuf = tb_lds + buf * kTb + (64 * qh + l32) * 8;
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      if (qt > 0 && q0 + 32 * qt >= N) continue;
      f32x16_t s;
#pragma unroll
      for (int a = 0; a < 4; ++a) {  // registers 4 a .. 4 a + 3: keys 8 a + 4 lh .. + 3 = chunk 2 a + lh
        const u32x4_t t = tbuf[qt * 256 + ((2 * a + lh) ^ tb_key)];
#pragma unroll
        for (int e = 0; e < 4; ++e) s[4 * a + e] = __uint_as_float(t[e]);
      }
      if (has_mb) s = mask_step(mb * logit_scale, s);
#pragma unroll
      for (int st = 0; st < STEPS; ++st) {  // smallest terms first
        s = mfma_32x32x16_f16(op.k[st][1], qop[qt][st][0], s);
        s = mfma_32x32x16_f16(op.k[st][0], qop[qt][st][1], s);
        s = mfma_32x32x16_f16(op.k[st][0], qop[qt][st][0], s);
      }
      if constexpr (kLevel) {
        // register v holds key 8 (v >> 2) + 4 lh + (v & 3) of the tile, and so do the weights' operands: all 2^kLift, of keys below N
        constexpr uint32_t kOne = 0x4C00u;
        static_assert(kLift == 4.f, "fp16(16)");
        const int left = keys_left - 4 * lh;
        if (keys_left >= 32) {
#pragma unroll
          for (int v = 0; v < 16; ++v) uneven[qt] |= __float_as_uint(s[v]) ^ level_at;  // NaN too
        } else {
#pragma unroll
          for (int v = 0; v < 16; ++v) uneven[qt] |= acc_row(v, 0) < left ? __float_as_uint(s[v]) ^ level_at : 0u;
        }
        if (qt > 0) continue;
#pragma unroll
        for (int st = 0; st < 2; ++st) {
          u32x4_t ph;
#pragma unroll
          for (int w = 0; w < 4; ++w) ph[w] = (acc_row(8 * st + 2 * w, 0) < left ? kOne : 0u) | (acc_row(8 * st + 2 * w + 1, 0) < left ? kOne << 16 : 0u);
          if constexpr (STEPS == 2) oacc[0] = mfma_32x32x16_f16(op.v[st][STEPS - 1], ph, oacc[0]);
          oacc[0] = mfma_32x32x16_f16(op.v[st][0], ph, oacc[0]);
        }
        continue;
      }
      float lsum = 0.f;
      if constexpr (kTrack) {
        const float m_new = fmaxf(m_run[qt], largest(s));
        const float alpha = __builtin_amdgcn_exp2f((m_run[qt] - m_new) * to_exp2);
        m_run[qt] = m_new;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          s[v] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[v] - m_new, to_exp2, kLift));
          lsum += s[v];
        }
        l_run[qt] = l_run[qt] * alpha + lsum;
#pragma unroll
        for (int v = 0; v < 16; ++v) oacc[qt][v] *= alpha;
      } else {
        if (fresh) m_run[qt] = fmaxf(largest(s) * to_exp2, kFloor) - kLift;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          s[v] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[v], to_exp2, -m_run[qt]));
          lsum += s[v];
        }
        if (__builtin_amdgcn_ballot_w64(lsum > kHigh) != 0) {
          const float top = fmaxf(lsum, __shfl_xor(lsum, 32, 64));  // both halves of the query's keys
          const int down = top > kHigh ? __builtin_amdgcn_frexp_expf(top) - (int)kLift : 0;
          m_run[qt] += (float)down;
          lsum = __builtin_ldexpf(lsum, -down);
          l_run[qt] = __builtin_ldexpf(l_run[qt], -down);
#pragma unroll
          for (int v = 0; v < 16; ++v) s[v] = __builtin_ldexpf(s[v], -down), oacc[qt][v] = __builtin_ldexpf(oacc[qt][v], -down);
        }
        l_run[qt] += lsum;
      }
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        float x[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = s[8 * st + e];
        u32x4_t ph, pl;
        split8h(x, ph, pl);
        if constexpr (STEPS == 1) {
          oacc[qt] = mfma_32x32x16_f16(op.v[st][0], pl, oacc[qt]);
          oacc[qt] = mfma_32x32x16_f16(op.v[st][0], ph, oacc[qt]);
        } else {
          oacc[qt] = mfma_32x32x16_f16(op.v[st][STEPS - 1], ph, oacc[qt]);
          oacc[qt] = mfma_32x32x16_f16(op.v[st][0], pl, oacc[qt]);
          oacc[qt] = mfma_32x32x16_f16(op.v[st][0], ph, oacc[qt]);
        }
      }
    }
    if (!kTrack && !kLevel) fresh = false;
  };

  float mv_next;
  auto first_loads = [&]() {
    mv_next = load_mask(0);
    issue_bias(0, 0);
    issue_kv(0);
  };
  auto pass = [&](auto kind) {
    constexpr bool kLevel = decltype(kind)::value == kLevelled;
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      oacc[qt] = zero16();
      m_run[qt] = kFloor;
      l_run[qt] = 0.f;
      uneven[qt] = 0u;
    }
    auto step = [&](int kt, int buf) {  // buf is a constant at both call sites: LDS addresses are immediates
      wait_vmcnt<0>();               // this wave's loads of tile kt (and its mask values) have landed ...
      __builtin_amdgcn_s_barrier();  // ... and everybody's; nobody reads tile kt - 1's buffers any more
      compiler_fence();
      const float mb = mask_bias(kt, mv_next);
      if (kLevel && kt == 0) level_at = __builtin_amdgcn_readfirstlane(__float_as_uint(mb * logit_scale));
      const int ktn = kt + 1 < nkt ? kt + 1 : nkt - 1;
      mv_next = load_mask(ktn);
      issue_bias(ktn, buf ^ 1);
      const Operands op = read_operands();
      wait_lds_reads();
      if (QW == 2) __builtin_amdgcn_s_barrier();  // both waves of the row hold the operands in registers: their place is free
      compiler_fence();
      issue_kv(ktn);
      tile(kind, buf, mb, op, N - 32 * kt);
      compiler_fence();
    };
    for (int kt = 0; kt < nkt; kt += 2) {
      step(kt, 0);
      if (kt + 1 < nkt) step(kt + 1, 1);
    }
    wait_vmcnt<0>();  // the loads issued past the end must not outlive the pass (or the work-group's LDS)
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      if (kLevel && qt > 0) oacc[qt] = oacc[0];
      l_tot[qt] = kLevel ? (float)N * 16.f : l_run[qt] + __shfl_xor(l_run[qt], 32, 64);
    }
  };

  // A work-group with a row whose sampled keys are all masked goes to the second pass at once, as in the bf16 core.
  first_loads();
  const uint64_t masked = __builtin_amdgcn_ballot_w64(sample < -1e8f);
  // Where all of its rows look so, a pass that sees whether all logits are the mask bias itself, which takes those of an ordinary size up: the
  // weights are then equal, their sum N and the result the mean of v, the same for every query (three templates of 200, 20 tokens padded, 868 / 858
  // us, a trunk block at 600, 100 padded, 3170 / 3114).
  bool again = false, level = true;  // the same in every wave of the work-group
#pragma unroll
  for (int r = 0; r < kRows; ++r) {
    const bool all = ((masked >> (4 * r)) & 15u) == 15u;
    again |= all;
    level &= all || rg * kRows + r >= N;
  }
  level &= again;
  auto any_wave = [&](bool bad) {  // the vote goes through the bias buffers
    uint32_t* votes = reinterpret_cast<uint32_t*>(lds4);
    __syncthreads();
    const uint32_t wave_bad = __builtin_amdgcn_ballot_w64(bad) != 0;
    if (lane == 0) votes[wave] = wave_bad;
    __syncthreads();
    uint32_t any = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) any |= votes[w];
    const bool result = __builtin_amdgcn_readfirstlane(any) != 0;
    if (result) {
      __syncthreads();  // every wave has read the votes before loads land on them
      first_loads();
    }
    return result;
  };
  if (level) {
    pass(std::integral_constant<int, kLevelled>{});
    bool bad = false;
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) bad |= row_valid && q0 + 32 * qt + l32 < N && uneven[qt] != 0;
    again = any_wave(bad);
  } else if (!again) {
    pass(std::integral_constant<int, kFirst>{});
    bool bad = false;
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      const bool in_range = l_tot[qt] > 0.f && l_tot[qt] <= 0x1p60f;  // false for NaN and +inf (a logit 80 above the first tile's) too
      bad |= row_valid && (q0 + 32 * qt + l32 < N) && !in_range;
    }
    again = any_wave(bad);
  }
  if (again) pass(std::integral_constant<int, kTracked>{});

  if (row_valid) {
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      const int q = q0 + 32 * qt + l32;
      if (q >= N) continue;
      const float inv = 1.0f / l_tot[qt];  // o keeps the scales of v's channels, w_o has their inverses
      if constexpr (STEPS == 1) {
#pragma unroll
        for (int v = 0; v < 8; ++v) oacc[qt][v] += oacc[qt][v + 8];
      }
      float* dst = p.o + ((((size_t)b * N + i) * N + q) * H + h) * D + 4 * lh;
#pragma unroll
      for (int a = 0; a < D / 8; ++a)  // registers 4 a .. 4 a + 3 are head channels 8 a + 4 lh .. + 3
        *reinterpret_cast<float4*>(dst + 8 * a) = make_float4(oacc[qt][4 * a] * inv, oacc[qt][4 * a + 1] * inv,
                                                              oacc[qt][4 * a + 2] * inv, oacc[qt][4 * a + 3] * inv);
    }
  }
}

template <int STEPS, int QW>
hipError_t launch(const TriattnF32& p, hipStream_t stream) {
  typedef CoreH2<STEPS, QW> L;
  const hipError_t e = allow_dynamic_lds<triattn_core_h2_f32<STEPS, QW>>(L::kLds);
  if (e != hipSuccess) return e;
  const int n_qc = (p.N + L::kQueries - 1) / L::kQueries, n_rg = (p.N + L::kRows - 1) / L::kRows;
  const long total = (long)n_qc * n_rg * p.B * p.H;
  if (total > 0x7fffffffL - 8) return hipErrorInvalidValue;
  const int per_xcd = (int)((total + 7) / 8);
  hipLaunchKernelGGL((triattn_core_h2_f32<STEPS, QW>), dim3(per_xcd * 8), dim3(64 * kWaves), L::kLds, stream, p, n_qc, n_rg, (int)total, per_xcd);
  return hipGetLastError();
}

}  // namespace

hipError_t triattn_core_h2_f32_launch(const TriattnF32& p, hipStream_t stream) {
  // 64 queries of four rows instead of 128 of two, with one barrier a key tile less and twice the K and V^T through LDS, where the last range of
  // 128 would be at most half full.  us a launch, 64 / 128: heads of 16, templates 1 x 140 13.7 / 16.6, 2 x 187 30.6 / 34.1, 4 x 300 190 / 205, 1 x 400 109
  // / 119; others level (2 x 384 171.5 / 170.5, a pass of 3 x 200 874 / 870).  Heads of 32, whose K and V^T are twice as long: N = 300 80 / 87, 400
  // 177 / 184; others slower (128 12.6 / 12.3, 384 147 / 141, 768 931 / 891); and where 128 leave no second round only if the last of those is a quarter
  // (150 18.7 / 21.4; 180 27.0 / 26.2).  Beyond 512 tokens the unused half is at most a tenth of a launch, which the second reading of K and V^T costs: whole pair
  // stacks 64 / 128, us, 300 578 / 587, 390 1044 / 1053, 430 1233 / 1253, 448 1298 / 1304, but 520 1946 / 1929, 550 2202 / 2183, 576 2286 / 2293, 660 3244 / 3257.
  static int cache[kMaxDevices];
  int cus = 0;
  const hipError_t e = per_device(cache, [](int dev, int* v) { return cu_count(dev, v); }, &cus);
  if (e != hipSuccess) return e;
  typedef CoreH2<2, 2> Wide;
  const int last = p.N > Wide::kQueries ? p.N % Wide::kQueries : 0;
  if (p.D == 16) return last > 0 && last <= 64 ? launch<1, 1>(p, stream) : launch<1, 2>(p, stream);
  const long wide = (long)((p.N + Wide::kQueries - 1) / Wide::kQueries) * ((p.N + Wide::kRows - 1) / Wide::kRows) * p.B * p.H;
  const bool narrow = p.N <= 512 && last > 0 && last <= (wide > (long)kPerCu<2> * cus ? 64 : 32);
  return narrow ? launch<2, 1>(p, stream) : launch<2, 2>(p, stream);
}

}  // namespace of3
