// C-ABI layer of libof3pair: argument validation, workspace carving, kernel sequencing.
// The contract of every entry point is stated in include/of3pair.h.
#include "../../include/of3pair.h"

#include <hip/hip_runtime.h>

#include <mutex>

#include "of3_kernels.h"
#include "of3_launch.h"
#include "of3_weight_split.h"

// Built-in scratch of of3_trimul_fwd_static: one copy per GPU the library runs on, held until the
// process ends.  In host code this name is only a handle for hipGetSymbolAddress; the device
// address it yields (one per device) is what kernels and copies are given.
static __device__ __align__(256) unsigned char scratch[OF3_STATIC_SCRATCH_BYTES];

namespace {

std::mutex g_scratch_mutex;
void* g_scratch_ptr[of3::kMaxDevices];  // device address of `scratch` on each device, null until looked up

// Address of the current device's copy of `scratch` (looked up on the first call on that device).
hipError_t static_scratch(void** out) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= of3::kMaxDevices) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void* ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    if (!ptr) return hipErrorInvalidSymbol;
    g_scratch_ptr[dev] = ptr;
  }
  *out = g_scratch_ptr[dev];
  return hipSuccess;
}

thread_local int g_last_hip_error = 0;

inline int fail_hip(hipError_t e) {
  g_last_hip_error = (int)e;
  return OF3_EHIP;
}

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
inline int64_t align256(int64_t n) { return (n + 255) & ~(int64_t)255; }
inline int64_t padded(int64_t n) { return (n + 127) / 128 * 128; }

// The kernels count positions, tiles and work-groups in 32-bit integers: every shape whose padded
// position count B * NP * NP does not fit one is refused before any launch (such a pair tensor
// would exceed the memory of the device by far).
inline bool positions_ok(int64_t B, int64_t N) {
  if (B < 1 || N < 1 || N > (1 << 20) || B > 0x7fffffffll) return false;
  const int64_t np = padded(N);
  return np * np <= 0x7fffffffll / B;
}

inline bool trimul_dims_ok(int64_t B, int64_t N, int64_t C, int64_t CH) {
  if (!positions_ok(B, N)) return false;
  return (C == 128 && CH == 128) || (C == 64 && CH == 64);
}
inline bool triattn_dims_ok(int64_t B, int64_t N, int64_t C, int64_t H, int64_t D) {
  if (!positions_ok(B, N)) return false;
  if (B * H > 65535 || (N + 3) / 4 > 65535) return false;
  return H == 4 && ((C == 128 && D == 32) || (C == 64 && D == 16));
}
inline bool strides_ok(const int64_t s[3]) {
  return s && s[0] >= 0 && s[1] > 0 && s[2] > 0 && (s[0] % 8 == 0) && (s[1] % 8 == 0) && (s[2] % 8 == 0);
}
inline bool mask_ok(const float* mask, const int64_t s[3]) {
  if (!mask) return true;
  return s && s[0] >= 0 && s[1] >= 0 && s[2] >= 0;
}

inline bool f32_trimul_dims_ok(int64_t B, int64_t N, int64_t C, int64_t CH) {
  return positions_ok(B, N) && N <= (1 << 16) && C >= 1 && C <= 256 && CH >= 1 && CH <= 256;
}
inline bool f32_triattn_dims_ok(int64_t B, int64_t N, int64_t C, int64_t H, int64_t D) {
  return positions_ok(B, N) && N <= (1 << 16) && C >= 1 && C <= 256 && H >= 1 && D >= 1 && D <= 64 && H * D <= 256;
}
inline int64_t f32_triattn_qkv_bytes(int64_t B, int64_t N, int64_t H, int64_t D) {
  const int64_t fp32 = 3 * align256(B * N * N * H * D * 4), split = align256((int64_t)of3::triattn_qkv_split_bytes(B, N, H, D));
  return fp32 > split ? fp32 : split;
}
inline int64_t f32_trimul_ab_bytes(int64_t B, int64_t N, int64_t CH) {
  const int64_t fp32 = 2 * align256(B * CH * N * N * 4), split = align256((int64_t)of3::trimul_ab_split_bytes(B, N, CH));
  return fp32 > split ? fp32 : split;
}
// the triangle bias, rows padded to whole 32-key tiles
inline int64_t f32_triattn_tb_bytes(int64_t B, int64_t N, int64_t H) { return align256(B * H * N * ((N + 31) / 32 * 32) * 4); }
inline bool f32_strides_ok(const int64_t s[3]) { return s && s[0] >= 0 && s[1] > 0 && s[2] > 0; }
inline bool aligned4(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 3u) == 0; }

inline of3::PairView view(const int64_t s[3], bool swap) {
  of3::PairView v;
  v.stride_b = s[0];
  v.stride_r = swap ? s[2] : s[1];
  v.stride_k = swap ? s[1] : s[2];
  return v;
}
inline of3::PairView mask_view(const float* mask, const int64_t s[3], bool swap) {
  of3::PairView v = {0, 0, 0};
  if (mask) v = view(s, swap);
  return v;
}

inline const of3::bf16_t* bf(const void* p) { return static_cast<const of3::bf16_t*>(p); }
inline of3::bf16_t* bf(void* p) { return static_cast<of3::bf16_t*>(p); }

// compute units of the current device (one persistent work-group of the contraction each); 256, the
// MI355X, when no device can be asked (the shape queries are also answered without a GPU)
inline int64_t current_cu_count() {
  static int cache[of3::kMaxDevices];
  int cus = 0;
  hipError_t e = of3::per_device(cache, [](int dev, int* v) { return of3::cu_count(dev, v); }, &cus);
  if (e != hipSuccess) {
    (void)hipGetLastError();  // a shape query must not leave an error behind for the next HIP call
    return 256;
  }
  return cus >= 8 ? (cus / 8) * 8 : 8;
}

inline int contract_variant_auto(int64_t planes, int64_t Np) {
  // Cheapest of the four output tile shapes for this problem on the device's compute units (256 on
  // an MI355X): rounds of persistent work-groups x padded tile area, with a small bonus for the wider
  // tiles, which move fewer operand bytes per flop.  (768: 384x192 gives every work-group
  // exactly 4 tiles and every XCD whole planes per round; 512, 1024, 2048: 256x256 divides the
  // plane without waste.)
  const int64_t cus = current_cu_count();
  const int64_t bm[4] = {256, 256, 256, 384};
  const int64_t bn[4] = {192, 128, 256, 192};
  const double eff[4] = {0.93, 0.85, 1.00, 1.00};
  int best = 1;
  double best_cost = 0;
  for (int v = 0; v < 4; ++v) {
    const int64_t tiles = planes * ((Np + bm[v] - 1) / bm[v]) * ((Np + bn[v] - 1) / bn[v]);
    const double cost = (double)((tiles + cus - 1) / cus) * (double)(bm[v] * bn[v]) / eff[v];
    if (v == 0 || cost < best_cost) {
      best = v + 1;
      best_cost = cost;
    }
  }
  return best;
}

}  // namespace

extern "C" {

int of3_version(void) { return 1; }
int of3_last_hip_error(void) { return g_last_hip_error; }

const char* of3_status_string(int status) {
  switch (status) {
    case OF3_OK:
      return "ok";
    case OF3_EINVAL:
      return "invalid argument (shape, stride, alignment, dtype or null pointer)";
    case OF3_ENOSPC:
      return "workspace too small";
    case OF3_EHIP:
      return "HIP error (see of3_last_hip_error)";
    case OF3_ESTATIC:
      return "problem needs more scratch than the library's built-in OF3_STATIC_SCRATCH_BYTES; use the entry "
             "point that takes a workspace";
    default:
      return "unknown status";
  }
}

int64_t of3_padded_n(int64_t n) { return n < 1 ? 0 : padded(n); }

int of3_trimul_contract_variant(int64_t B, int64_t N, int64_t CH) {
  if (!positions_ok(B, N) || (CH != 128 && CH != 64)) return OF3_EINVAL;
  return contract_variant_auto(B * CH, padded(N));
}

int64_t of3_trimul_workspace_bytes(int64_t B, int64_t N, int64_t C, int64_t CH) {
  if (!trimul_dims_ok(B, N, C, CH)) return OF3_EINVAL;
  const int64_t Np = padded(N);
  return 3 * align256(B * CH * Np * Np * 2);
}

int64_t of3_trimul_workspace_bytes_for(int dtype, int64_t B, int64_t N, int64_t C, int64_t CH) {
  if (dtype == OF3_DTYPE_BF16) return of3_trimul_workspace_bytes(B, N, C, CH);
  if (dtype != OF3_DTYPE_F32 || !f32_trimul_dims_ok(B, N, C, CH)) return OF3_EINVAL;
  // a, b (fp32, or split into terms in whole 32-wide panels: room for three bf16 ones), x and the weights split likewise
  return f32_trimul_ab_bytes(B, N, CH) + align256(B * CH * N * N * 4) + align256((int64_t)of3::trimul_wsplit_bytes(C, CH));
}

// a module's output pass that waits for the next module's input pass (pair_join_bf16.hip)
struct ModuleEnd {
  enum { kMul, kAtt } is;
  of3::TrimulOutArgs mul;
  of3::TriattnOutArgs att;
  of3::TriattnF32 att_f32;  // fp32: o is null where the pass has not been deferred
};

static int trimul_proj(int packed, const void* z, const int64_t z_strides[3], const float* mask,
                       const int64_t mask_strides[3], const void* ln_in_w, const void* ln_in_b, const void* w_a_p,
                       const void* w_a_g, const void* w_b_p, const void* w_b_g, void* a, void* b, int64_t B, int64_t N,
                       int64_t C, int64_t CH, int outgoing, void* stream, const ModuleEnd* before = nullptr) {
  if (!trimul_dims_ok(B, N, C, CH) || !strides_ok(z_strides) || !mask_ok(mask, mask_strides)) return OF3_EINVAL;
  const void* ptrs[] = {z, ln_in_w, ln_in_b, w_a_p, w_a_g, w_b_p, w_b_g, a, b};
  for (const void* p : ptrs)
    if (!p || !aligned16(p)) return OF3_EINVAL;
  of3::TrimulProjArgs args;
  args.z = bf(z);
  args.mask = mask;
  args.z_view = view(z_strides, !outgoing);
  args.mask_view = mask_view(mask, mask_strides, !outgoing);
  args.ln_w = bf(ln_in_w);
  args.ln_b = bf(ln_in_b);
  args.w_ap = bf(w_a_p);
  args.w_ag = bf(w_a_g);
  args.w_bp = bf(w_b_p);
  args.w_bg = bf(w_b_g);
  args.a = bf(a);
  args.b = bf(b);
  args.B = (int)B;
  args.N = (int)N;
  args.Np = (int)padded(N);
  args.packed = packed;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  hipError_t e = !before                             ? of3::trimul_proj_launch(args, (int)C, (int)CH, s)
                 : before->is == ModuleEnd::kMul ? of3::trimul_trimul_launch(before->mul, args, (int)C, s)
                                                 : of3::triattn_trimul_launch(before->att, args, (int)C, s);
  return e == hipSuccess ? OF3_OK : fail_hip(e);
}

int of3_trimul_proj(const void* z, const int64_t z_strides[3], const float* mask, const int64_t mask_strides[3],
                    const void* ln_in_w, const void* ln_in_b, const void* w_a_p, const void* w_a_g,
                    const void* w_b_p, const void* w_b_g, void* a, void* b, int64_t B, int64_t N, int64_t C,
                    int64_t CH, int outgoing, void* stream) {
  return trimul_proj(0, z, z_strides, mask, mask_strides, ln_in_w, ln_in_b, w_a_p, w_a_g, w_b_p, w_b_g, a, b, B, N,
                     C, CH, outgoing, stream);
}

// transposed: every plane of x as its transpose (variants 2 and 3)
static int trimul_contract(const void* a, const void* b, void* x, int64_t B, int64_t N, int64_t CH, int variant, bool transposed,
                           void* stream) {
  if (!positions_ok(B, N) || (CH != 128 && CH != 64) || variant < 0 || variant > 4) return OF3_EINVAL;
  if (!a || !b || !x || !aligned16(a) || !aligned16(b) || !aligned16(x)) return OF3_EINVAL;
  const int64_t Np = padded(N);
  if (variant == 0) variant = contract_variant_auto(B * CH, Np);
  hipError_t e = of3::trimul_contract_launch(bf(a), bf(b), bf(x), (int)(B * CH), (int)Np, (int)((N + 31) / 32), variant,
                                             transposed, static_cast<hipStream_t>(stream));
  return e == hipSuccess ? OF3_OK : fail_hip(e);
}

int of3_trimul_contract(const void* a, const void* b, void* x, int64_t B, int64_t N, int64_t CH, int variant,
                        void* stream) {
  return trimul_contract(a, b, x, B, N, CH, variant, false, stream);
}

static int trimul_out(int packed, const void* x, const void* z, const int64_t z_strides[3], void* out,
                      const void* ln_in_w, const void* ln_in_b, const void* ln_out_w, const void* ln_out_b,
                      const void* w_g, const void* w_z, int64_t B, int64_t N, int64_t C, int64_t CH, int add_residual,
                      void* stream, ModuleEnd* deferred = nullptr) {
  if (!trimul_dims_ok(B, N, C, CH) || !strides_ok(z_strides)) return OF3_EINVAL;
  const void* ptrs[] = {x, z, out, ln_in_w, ln_in_b, ln_out_w, ln_out_b, w_g, w_z};
  for (const void* p : ptrs)
    if (!p || !aligned16(p)) return OF3_EINVAL;
  of3::TrimulOutArgs args;
  args.x = bf(x);
  args.z = bf(z);
  args.out = bf(out);
  args.z_view = view(z_strides, false);
  args.ln_in_w = bf(ln_in_w);
  args.ln_in_b = bf(ln_in_b);
  args.ln_out_w = bf(ln_out_w);
  args.ln_out_b = bf(ln_out_b);
  args.w_g = bf(w_g);
  args.w_z = bf(w_z);
  args.B = (int)B;
  args.N = (int)N;
  args.Np = (int)padded(N);
  args.add_residual = add_residual ? 1 : 0;
  args.packed = packed;
  if (deferred) {
    deferred->mul = args;
    deferred->is = ModuleEnd::kMul;
    return OF3_OK;
  }
  hipError_t e = of3::trimul_out_launch(args, (int)C, (int)CH, static_cast<hipStream_t>(stream));
  return e == hipSuccess ? OF3_OK : fail_hip(e);
}

int of3_trimul_out(const void* x, const void* z, const int64_t z_strides[3], void* out, const void* ln_in_w,
                   const void* ln_in_b, const void* ln_out_w, const void* ln_out_b, const void* w_g,
                   const void* w_z, int64_t B, int64_t N, int64_t C, int64_t CH, int add_residual, void* stream) {
  return trimul_out(0, x, z, z_strides, out, ln_in_w, ln_in_b, ln_out_w, ln_out_b, w_g, w_z, B, N, C, CH,
                    add_residual, stream);
}

// presplit: the fp32 weights as a block's call has split them, or null; packed: the bf16 weight matrices are copies in
// MFMA operand order; before (bf16): the end of the module before this one, launched with this one's input pass;
// deferred (bf16): the output pass is not launched but handed on, to the `before` of the next module, in whose frame
// (transposed: of the canonical one) x is written
static int trimul_fwd(const of3::WeightX3* presplit, int packed, const void* z, const int64_t z_strides[3], const float* mask,
                   const int64_t mask_strides[3], const void* ln_in_w, const void* ln_in_b, const void* ln_out_w, const void* ln_out_b,
                   const void* w_a_p, const void* w_a_g, const void* w_b_p, const void* w_b_g, const void* w_g,
                   const void* w_z, void* out, int64_t B, int64_t N, int64_t C, int64_t CH, int outgoing,
                   int add_residual, void* workspace, int64_t workspace_bytes, int dtype, void* stream,
                   const ModuleEnd* before = nullptr, ModuleEnd* deferred = nullptr, bool transposed = false) {
  if (dtype == OF3_DTYPE_F32) {
    if (!f32_trimul_dims_ok(B, N, C, CH) || !f32_strides_ok(z_strides) || !mask_ok(mask, mask_strides)) return OF3_EINVAL;
    const void* ptrs[] = {z, ln_in_w, ln_in_b, ln_out_w, ln_out_b, w_a_p, w_a_g, w_b_p, w_b_g, w_g, w_z, out};
    for (const void* p : ptrs)
      if (!p || !aligned4(p)) return OF3_EINVAL;
    if (!workspace || (reinterpret_cast<uintptr_t>(workspace) & 255u)) return OF3_EINVAL;
    if (workspace_bytes < of3_trimul_workspace_bytes_for(dtype, B, N, C, CH)) return OF3_ENOSPC;
    const int64_t part = align256(B * CH * N * N * 4);
    char* ws = static_cast<char*>(workspace);
    auto f = [](const void* p) { return static_cast<const float*>(p); };
    of3::TrimulF32Args a;
    a.z = f(z);
    a.mask = mask;
    a.z_view = view(z_strides, !outgoing);
    a.mask_view = mask_view(mask, mask_strides, !outgoing);
    a.z_canonical = view(z_strides, false);
    a.ln_in_w = f(ln_in_w);
    a.ln_in_b = f(ln_in_b);
    a.ln_out_w = f(ln_out_w);
    a.ln_out_b = f(ln_out_b);
    a.w_ap = f(w_a_p);
    a.w_ag = f(w_a_g);
    a.w_bp = f(w_b_p);
    a.w_bg = f(w_b_g);
    a.w_g = f(w_g);
    a.w_z = f(w_z);
    const int64_t ab = f32_trimul_ab_bytes(B, N, CH);
    a.a = reinterpret_cast<float*>(ws);
    a.b = reinterpret_cast<float*>(ws + part);
    a.ab_split = ws;  // in place of a and b
    a.x = reinterpret_cast<float*>(ws + ab);
    a.wsplit = ws + ab + part;
    a.presplit = presplit;
    a.out = static_cast<float*>(out);
    a.B = (int)B;
    a.N = (int)N;
    a.C = (int)C;
    a.CH = (int)CH;
    a.add_residual = add_residual ? 1 : 0;
    hipError_t e = of3::trimul_fwd_f32(a, static_cast<hipStream_t>(stream));
    return e == hipSuccess ? OF3_OK : (e == hipErrorInvalidValue ? (int)OF3_EINVAL : fail_hip(e));
  }
  if (dtype != OF3_DTYPE_BF16) return OF3_EINVAL;
  if (!trimul_dims_ok(B, N, C, CH)) return OF3_EINVAL;
  if (!workspace || (reinterpret_cast<uintptr_t>(workspace) & 255u)) return OF3_EINVAL;
  if (workspace_bytes < of3_trimul_workspace_bytes(B, N, C, CH)) return OF3_ENOSPC;
  const int64_t Np = padded(N);
  const int64_t part = align256(B * CH * Np * Np * 2);
  char* ws = static_cast<char*>(workspace);
  void* a = ws;
  void* b = ws + part;
  void* x = ws + 2 * part;
  int st = trimul_proj(packed, z, z_strides, mask, mask_strides, ln_in_w, ln_in_b, w_a_p, w_a_g, w_b_p, w_b_g, a, b, B, N,
                           C, CH, outgoing, stream, before);
  if (st != OF3_OK) return st;
  st = trimul_contract(a, b, x, B, N, CH, 0, transposed, stream);
  if (st != OF3_OK) return st;
  return trimul_out(packed, x, z, z_strides, out, ln_in_w, ln_in_b, ln_out_w, ln_out_b, w_g, w_z, B, N, C, CH,
                        add_residual, stream, deferred);
}

int of3_trimul_fwd(const void* z, const int64_t z_strides[3], const float* mask, const int64_t mask_strides[3],
                   const void* ln_in_w, const void* ln_in_b, const void* ln_out_w, const void* ln_out_b,
                   const void* w_a_p, const void* w_a_g, const void* w_b_p, const void* w_b_g, const void* w_g,
                   const void* w_z, void* out, int64_t B, int64_t N, int64_t C, int64_t CH, int outgoing,
                   int add_residual, void* workspace, int64_t workspace_bytes, int dtype, void* stream) {
  return trimul_fwd(nullptr, 0, z, z_strides, mask, mask_strides, ln_in_w, ln_in_b, ln_out_w, ln_out_b, w_a_p, w_a_g, w_b_p,
                    w_b_g, w_g, w_z, out, B, N, C, CH, outgoing, add_residual, workspace, workspace_bytes, dtype, stream);
}

int of3_trimul_fwd_static(const void* z, const int64_t z_strides[3], const float* mask,
                          const int64_t mask_strides[3], const void* ln_in_w, const void* ln_in_b, const void* ln_out_w,
                          const void* ln_out_b, const void* w_a_p, const void* w_a_g, const void* w_b_p,
                          const void* w_b_g, const void* w_g, const void* w_z, void* out, int64_t B, int64_t N,
                          int64_t C, int64_t CH, int outgoing, int add_residual, int dtype, void* stream) {
  const int64_t need = of3_trimul_workspace_bytes_for(dtype, B, N, C, CH);
  if (need < 0) return OF3_EINVAL;
  if (need > (int64_t)OF3_STATIC_SCRATCH_BYTES) return OF3_ESTATIC;
  void* ws = nullptr;
  hipError_t e = static_scratch(&ws);
  if (e != hipSuccess) return fail_hip(e);
  // a, b and x are written in full before they are read (entries beyond N that the kernels read
  // feed only outputs beyond N, which nothing reads), so what the last call left needs no clearing
  return of3_trimul_fwd(z, z_strides, mask, mask_strides, ln_in_w, ln_in_b, ln_out_w, ln_out_b, w_a_p, w_a_g, w_b_p,
                        w_b_g, w_g, w_z, out, B, N, C, CH, outgoing, add_residual, ws, (int64_t)OF3_STATIC_SCRATCH_BYTES,
                        dtype, stream);
}

int64_t of3_triattn_workspace_bytes(int64_t B, int64_t N, int64_t C, int64_t H, int64_t D) {
  if (!triattn_dims_ok(B, N, C, H, D)) return OF3_EINVAL;
  const int64_t Np = padded(N);
  const int64_t qkv = align256(B * N * H * Np * D * 2);
  return 3 * qkv + align256(B * H * N * Np * 4) + align256(B * N * Np * 4) + align256(B * N * N * H * D * 2);
}

int64_t of3_triattn_workspace_bytes_for(int dtype, int64_t B, int64_t N, int64_t C, int64_t H, int64_t D) {
  if (dtype == OF3_DTYPE_BF16) return of3_triattn_workspace_bytes(B, N, C, H, D);
  if (dtype != OF3_DTYPE_F32 || !f32_triattn_dims_ok(B, N, C, H, D)) return OF3_EINVAL;
  // q, k, v (fp32, or split into terms in whole 32-position tiles: room for three bf16 ones), o, the triangle bias
  // and the weights split likewise
  return f32_triattn_qkv_bytes(B, N, H, D) + align256(B * N * N * H * D * 4) + f32_triattn_tb_bytes(B, N, H) +
         align256((int64_t)of3::triattn_wsplit_bytes(C, H, D));
}

static int triattn_proj(int packed, const void* x, const int64_t x_strides[3], const float* mask,
                        const int64_t mask_strides[3], const void* ln_w, const void* ln_b, const void* w_q,
                        const void* w_k, const void* w_v, const void* w_bias, void* q, void* k, void* vt, float* tbias,
                        float* mbias, int64_t B, int64_t N, int64_t C, int64_t H, int64_t D, float inf, void* stream,
                        const ModuleEnd* before = nullptr) {
  if (!triattn_dims_ok(B, N, C, H, D) || !strides_ok(x_strides) || !mask_ok(mask, mask_strides)) return OF3_EINVAL;
  const void* ptrs[] = {x, ln_w, ln_b, w_q, w_k, w_v, w_bias, q, k, vt, tbias, mbias};
  for (const void* p : ptrs)
    if (!p || !aligned16(p)) return OF3_EINVAL;
  of3::TriattnProjArgs args;
  args.x = bf(x);
  args.mask = mask;
  args.x_view = view(x_strides, false);
  args.mask_view = mask_view(mask, mask_strides, false);
  args.ln_w = bf(ln_w);
  args.ln_b = bf(ln_b);
  args.w_q = bf(w_q);
  args.w_k = bf(w_k);
  args.w_v = bf(w_v);
  args.w_b = bf(w_bias);
  args.q = bf(q);
  args.k = bf(k);
  args.vt = bf(vt);
  args.tbias = tbias;
  args.mbias = mbias;
  args.B = (int)B;
  args.N = (int)N;
  args.Jp = (int)padded(N);
  args.H = (int)H;
  args.inf = inf;
  args.packed = packed;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  hipError_t e = !before                             ? of3::triattn_proj_launch(args, (int)C, (int)D, s)
                 : before->is == ModuleEnd::kMul ? of3::trimul_triattn_launch(before->mul, args, (int)C, s)
                                                 : of3::triattn_triattn_launch(before->att, args, (int)C, s);
  return e == hipSuccess ? OF3_OK : fail_hip(e);
}

int of3_triattn_proj(const void* x, const int64_t x_strides[3], const float* mask, const int64_t mask_strides[3],
                     const void* ln_w, const void* ln_b, const void* w_q, const void* w_k, const void* w_v,
                     const void* w_bias, void* q, void* k, void* vt, float* tbias, float* mbias, int64_t B,
                     int64_t N, int64_t C, int64_t H, int64_t D, float inf, void* stream) {
  return triattn_proj(0, x, x_strides, mask, mask_strides, ln_w, ln_b, w_q, w_k, w_v, w_bias, q, k, vt, tbias, mbias,
                      B, N, C, H, D, inf, stream);
}

int of3_triattn_flash(const void* q, const void* k, const void* vt, const float* tbias, const float* mbias, void* o,
                      int64_t B, int64_t N, int64_t H, int64_t D, void* stream) {
  const int64_t C = (D == 32) ? 128 : 64;
  if (!triattn_dims_ok(B, N, C, H, D)) return OF3_EINVAL;
  const void* ptrs[] = {q, k, vt, tbias, mbias, o};
  for (const void* p : ptrs)
    if (!p || !aligned16(p)) return OF3_EINVAL;
  of3::TriattnFlashArgs args;
  args.q = bf(q);
  args.k = bf(k);
  args.vt = bf(vt);
  args.tbias = tbias;
  args.mbias = mbias;
  args.o = bf(o);
  args.B = (int)B;
  args.N = (int)N;
  args.Jp = (int)padded(N);
  args.H = (int)H;
  hipError_t e = of3::triattn_flash_launch(args, (int)D, static_cast<hipStream_t>(stream));
  return e == hipSuccess ? OF3_OK : fail_hip(e);
}

static int triattn_out(int packed, const void* o, const void* x, const int64_t x_strides[3], void* out,
                       const void* ln_w, const void* ln_b, const void* w_g, const void* w_o, int64_t B, int64_t N,
                       int64_t C, int64_t H, int64_t D, int add_residual, void* stream, ModuleEnd* deferred = nullptr) {
  if (!triattn_dims_ok(B, N, C, H, D) || !strides_ok(x_strides)) return OF3_EINVAL;
  const void* ptrs[] = {o, x, out, ln_w, ln_b, w_g, w_o};
  for (const void* p : ptrs)
    if (!p || !aligned16(p)) return OF3_EINVAL;
  of3::TriattnOutArgs args;
  args.o = bf(o);
  args.x = bf(x);
  args.out = bf(out);
  args.x_view = view(x_strides, false);
  args.ln_w = bf(ln_w);
  args.ln_b = bf(ln_b);
  args.w_g = bf(w_g);
  args.w_o = bf(w_o);
  args.B = (int)B;
  args.N = (int)N;
  args.add_residual = add_residual ? 1 : 0;
  args.packed = packed;
  if (deferred) {
    deferred->att = args;
    deferred->is = ModuleEnd::kAtt;
    return OF3_OK;
  }
  hipError_t e = of3::triattn_out_launch(args, (int)C, (int)(H * D), static_cast<hipStream_t>(stream));
  return e == hipSuccess ? OF3_OK : fail_hip(e);
}

int of3_triattn_out(const void* o, const void* x, const int64_t x_strides[3], void* out, const void* ln_w,
                    const void* ln_b, const void* w_g, const void* w_o, int64_t B, int64_t N, int64_t C, int64_t H,
                    int64_t D, int add_residual, void* stream) {
  return triattn_out(0, o, x, x_strides, out, ln_w, ln_b, w_g, w_o, B, N, C, H, D, add_residual, stream);
}

static int triattn_fwd(const of3::WeightX3* presplit, int packed, const void* x, const int64_t x_strides[3], const float* mask,
                    const int64_t mask_strides[3], const void* ln_w, const void* ln_b, const void* w_bias, const void* w_q, const void* w_k,
                    const void* w_v, const void* w_g, const void* w_o, void* out, int64_t B, int64_t N, int64_t C,
                    int64_t H, int64_t D, float inf, int add_residual, void* workspace, int64_t workspace_bytes,
                    int dtype, void* stream, const ModuleEnd* before = nullptr, ModuleEnd* deferred = nullptr) {
  if (dtype == OF3_DTYPE_F32) {
    if (!f32_triattn_dims_ok(B, N, C, H, D) || !f32_strides_ok(x_strides) || !mask_ok(mask, mask_strides)) return OF3_EINVAL;
    const void* ptrs[] = {x, ln_w, ln_b, w_bias, w_q, w_k, w_v, w_g, w_o, out};
    for (const void* p : ptrs)
      if (!p || !aligned4(p)) return OF3_EINVAL;
    if (!workspace || (reinterpret_cast<uintptr_t>(workspace) & 255u)) return OF3_EINVAL;
    if (workspace_bytes < of3_triattn_workspace_bytes_for(dtype, B, N, C, H, D)) return OF3_ENOSPC;
    const int64_t part = align256(B * N * N * H * D * 4);
    char* ws = static_cast<char*>(workspace);
    auto f = [](const void* p) { return static_cast<const float*>(p); };
    of3::TriattnF32Args a;
    a.x = f(x);
    a.mask = mask;
    a.x_view = view(x_strides, false);
    a.mask_view = mask_view(mask, mask_strides, false);
    a.ln_w = f(ln_w);
    a.ln_b = f(ln_b);
    a.w_q = f(w_q);
    a.w_k = f(w_k);
    a.w_v = f(w_v);
    a.w_b = f(w_bias);
    a.w_g = f(w_g);
    a.w_o = f(w_o);
    a.q = reinterpret_cast<float*>(ws);
    a.k = reinterpret_cast<float*>(ws + part);
    a.v = reinterpret_cast<float*>(ws + 2 * part);
    const int64_t qkv = f32_triattn_qkv_bytes(B, N, H, D);
    a.qkv_split = ws;  // in place of q, k, v
    a.o = reinterpret_cast<float*>(ws + qkv);
    a.tb = reinterpret_cast<float*>(ws + qkv + part);
    a.wsplit = ws + qkv + part + f32_triattn_tb_bytes(B, N, H);
    a.presplit = presplit;
    a.out = static_cast<float*>(out);
    a.B = (int)B;
    a.N = (int)N;
    a.C = (int)C;
    a.H = (int)H;
    a.D = (int)D;
    a.add_residual = add_residual ? 1 : 0;
    a.inf = inf;
    if (deferred) {
      deferred->att_f32.o = nullptr;
      a.deferred = &deferred->att_f32;
    }
    hipError_t e = of3::triattn_fwd_f32(a, static_cast<hipStream_t>(stream));
    return e == hipSuccess ? OF3_OK : (e == hipErrorInvalidValue ? (int)OF3_EINVAL : fail_hip(e));
  }
  if (dtype != OF3_DTYPE_BF16) return OF3_EINVAL;
  if (!triattn_dims_ok(B, N, C, H, D)) return OF3_EINVAL;
  if (!workspace || (reinterpret_cast<uintptr_t>(workspace) & 255u)) return OF3_EINVAL;
  if (workspace_bytes < of3_triattn_workspace_bytes(B, N, C, H, D)) return OF3_ENOSPC;
  const int64_t Np = padded(N);
  const int64_t qkv = align256(B * N * H * Np * D * 2);
  char* ws = static_cast<char*>(workspace);
  void* q = ws;
  void* k = ws + qkv;
  void* vt = ws + 2 * qkv;
  float* tbias = reinterpret_cast<float*>(ws + 3 * qkv);
  float* mbias = reinterpret_cast<float*>(ws + 3 * qkv + align256(B * H * N * Np * 4));
  void* o = ws + 3 * qkv + align256(B * H * N * Np * 4) + align256(B * N * Np * 4);
  int st = triattn_proj(packed, x, x_strides, mask, mask_strides, ln_w, ln_b, w_q, w_k, w_v, w_bias, q, k, vt, tbias,
                            mbias, B, N, C, H, D, inf, stream, before);
  if (st != OF3_OK) return st;
  st = of3_triattn_flash(q, k, vt, tbias, mbias, o, B, N, H, D, stream);
  if (st != OF3_OK) return st;
  return triattn_out(packed, o, x, x_strides, out, ln_w, ln_b, w_g, w_o, B, N, C, H, D, add_residual, stream, deferred);
}

int of3_triattn_fwd(const void* x, const int64_t x_strides[3], const float* mask, const int64_t mask_strides[3],
                    const void* ln_w, const void* ln_b, const void* w_bias, const void* w_q, const void* w_k,
                    const void* w_v, const void* w_g, const void* w_o, void* out, int64_t B, int64_t N, int64_t C,
                    int64_t H, int64_t D, float inf, int add_residual, void* workspace, int64_t workspace_bytes,
                    int dtype, void* stream) {
  return triattn_fwd(nullptr, 0, x, x_strides, mask, mask_strides, ln_w, ln_b, w_bias, w_q, w_k, w_v, w_g, w_o, out, B, N, C,
                     H, D, inf, add_residual, workspace, workspace_bytes, dtype, stream);
}

int64_t of3_transition_workspace_bytes_for(int dtype, int64_t B, int64_t N, int64_t C, int64_t HID) {
  if (dtype == OF3_DTYPE_BF16) return (B >= 1 && N >= 1) ? 0 : (int64_t)OF3_EINVAL;
  if (dtype != OF3_DTYPE_F32 || B < 1 || N < 1 || C < 1 || C > 256 || HID < 1 || HID > 1024) return OF3_EINVAL;
  return align256((int64_t)of3::transition_wsplit_bytes(C, HID));  // the weights split into terms
}

int of3_transition_fwd(const void* x, const int64_t x_strides[3], const float* mask, const int64_t mask_strides[3],
                       const void* ln_w, const void* ln_b, const void* w_a, const void* w_b, const void* w_out,
                       void* out, int64_t B, int64_t N, int64_t C, int64_t HID, int add_residual, int dtype,
                       void* stream) {
  return of3_transition_fwd_ws(x, x_strides, mask, mask_strides, ln_w, ln_b, w_a, w_b, w_out, out, B, N, C, HID,
                               add_residual, nullptr, 0, dtype, stream);
}

// A block's pair bias of the attention over s, to go with its last pair launch
struct BlockBias {
  of3::PairBiasArgs bf16;
  of3::PairBiasF32Args f32;
};

// presplit as above; operands: w_a, w_b, w_out in MFMA operand order (bf16), or null.  before: the attention whose output pass the
// launch begins with; takes_end: says whether it could, and launches nothing; bias: a pair bias of the result that goes with `before`
static int transition_fwd(const of3::WeightX3* presplit, const void* const* operands, const void* x, const int64_t x_strides[3], const float* mask,
                          const int64_t mask_strides[3], const void* ln_w, const void* ln_b, const void* w_a, const void* w_b, const void* w_out,
                          void* out, int64_t B, int64_t N, int64_t C, int64_t HID, int add_residual, void* workspace,
                          int64_t workspace_bytes, int dtype, void* stream, const ModuleEnd* before = nullptr, bool* takes_end = nullptr,
                          const BlockBias* bias = nullptr, bool* bias_done = nullptr) {
  if (takes_end) *takes_end = false;
  const void* ptrs[] = {x, ln_w, ln_b, w_a, w_b, w_out, out};
  if (!positions_ok(B, N) || !mask_ok(mask, mask_strides)) return OF3_EINVAL;
  if (dtype == OF3_DTYPE_F32) {
    if (N > (1 << 16) || C < 1 || C > 256 || HID < 1 || HID > 1024 || !f32_strides_ok(x_strides)) return OF3_EINVAL;
    for (const void* p : ptrs)
      if (!p || !aligned4(p)) return OF3_EINVAL;
    auto f = [](const void* p) { return static_cast<const float*>(p); };
    of3::TransitionF32Args a;
    a.x = f(x);
    a.mask = mask;
    a.x_view = view(x_strides, false);
    a.mask_view = mask_view(mask, mask_strides, false);
    a.ln_w = f(ln_w);
    a.ln_b = f(ln_b);
    a.w_a = f(w_a);
    a.w_b = f(w_b);
    a.w_out = f(w_out);
    // with room for the split weights the split-operand kernel runs (where the shape allows)
    a.wsplit = nullptr;
    a.presplit = presplit;
    if (workspace) {
      if (reinterpret_cast<uintptr_t>(workspace) & 255u) return OF3_EINVAL;
      if (workspace_bytes < of3_transition_workspace_bytes_for(dtype, B, N, C, HID)) return OF3_ENOSPC;
      a.wsplit = workspace;
    }
    a.out = static_cast<float*>(out);
    a.B = (int)B;
    a.N = (int)N;
    a.C = (int)C;
    a.HID = (int)HID;
    a.add_residual = add_residual ? 1 : 0;
    if (before && before->att_f32.o) a.end = &before->att_f32;
    if (takes_end) return OF3_OK;
    if (a.end && bias) a.bias = &bias->f32, a.bias_done = bias_done;
    hipError_t e = of3::transition_fwd_f32(a, static_cast<hipStream_t>(stream));
    return e == hipSuccess ? OF3_OK : fail_hip(e);
  }
  if (dtype != OF3_DTYPE_BF16) return OF3_EINVAL;
  if (!(C == 128 || C == 64) || HID < 128 || HID % 32 != 0 || HID > (1 << 16) || !strides_ok(x_strides))
    return OF3_EINVAL;
  // A tensor (and mask) whose rows follow one another without gaps is one row of N*N positions per
  // batch element: the kernel's 256-position tiles then do not stop at row ends, which matters when
  // N is not a multiple of 256.  Positions along a row are addressed with 32-bit byte offsets.
  int64_t rows = N, row_len = N;
  if (x_strides[1] == N * x_strides[2] && (!mask || mask_strides[1] == N * mask_strides[2]) &&
      (N * N - 1) * x_strides[2] * 2 + 2 * C <= 0xffffffffll &&
      (!mask || (N * N - 1) * mask_strides[2] * 4 + 4 <= 0xffffffffll)) {
    rows = 1;
    row_len = N * N;
  }
  if ((row_len - 1) * x_strides[2] * 2 + 2 * C > 0xffffffffll) return OF3_EINVAL;
  if (mask && (row_len - 1) * mask_strides[2] * 4 + 4 > 0xffffffffll) return OF3_EINVAL;
  if (B * rows * ((row_len + 255) / 256) > 0x7fffffffll) return OF3_EINVAL;
  for (const void* p : ptrs)
    if (!p || !aligned16(p)) return OF3_EINVAL;
  of3::TransitionArgs args;
  args.x = bf(x);
  args.mask = mask;
  args.x_view = view(x_strides, false);
  args.mask_view = mask_view(mask, mask_strides, false);
  args.ln_w = bf(ln_w);
  args.ln_b = bf(ln_b);
  args.w_a = bf(w_a);
  args.w_b = bf(w_b);
  args.w_out = bf(w_out);
  args.out = bf(out);
  args.B = (int)B;
  args.N = (int)row_len;
  args.R = (int)rows;
  args.HID = (int)HID;
  args.add_residual = add_residual ? 1 : 0;
  for (int i = 0; i < 3 && operands; ++i) args.operands[i] = bf(operands[i]);
  if (takes_end) {
    const hipError_t e = operands && rows == 1 ? of3::transition_after_attention(args, (int)C, takes_end) : hipSuccess;
    return e == hipSuccess ? OF3_OK : fail_hip(e);
  }
  hipError_t e = before ? of3::triattn_transition_launch(before->att, args, bias ? &bias->bf16 : nullptr, (int)C, static_cast<hipStream_t>(stream))
                        : of3::transition_launch(args, (int)C, static_cast<hipStream_t>(stream));
  if (before && bias) *bias_done = true;
  return e == hipSuccess ? OF3_OK : fail_hip(e);
}

int of3_transition_fwd_ws(const void* x, const int64_t x_strides[3], const float* mask, const int64_t mask_strides[3],
                          const void* ln_w, const void* ln_b, const void* w_a, const void* w_b, const void* w_out,
                          void* out, int64_t B, int64_t N, int64_t C, int64_t HID, int add_residual, void* workspace,
                          int64_t workspace_bytes, int dtype, void* stream) {
  return transition_fwd(nullptr, nullptr, x, x_strides, mask, mask_strides, ln_w, ln_b, w_a, w_b, w_out, out, B, N, C, HID,
                        add_residual, workspace, workspace_bytes, dtype, stream);
}

int of3_pair_bias_fwd(const void* z, const int64_t z_strides[3], const void* ln_w, const void* ln_b, const void* w,
                      void* out, int64_t B, int64_t N, int64_t C, int64_t H, int dtype, void* stream) {
  if (!positions_ok(B, N) || N > (1 << 16) || H < 1 || !z || !ln_w || !w || !out) return OF3_EINVAL;
  if (dtype == OF3_DTYPE_F32) {
    if (C < 1 || C > 256 || H > 64 || !f32_strides_ok(z_strides)) return OF3_EINVAL;
    if (!aligned4(z) || !aligned4(ln_w) || !aligned4(ln_b) || !aligned4(w) || !aligned4(out)) return OF3_EINVAL;
    of3::PairBiasF32Args a;
    a.z = static_cast<const float*>(z);
    a.z_view = view(z_strides, false);
    a.ln_w = static_cast<const float*>(ln_w);
    a.ln_b = static_cast<const float*>(ln_b);
    a.w = static_cast<const float*>(w);
    a.out = static_cast<float*>(out);
    a.B = (int)B;
    a.N = (int)N;
    a.C = (int)C;
    a.H = (int)H;
    hipError_t e = of3::pair_bias_fwd_f32(a, static_cast<hipStream_t>(stream));
    return e == hipSuccess ? OF3_OK : fail_hip(e);
  }
  if (dtype != OF3_DTYPE_BF16) return OF3_EINVAL;
  if (!(C == 128 || C == 64) || H > 32 || !strides_ok(z_strides)) return OF3_EINVAL;
  if (!aligned16(z) || !aligned16(ln_w) || !aligned16(ln_b) || !aligned16(w) || !aligned16(out)) return OF3_EINVAL;
  of3::PairBiasArgs a;
  a.z = bf(z);
  a.z_view = view(z_strides, false);
  a.ln_w = bf(ln_w);
  a.ln_b = bf(ln_b);
  a.w = bf(w);
  a.out = bf(out);
  a.B = (int)B;
  a.N = (int)N;
  a.H = (int)H;
  hipError_t e = of3::pair_bias_launch(a, (int)C, static_cast<hipStream_t>(stream));
  return e == hipSuccess ? OF3_OK : fail_hip(e);
}

int of3_layer_norm_fwd(const void* x, const void* ln_w, const void* ln_b, void* out, int64_t rows, int64_t C,
                       int dtype, void* stream) {
  if (rows < 1 || !x || !ln_w || !ln_b || !out) return OF3_EINVAL;
  if (dtype == OF3_DTYPE_F32) {
    if (C < 1 || C > 256) return OF3_EINVAL;
    if (!aligned4(x) || !aligned4(ln_w) || !aligned4(ln_b) || !aligned4(out)) return OF3_EINVAL;
    hipError_t e = of3::layer_norm_fwd_f32(static_cast<const float*>(x), static_cast<const float*>(ln_w),
                                           static_cast<const float*>(ln_b), static_cast<float*>(out), (long)rows,
                                           (int)C, static_cast<hipStream_t>(stream));
    return e == hipSuccess ? OF3_OK : fail_hip(e);
  }
  if (dtype != OF3_DTYPE_BF16) return OF3_EINVAL;
  if (!(C == 128 || C == 64)) return OF3_EINVAL;
  if (!aligned16(x) || !aligned16(ln_w) || !aligned16(ln_b) || !aligned16(out)) return OF3_EINVAL;
  hipError_t e = of3::layer_norm_launch(bf(x), bf(ln_w), bf(ln_b), bf(out), (long)rows, (int)C,
                                        static_cast<hipStream_t>(stream));
  return e == hipSuccess ? OF3_OK : fail_hip(e);
}

int of3_template_tail_fwd(const void* t, const void* ln_w, const void* ln_b, const void* w, void* out, int64_t B,
                          int64_t T, int64_t P, int64_t C_t, int64_t C_z, int apply_ln, int dtype, void* stream) {
  if (B < 1 || T < 1 || T > 1024 || P < 1 || !t || !w || !out) return OF3_EINVAL;
  if (apply_ln && (!ln_w || !ln_b)) return OF3_EINVAL;
  if (B > 0x7fffffffll || P > (1ll << 40)) return OF3_EINVAL;
  if (dtype == OF3_DTYPE_F32) {
    if (C_t < 1 || C_t > 256 || C_z < 1 || C_z > 4096) return OF3_EINVAL;
    if (!aligned4(t) || !aligned4(ln_w) || !aligned4(ln_b) || !aligned4(w) || !aligned4(out)) return OF3_EINVAL;
    of3::TemplateTailF32Args a;
    a.t = static_cast<const float*>(t);
    a.ln_w = static_cast<const float*>(ln_w);
    a.ln_b = static_cast<const float*>(ln_b);
    a.w = static_cast<const float*>(w);
    a.out = static_cast<float*>(out);
    a.P = (long)P;
    a.B = (int)B;
    a.T = (int)T;
    a.CT = (int)C_t;
    a.CZ = (int)C_z;
    a.apply_ln = apply_ln ? 1 : 0;
    hipError_t e = of3::template_tail_fwd_f32(a, static_cast<hipStream_t>(stream));
    return e == hipSuccess ? OF3_OK : fail_hip(e);
  }
  if (dtype != OF3_DTYPE_BF16) return OF3_EINVAL;
  if (C_t != 64 || C_z != 128) return OF3_EINVAL;
  if (!aligned16(t) || !aligned16(ln_w) || !aligned16(ln_b) || !aligned16(w) || !aligned16(out)) return OF3_EINVAL;
  of3::TemplateTailArgs a;
  a.t = bf(t);
  a.ln_w = bf(ln_w);
  a.ln_b = bf(ln_b);
  a.w = bf(w);
  a.out = bf(out);
  a.P = (long)P;
  a.B = (int)B;
  a.T = (int)T;
  a.apply_ln = apply_ln ? 1 : 0;
  hipError_t e = of3::template_tail_launch(a, (int)C_t, (int)C_z, static_cast<hipStream_t>(stream));
  return e == hipSuccess ? OF3_OK : fail_hip(e);
}

int64_t of3_attn_pair_bias_workspace_bytes(int64_t B, int64_t N, int64_t C_s, int64_t H, int64_t D) {
  if (B < 1 || N < 1 || N > (1 << 16) || C_s != 384 || H < 1 || D < 8 || D > 24 || (D % 8) != 0 || H * D != C_s)
    return OF3_EINVAL;
  const int64_t Np = (N + 31) / 32 * 32;
  return 3 * align256(B * H * Np * 32 * 2) + 2 * align256(B * N * H * D * 2);
}

int64_t of3_attn_pair_bias_workspace_bytes_for(int dtype, int64_t B, int64_t N, int64_t C_s, int64_t H, int64_t D) {
  if (dtype == OF3_DTYPE_BF16) return of3_attn_pair_bias_workspace_bytes(B, N, C_s, H, D);
  if (dtype != OF3_DTYPE_F32 || B < 1 || B > 65535 || N < 1 || N > (1 << 16) || C_s < 1 || C_s > 512 || H < 1 ||
      D < 1 || D > 64 || H * D > 512)
    return OF3_EINVAL;
  return 5 * align256(B * N * H * D * 4);
}

// phases: which of the launches (of3_kernels.h)
static int attn_pair_bias(int phases, const void* a, const void* pair_bias, const float* mask, const void* ln_w,
                           const void* ln_b, const void* w_q, const void* b_q, const void* w_k, const void* w_v,
                           const void* w_g, const void* w_o, void* out, int64_t B, int64_t N, int64_t C_s, int64_t H,
                           int64_t D, float inf, int add_residual, void* workspace, int64_t workspace_bytes,
                           int dtype, void* stream) {
  if (dtype == OF3_DTYPE_F32) {
    const int64_t need32 = of3_attn_pair_bias_workspace_bytes_for(dtype, B, N, C_s, H, D);
    if (need32 < 0) return OF3_EINVAL;
    const void* p32[] = {a, pair_bias, ln_w, ln_b, w_q, b_q, w_k, w_v, w_g, w_o, out, workspace};
    for (const void* p : p32)
      if (!p || !aligned4(p)) return OF3_EINVAL;
    if (mask && !aligned4(mask)) return OF3_EINVAL;
    if (workspace_bytes < need32) return OF3_ENOSPC;
    const int64_t part = align256(B * N * H * D * 4);
    char* ws = static_cast<char*>(workspace);
    auto f = [](const void* p) { return static_cast<const float*>(p); };
    of3::SingleAttnF32Args s;
    s.a = f(a);
    s.pair_bias = f(pair_bias);
    s.mask = mask;
    s.ln_w = f(ln_w);
    s.ln_b = f(ln_b);
    s.wq = f(w_q);
    s.bq = f(b_q);
    s.wk = f(w_k);
    s.wv = f(w_v);
    s.wg = f(w_g);
    s.wo = f(w_o);
    s.q = reinterpret_cast<float*>(ws);
    s.k = reinterpret_cast<float*>(ws + part);
    s.v = reinterpret_cast<float*>(ws + 2 * part);
    s.g = reinterpret_cast<float*>(ws + 3 * part);
    s.og = reinterpret_cast<float*>(ws + 4 * part);
    s.out = static_cast<float*>(out);
    s.inf = inf;
    s.B = (int)B;
    s.N = (int)N;
    s.C = (int)C_s;
    s.H = (int)H;
    s.D = (int)D;
    s.add_residual = add_residual ? 1 : 0;
    s.phases = phases;
    hipError_t e = of3::single_attn_fwd_f32(s, static_cast<hipStream_t>(stream));
    return e == hipSuccess ? OF3_OK : fail_hip(e);
  }
  if (dtype != OF3_DTYPE_BF16) return OF3_EINVAL;
  const int64_t need = of3_attn_pair_bias_workspace_bytes(B, N, C_s, H, D);
  if (need < 0 || B > 65535) return OF3_EINVAL;
  const void* ptrs[] = {a, pair_bias, ln_w, ln_b, w_q, b_q, w_k, w_v, w_g, w_o, out, workspace};
  for (const void* p : ptrs)
    if (!p || !aligned16(p)) return OF3_EINVAL;
  if (mask && !aligned4(mask)) return OF3_EINVAL;
  if (workspace_bytes < need) return OF3_ENOSPC;
  const int64_t Np = (N + 31) / 32 * 32;
  const int64_t qk = align256(B * H * Np * 32 * 2), go = align256(B * N * H * D * 2);
  char* ws = static_cast<char*>(workspace);
  of3::SingleAttnArgs s;
  s.a = bf(a);
  s.pair_bias = bf(pair_bias);
  s.mask = mask;
  s.ln_w = bf(ln_w);
  s.ln_b = bf(ln_b);
  s.wq = bf(w_q);
  s.bq = bf(b_q);
  s.wk = bf(w_k);
  s.wv = bf(w_v);
  s.wg = bf(w_g);
  s.wo = bf(w_o);
  s.q = reinterpret_cast<of3::bf16_t*>(ws);
  s.k = reinterpret_cast<of3::bf16_t*>(ws + qk);
  s.vt = reinterpret_cast<of3::bf16_t*>(ws + 2 * qk);
  s.g = reinterpret_cast<of3::bf16_t*>(ws + 3 * qk);
  s.og = reinterpret_cast<of3::bf16_t*>(ws + 3 * qk + go);
  s.out = bf(out);
  s.inf = inf;
  s.B = (int)B;
  s.N = (int)N;
  s.Np = (int)Np;
  s.H = (int)H;
  s.D = (int)D;
  s.add_residual = add_residual ? 1 : 0;
  s.phases = phases;
  hipError_t e = of3::single_attn_launch(s, static_cast<hipStream_t>(stream));
  return e == hipSuccess ? OF3_OK : fail_hip(e);
}

int of3_attn_pair_bias_fwd(const void* a, const void* pair_bias, const float* mask, const void* ln_w,
                           const void* ln_b, const void* w_q, const void* b_q, const void* w_k, const void* w_v,
                           const void* w_g, const void* w_o, void* out, int64_t B, int64_t N, int64_t C_s, int64_t H,
                           int64_t D, float inf, int add_residual, void* workspace, int64_t workspace_bytes,
                           int dtype, void* stream) {
  return attn_pair_bias(of3::kSingleProject | of3::kSingleAttend, a, pair_bias, mask, ln_w, ln_b, w_q, b_q, w_k, w_v, w_g,
                        w_o, out, B, N, C_s, H, D, inf, add_residual, workspace, workspace_bytes, dtype, stream);
}

int64_t of3_transition_rows_workspace_bytes(int64_t rows, int64_t C, int64_t HID) {
  if (rows < 1 || rows > (1ll << 31) || C != 384 || HID < C || (HID % C) != 0 || HID > 5 * C) return OF3_EINVAL;
  return align256(rows * HID * 2);
}

int64_t of3_transition_rows_workspace_bytes_for(int dtype, int64_t rows, int64_t C, int64_t HID) {
  if (dtype == OF3_DTYPE_BF16) return of3_transition_rows_workspace_bytes(rows, C, HID);
  if (dtype != OF3_DTYPE_F32 || rows < 1 || rows > (1ll << 31) || C < 1 || C > 512 || HID < 1 || HID > 2048)
    return OF3_EINVAL;
  return 0;  // the hidden activations stay on chip (of3_transition_rows_fast_workspace_bytes: room for the faster kernels)
}

int64_t of3_transition_rows_fast_workspace_bytes(int dtype, int64_t rows, int64_t C, int64_t HID) {
  const int64_t need = of3_transition_rows_workspace_bytes_for(dtype, rows, C, HID);
  if (need < 0 || dtype == OF3_DTYPE_BF16) return need;
  return C % 32 == 0 && HID % 32 == 0 ? align256(rows * HID * 4) : need;
}

int of3_transition_rows_fwd(const void* x, const float* mask, const void* ln_w, const void* ln_b, const void* w_a,
                            const void* w_b, const void* w_out, void* out, int64_t rows, int64_t C, int64_t HID,
                            int add_residual, void* workspace, int64_t workspace_bytes, int dtype, void* stream) {
  if (dtype == OF3_DTYPE_F32) {
    if (of3_transition_rows_workspace_bytes_for(dtype, rows, C, HID) < 0) return OF3_EINVAL;
    const void* p32[] = {x, ln_w, ln_b, w_a, w_b, w_out, out};
    for (const void* p : p32)
      if (!p || !aligned4(p)) return OF3_EINVAL;
    if (mask && !aligned4(mask)) return OF3_EINVAL;
    auto f = [](const void* p) { return static_cast<const float*>(p); };
    of3::RowTransitionF32Args a;
    a.x = f(x);
    a.mask = mask;
    a.ln_w = f(ln_w);
    a.ln_b = f(ln_b);
    a.wa = f(w_a);
    a.wb = f(w_b);
    a.wout = f(w_out);
    // with room for the hidden activations the matrix-instruction kernels run (where the shape allows)
    const int64_t fast = of3_transition_rows_fast_workspace_bytes(dtype, rows, C, HID);
    a.hidden = workspace && fast > 0 && workspace_bytes >= fast ? static_cast<float*>(workspace) : nullptr;
    a.out = static_cast<float*>(out);
    a.rows = (long)rows;
    a.C = (int)C;
    a.HID = (int)HID;
    a.add_residual = add_residual ? 1 : 0;
    hipError_t e = of3::row_transition_fwd_f32(a, static_cast<hipStream_t>(stream));
    return e == hipSuccess ? OF3_OK : fail_hip(e);
  }
  if (dtype != OF3_DTYPE_BF16) return OF3_EINVAL;
  const int64_t need = of3_transition_rows_workspace_bytes(rows, C, HID);
  if (need < 0) return OF3_EINVAL;
  const void* ptrs[] = {x, ln_w, ln_b, w_a, w_b, w_out, out, workspace};
  for (const void* p : ptrs)
    if (!p || !aligned16(p)) return OF3_EINVAL;
  if (mask && !aligned4(mask)) return OF3_EINVAL;
  if (workspace_bytes < need) return OF3_ENOSPC;
  of3::RowTransitionArgs a;
  a.x = bf(x);
  a.mask = mask;
  a.ln_w = bf(ln_w);
  a.ln_b = bf(ln_b);
  a.wa = bf(w_a);
  a.wb = bf(w_b);
  a.wout = bf(w_out);
  a.h = static_cast<of3::bf16_t*>(workspace);
  a.out = bf(out);
  a.rows = (long)rows;
  a.HID = (int)HID;
  a.add_residual = add_residual ? 1 : 0;
  hipError_t e = of3::row_transition_launch(a, static_cast<hipStream_t>(stream));
  return e == hipSuccess ? OF3_OK : fail_hip(e);
}

// ---- whole blocks in one call ---------------------------------------------------------------
// A block is 12 to 24 kernel launches of 5 to 10 us each at the lengths of small proteins.  Issued module by
// module from Python they cost 260 us of host time per PairFormerBlock, more than the kernels take; from one
// call the launches themselves (2.5 us each) are what is left.

// room for all matrices of a block split at once (fp32), after the modules' own workspace
static int64_t block_split_bytes(int64_t C, int64_t CH, int64_t H, int64_t D, int64_t HID) {
  return align256((int64_t)(2 * of3::trimul_wsplit_bytes(C, CH) + 2 * of3::triattn_wsplit_bytes(C, H, D) +
                            (HID ? of3::transition_wsplit_bytes(C, HID) : 0)));
}
// Short bf16 sequences: the launch that ends one module and begins the next reads the one's workspace and writes the other's,
// so a triangle multiplication's and an attention's lie side by side.  Whether a call takes such launches depends on the
// device (join_rows), the room does not: up to 6144 tiles of 32 positions.
static bool join_room(int dtype, int64_t B, int64_t N) {
  return dtype == OF3_DTYPE_BF16 && N <= of3::kJoinTokens && B <= 8192 && B * N * ((N + 31) / 32) <= 6144;
}
static int64_t pair_block_module_bytes(int dtype, int64_t B, int64_t N, int64_t C, int64_t CH, int64_t H, int64_t D,
                                       int64_t HID) {
  int64_t need = of3_trimul_workspace_bytes_for(dtype, B, N, C, CH);
  const int64_t att = of3_triattn_workspace_bytes_for(dtype, B, N, C, H, D);
  if (need < 0 || att < 0) return OF3_EINVAL;
  if (join_room(dtype, B, N)) need += att;
  else if (att > need) need = att;
  if (HID != 0) {
    if (dtype == OF3_DTYPE_BF16 && (HID < 128 || HID % 32 != 0 || HID > (1 << 16))) return OF3_EINVAL;
    const int64_t tr = of3_transition_workspace_bytes_for(dtype, B, N, C, HID);
    if (tr < 0) return OF3_EINVAL;
    if (tr > need) need = tr;
  }
  return need;
}

// A block's weights as its kernels read them.  fp32 on split operands: all matrices split; bf16: those of the passes
// in MFMA operand order.
struct BlockDims {
  int dtype;
  int64_t B, N, C, CH, H, D, HID;
  float inf;
  bool rows16 = false;  // fp32: z and the result have their rows on 16-byte boundaries, and near each other
  bool wide() const { return dtype == OF3_DTYPE_F32; }
  int weights() const { return OF3_PAIR_BLOCK_WEIGHTS - (HID == 0 ? 5 : 0); }
  int64_t prepared_bytes() const {
    return wide() ? block_split_bytes(C, CH, H, D, HID)
                  : align256(2 * (2 * (4 * CH * C + C * C + C * CH + 5 * H * D * C) + 3 * C * HID));
  }
};
struct BlockWeights {
  const void* w[OF3_PAIR_BLOCK_WEIGHTS];
  of3::WeightX3 split[of3::SplitJobs::kBlock];
  const of3::WeightX3 *mul, *att, *tr;
  const void* tr_operands[3];  // bf16 transition, beside w
  int packed;
};

// Prepares the matrices of n <= kPrepared blocks at dst by one launch (4 to 5 us however many they are)
constexpr int kPrepared = of3::PackJobs::kMax / of3::PackJobs::kBlock;
static_assert(kPrepared * of3::SplitJobs::kBlock <= of3::SplitJobs::kMax, "");
static hipError_t prepare_blocks(const void* const* const* weights, int n, const BlockDims& k, const float* mask, const int64_t mask_strides[3],
                                 void* dst, BlockWeights* out, hipStream_t stream) {
  const int64_t C = k.C, CH = k.CH, HD = k.H * k.D;
  if (k.wide()) {
    of3::WeightSplitter splitter(dst);
    auto f = [](const void* p) { return static_cast<const float*>(p); };
    for (int q = 0; q < n; ++q) {
      BlockWeights& o = out[q];
      for (int i = 0; i < k.weights(); ++i) o.w[i] = weights[q][i];
      o.packed = 0;
      o.mul = o.att = o.tr = nullptr;
      splitter.w = reinterpret_cast<of3::bf16_t*>(static_cast<char*>(dst) + q * k.prepared_bytes());
      of3::WeightX3* next = o.split;
      if (of3::trimul_split_widths(C, CH)) {
        o.mul = next;
        for (int d = 0; d < 2; ++d, next += of3::kTrimulMatrices) {
          const void* const* w = o.w + 10 * d;
          of3::TrimulF32Args a;
          a.ln_in_w = f(w[0]), a.ln_in_b = f(w[1]), a.ln_out_w = f(w[2]), a.ln_out_b = f(w[3]);
          a.w_ap = f(w[4]), a.w_ag = f(w[5]), a.w_bp = f(w[6]), a.w_bg = f(w[7]), a.w_g = f(w[8]), a.w_z = f(w[9]);
          a.C = (int)C, a.CH = (int)CH, a.B = (int)k.B, a.N = (int)k.N;
          a.mask = mask;
          a.mask_view = mask_view(mask, mask_strides, false);
          of3::trimul_split_jobs(splitter, a, k.rows16 && of3::trimul_half_shapes(k.B, k.N, C, CH), next);
        }
      }
      if (of3::triattn_split_widths(C, k.H, k.D)) {
        o.att = next;
        for (int d = 0; d < 2; ++d, next += of3::kTriattnMatrices) {
          const void* const* w = o.w + 20 + 8 * d;
          of3::TriattnF32Args a;
          a.ln_w = f(w[0]), a.ln_b = f(w[1]);
          a.w_q = f(w[3]), a.w_k = f(w[4]), a.w_v = f(w[5]), a.w_g = f(w[6]), a.w_o = f(w[7]);
          a.C = (int)C, a.H = (int)k.H, a.D = (int)k.D, a.inf = k.inf;
          of3::triattn_split_jobs(splitter, a, k.rows16 && of3::triattn_half_shapes(k.B, k.N, C, k.H, k.D), next);
        }
      }
      if (k.HID && of3::transition_split_widths(C, k.HID)) {
        o.tr = next;
        of3::TransitionF32Args a;
        a.ln_w = f(o.w[36]), a.ln_b = f(o.w[37]);
        a.w_a = f(o.w[38]), a.w_b = f(o.w[39]), a.w_out = f(o.w[40]);
        a.C = (int)C, a.HID = (int)k.HID;
        of3::transition_split_jobs(splitter, a, k.rows16 && of3::transition_half_shapes(k.B, k.N, C, k.HID), next);
      }
    }
    return splitter.j.n > 0 ? splitter.launch(stream) : hipSuccess;
  }
  of3::PackJobs jobs;
  jobs.n = jobs.first[0] = 0;
  for (int q = 0; q < n; ++q) {
    BlockWeights& o = out[q];
    for (int i = 0; i < k.weights(); ++i) o.w[i] = weights[q][i];
    o.packed = 1;
    o.mul = o.att = o.tr = nullptr;
    of3::bf16_t* to = reinterpret_cast<of3::bf16_t*>(static_cast<char*>(dst) + q * k.prepared_bytes());
    auto add_to = [&](const void*& packed, int i, int64_t rows, int64_t K) {
      const int m = jobs.n++;
      jobs.src[m] = bf(o.w[i]);
      jobs.dst[m] = to;
      jobs.K[m] = (int)K;
      jobs.first[m + 1] = jobs.first[m] + (int)(rows * K / 8);
      packed = to;
      to += rows * K;
    };
    auto add = [&](int i, int64_t rows, int64_t K) { add_to(o.w[i], i, rows, K); };
    for (int d = 0; d < 2; ++d) {
      for (int i = 4; i < 8; ++i) add(10 * d + i, CH, C);
      add(10 * d + 8, C, C);
      add(10 * d + 9, C, CH);
    }
    for (int d = 0; d < 2; ++d) {
      for (int i = 3; i < 7; ++i) add(20 + 8 * d + i, HD, C);
      add(20 + 8 * d + 7, C, HD);
    }
    for (int i = 0; i < 3; ++i) o.tr_operands[i] = nullptr;
    if (k.HID)
      for (int i = 0; i < 3; ++i) add_to(o.tr_operands[i], 38 + i, i < 2 ? k.HID : C, i < 2 ? C : k.HID);
  }
  return of3::pack_weights_launch(jobs, stream);
}

// bias: where the launches allow it, the pair bias of the result goes with the last of them (*bias_done).  Its output may be the beginning of
// the workspace, no larger than a triangle multiplication's planes (bf16) or an attention's q, k and v (fp32): none of these is read by then.
static int run_pair_block(const BlockWeights& k, const BlockDims& d, const void* z, const int64_t z_strides[3],
                          const float* mask, const int64_t mask_strides[3], void* out, int flags, void* workspace,
                          int64_t workspace_bytes, void* stream, const BlockBias* bias = nullptr, bool* bias_done = nullptr) {
  const void* src = z;  // the first module reads z, every later one updates out in place
  int rows = 0;
  if (k.packed && d.CH == d.C && d.H == 4 && 4 * d.D == d.C && join_room(d.dtype, d.B, d.N)) {
    const hipError_t e = of3::join_rows((int)d.B, (int)d.N, (int)d.C, &rows);
    if (e != hipSuccess) return fail_hip(e);
    const int variant = contract_variant_auto(d.B * d.CH, padded(d.N));
    if (variant != 2 && variant != 3) rows = 0;  // has no transposed form
  }
  const bool joined = rows > 0, attention_first = flags & OF3_BLOCK_ATTENTION_FIRST;
  const int64_t skip = joined ? of3_trimul_workspace_bytes(d.B, d.N, d.C, d.CH) : 0;
  ModuleEnd ends[2];
  int module = 0;  // of the four
  // the end of the module before, and where this one leaves its own
  auto before = [&] { return joined && module > 0 ? &ends[(module - 1) & 1] : nullptr; };
  bool last_joined = false;  // the last module with the transition
  auto after = [&] { return (joined && module < 3) || (last_joined && module == 3) ? &ends[module & 1] : nullptr; };
  auto trimul = [&](int m) {
    const void* const* w = k.w + 10 * m;
    const int st = trimul_fwd(k.mul ? k.mul + m * of3::kTrimulMatrices : nullptr, k.packed, src, z_strides, mask, mask_strides,
                              w[0], w[1], w[2], w[3], w[4], w[5], w[6], w[7], w[8], w[9], out, d.B, d.N, d.C, d.CH, m == 0,
                              1, workspace, workspace_bytes, d.dtype, stream, before(), after(), joined && m == 0);
    src = out;
    ++module;
    return st;
  };
  auto triattn = [&](int m) {
    const void* const* w = k.w + 20 + 8 * m;
    const int64_t zt[3] = {z_strides[0], m ? z_strides[2] : z_strides[1], m ? z_strides[1] : z_strides[2]};
    int64_t mt[3] = {0, 0, 0};
    if (mask) mt[0] = mask_strides[0], mt[1] = mask_strides[m ? 2 : 1], mt[2] = mask_strides[m ? 1 : 2];
    const int st = triattn_fwd(k.att ? k.att + m * of3::kTriattnMatrices : nullptr, k.packed, src, zt, mask, mt, w[0], w[1],
                               w[2], w[3], w[4], w[5], w[6], w[7], out, d.B, d.N, d.C, d.H, d.D, d.inf, 1,
                               static_cast<char*>(workspace) + skip, workspace_bytes - skip, d.dtype, stream, before(), after());
    src = out;
    ++module;
    return st;
  };
  auto transition = [&](const ModuleEnd* end, bool* takes_end) {
    const void* const* w = k.w + 36;
    return transition_fwd(k.tr, d.wide() ? nullptr : k.tr_operands, out, z_strides, flags & OF3_BLOCK_TRANSITION_UNMASKED ? nullptr : mask,
                          mask_strides, w[0], w[1], w[2], w[3], w[4], out, d.B, d.N, d.C, d.HID, 1, d.wide() ? workspace : nullptr,
                          d.wide() ? workspace_bytes : 0, d.dtype, stream, end, takes_end, end ? bias : nullptr, bias_done);
  };
  int st = OF3_OK;
  if (joined && !attention_first && d.HID != 0) st = transition(nullptr, &last_joined);
  if (d.wide() && k.tr && !attention_first && d.HID != 0) last_joined = true;  // if both can; else transition_fwd_f32 takes them one by one
  for (int part = 0; part < 2; ++part)
    for (int m = 0; m < 2 && st == OF3_OK; ++m)
      st = (part == 0) == !attention_first ? trimul(m) : triattn(m);
  if (st != OF3_OK || d.HID == 0) return st;
  return transition(last_joined ? &ends[3 & 1] : nullptr, nullptr);
}

// what a block's call checks before its first launch: a block is updated in place, half of one is of no use
static bool pair_block_args_ok(const BlockDims& d, const void* const* weights, const void* z, const int64_t z_strides[3],
                               const float* mask, const int64_t mask_strides[3], const void* out, const void* workspace) {
  if (!weights || !z || !out || !mask_ok(mask, mask_strides)) return false;
  if (d.wide() ? !f32_strides_ok(z_strides) : !strides_ok(z_strides)) return false;
  if (!workspace || (reinterpret_cast<uintptr_t>(workspace) & 255u)) return false;
  for (int i = 0; i < d.weights(); ++i)
    if (!weights[i] || !(d.wide() ? aligned4(weights[i]) : aligned16(weights[i]))) return false;
  return d.wide() ? aligned4(z) && aligned4(out) : aligned16(z) && aligned16(out);
}

static bool rows16(const void* z, const void* out, const int64_t z_strides[3]) {
  return aligned16(z) && aligned16(out) && ((z_strides[0] | z_strides[1] | z_strides[2]) & 3) == 0 &&
         of3::near_rows(z_strides[1], z_strides[2]);
}

int64_t of3_pair_block_workspace_bytes(int dtype, int64_t B, int64_t N, int64_t C, int64_t CH, int64_t H, int64_t D,
                                       int64_t HID) {
  const int64_t need = pair_block_module_bytes(dtype, B, N, C, CH, H, D, HID);
  const BlockDims d = {dtype, B, N, C, CH, H, D, HID, 0.f};
  return need < 0 ? need : need + d.prepared_bytes();
}

static int pair_block_fwd(const void* const* weights, const void* z, const int64_t z_strides[3], const float* mask,
                          const int64_t mask_strides[3], void* out, int64_t B, int64_t N, int64_t C, int64_t CH, int64_t H,
                          int64_t D, int64_t HID, float inf, int flags, void* workspace, int64_t workspace_bytes, int dtype,
                          void* stream, const BlockBias* bias = nullptr, bool* bias_done = nullptr) {
  const int64_t need = of3_pair_block_workspace_bytes(dtype, B, N, C, CH, H, D, HID);
  BlockDims d = {dtype, B, N, C, CH, H, D, HID, inf};
  if (need < 0 || !pair_block_args_ok(d, weights, z, z_strides, mask, mask_strides, out, workspace)) return OF3_EINVAL;
  if (workspace_bytes < need) return OF3_ENOSPC;
  d.rows16 = rows16(z, out, z_strides);
  BlockWeights k;
  const hipError_t e = prepare_blocks(&weights, 1, d, mask, mask_strides, static_cast<char*>(workspace) + need - d.prepared_bytes(), &k,
                                      static_cast<hipStream_t>(stream));
  if (e != hipSuccess) return fail_hip(e);
  return run_pair_block(k, d, z, z_strides, mask, mask_strides, out, flags, workspace, workspace_bytes, stream, bias, bias_done);
}
int of3_pair_block_fwd(const void* const* weights, const void* z, const int64_t z_strides[3], const float* mask,
                       const int64_t mask_strides[3], void* out, int64_t B, int64_t N, int64_t C, int64_t CH, int64_t H,
                       int64_t D, int64_t HID, float inf, int flags, void* workspace, int64_t workspace_bytes, int dtype,
                       void* stream) {
  return pair_block_fwd(weights, z, z_strides, mask, mask_strides, out, B, N, C, CH, H, D, HID, inf, flags, workspace, workspace_bytes, dtype,
                        stream);
}

int64_t of3_pairformer_block_workspace_bytes(int dtype, int64_t B, int64_t N, int64_t C, int64_t CH, int64_t H, int64_t D,
                                             int64_t HID, int64_t C_s, int64_t H_s, int64_t D_s, int64_t HID_s) {
  int64_t need = of3_pair_block_workspace_bytes(dtype, B, N, C, CH, H, D, HID);
  const int64_t attn = of3_attn_pair_bias_workspace_bytes_for(dtype, B, N, C_s, H_s, D_s);
  const int64_t rows = of3_transition_rows_fast_workspace_bytes(dtype, B * N, C_s, HID_s);
  if (need < 0 || attn < 0 || rows < 0 || HID < 1 || H_s > (dtype == OF3_DTYPE_BF16 ? 32 : 64)) return OF3_EINVAL;
  const int64_t single = align256(B * H_s * N * N * (dtype == OF3_DTYPE_BF16 ? 2 : 4)) + attn;  // the pair bias, then its consumer's
  if (single > need) need = single;
  return rows > need ? rows : need;
}

// A block's pair bias, to go with its last pair launch; what of3_pair_bias_fwd would refuse, or the launch cannot take, is left to that call
static bool block_bias_args(const BlockDims& d, const void* const* ws_, int64_t H_s, const void* z, const int64_t z_strides[3], void* out,
                            BlockBias* bias) {
  if (d.C != 128 || H_s < 1 || H_s > 32 || !ws_[0] || !ws_[2] || !out) return false;
  if (!aligned16(ws_[0]) || !aligned16(ws_[1]) || !aligned16(ws_[2]) || !aligned16(out)) return false;
  if (d.wide()) {
    of3::PairBiasF32Args* a = &bias->f32;
    a->z = static_cast<const float*>(z);
    a->z_view = view(z_strides, false);
    a->ln_w = static_cast<const float*>(ws_[0]);
    a->ln_b = static_cast<const float*>(ws_[1]);
    a->w = static_cast<const float*>(ws_[2]);
    a->out = static_cast<float*>(out);
    a->B = (int)d.B;
    a->N = (int)d.N;
    a->C = (int)d.C;
    a->H = (int)H_s;
    return true;
  }
  of3::PairBiasArgs* a = &bias->bf16;
  a->z = nullptr;  // the launch's own result
  a->ln_w = bf(ws_[0]);
  a->ln_b = bf(ws_[1]);
  a->w = bf(ws_[2]);
  a->out = bf(out);
  a->B = (int)d.B;
  a->N = (int)d.N;
  a->H = (int)H_s;
  return true;
}

static bool single_args_ok(const BlockDims& d, const void* const* w, const void* s, const void* s_out, const float* single_mask) {
  for (int i = 0; i < OF3_PAIRFORMER_BLOCK_WEIGHTS - OF3_PAIR_BLOCK_WEIGHTS; ++i)
    if ((!w[i] && i != 1) || !(d.wide() ? aligned4(w[i]) : aligned16(w[i]))) return false;  // 1: no offset
  if (!s || !s_out || !(d.wide() ? aligned4(s) && aligned4(s_out) : aligned16(s) && aligned16(s_out))) return false;
  return !single_mask || aligned4(single_mask);
}

int of3_pairformer_block_fwd(const void* const* weights, const void* s, const void* z, const int64_t z_strides[3],
                             const float* single_mask, const float* pair_mask, const int64_t mask_strides[3], void* s_out,
                             void* z_out, int64_t B, int64_t N, int64_t C, int64_t CH, int64_t H, int64_t D, int64_t HID,
                             int64_t C_s, int64_t H_s, int64_t D_s, int64_t HID_s, float inf, float inf_s, int flags,
                             void* workspace, int64_t workspace_bytes, int dtype, void* stream) {
  const int64_t need = of3_pairformer_block_workspace_bytes(dtype, B, N, C, CH, H, D, HID, C_s, H_s, D_s, HID_s);
  const BlockDims d = {dtype, B, N, C, CH, H, D, HID, inf};
  if (need < 0 || B > 65535 || N > (1 << 16) || !weights) return OF3_EINVAL;
  const void* const* ws_ = weights + OF3_PAIR_BLOCK_WEIGHTS;
  if (!single_args_ok(d, ws_, s, s_out, single_mask)) return OF3_EINVAL;
  if (workspace_bytes < need) return OF3_ENOSPC;
  BlockBias bias;
  bool bias_done = false;
  const bool with_bias = block_bias_args(d, ws_, H_s, z_out, z_strides, workspace, &bias);
  int st = pair_block_fwd(weights, z, z_strides, pair_mask, mask_strides, z_out, B, N, C, CH, H, D, HID, inf, flags,
                          workspace, workspace_bytes, dtype, stream, with_bias ? &bias : nullptr, &bias_done);
  if (st != OF3_OK) return st;
  const int64_t bias_bytes = align256(B * H_s * N * N * (d.wide() ? 4 : 2));
  if (!bias_done) st = of3_pair_bias_fwd(z_out, z_strides, ws_[0], ws_[1], ws_[2], workspace, B, N, C, H_s, dtype, stream);
  if (st != OF3_OK) return st;
  st = of3_attn_pair_bias_fwd(s, workspace, single_mask, ws_[3], ws_[4], ws_[5], ws_[6], ws_[7], ws_[8], ws_[9], ws_[10],
                              s_out, B, N, C_s, H_s, D_s, inf_s, 1, static_cast<char*>(workspace) + bias_bytes,
                              workspace_bytes - bias_bytes, dtype, stream);
  if (st != OF3_OK) return st;
  return of3_transition_rows_fwd(s_out, flags & OF3_BLOCK_TRANSITION_UNMASKED ? nullptr : single_mask, ws_[11], ws_[12],
                                 ws_[13], ws_[14], ws_[15], s_out, B * N, C_s, HID_s, 1, workspace, workspace_bytes, dtype,
                                 stream);
}

// ---- a stack of PairFormerBlocks in one call --------------------------------------------------
// The pair representation of block i + 1 needs nothing of block i's single representation: with a second stream the
// attention and transition of s (33 us per block at 40 tokens, of 102) run beside the next block's pair updates, which
// do not fill the chip at the lengths where that time counts.

// Two streams of one call and the order between them; without a second stream nothing to order.  An event waited for on
// another stream costs the host 15 us, five launches, so there are as few as can be.
class StreamPair {
 public:
  enum { kBias, kFree, kJoin, kEvents };
  StreamPair(hipStream_t main, hipStream_t side) : main(main), side(side ? side : main) {}
  ~StreamPair() {
    if (open_) join();
    for (hipEvent_t e : events_)
      if (e) (void)hipEventDestroy(e);  // released once the work recorded in it is done
  }
  // what is issued to `to` from now on waits for what `from` has been given so far
  int order(hipStream_t from, hipStream_t to, int event) {
    const int st = record(from, event);
    return st == OF3_OK ? wait(to, event) : st;
  }
  int record(hipStream_t from, int event) {
    if (main == side) return OF3_OK;
    hipError_t e = hipSuccess;
    // both streams are one device's: the fence that makes results visible to the host is not needed
    if (!events_[event]) e = hipEventCreateWithFlags(&events_[event], hipEventDisableTiming | hipEventDisableSystemFence);
    if (e == hipSuccess) e = hipEventRecord(events_[event], from);
    return e == hipSuccess ? OF3_OK : fail_hip(e);
  }
  int wait(hipStream_t to, int event) {
    if (main == side) return OF3_OK;
    open_ |= to == side;
    const hipError_t e = hipStreamWaitEvent(to, events_[event], 0);
    return e == hipSuccess ? OF3_OK : fail_hip(e);
  }
  int join() {
    if (!open_) return OF3_OK;
    open_ = false;
    return order(side, main, kJoin);
  }
  const hipStream_t main, side;

 private:
  hipEvent_t events_[kEvents] = {};
  bool open_ = false;  // the side stream holds work that main does not wait for yet
};

// regions of a stack's workspace
struct StackSpace {
  int64_t module, prepared, bias, single, total;
  // pair biases: one per block up to 64 MB of them.  Above 32 MB it is one, as in the single block's call: the attention that
  // reads it is over long before the next block's pair updates are (six blocks at N = 1100, bf16, one / two of them:
  // 32.2 / 32.2 ms, 1357 / 1395 MB; four at N = 1024, fp32: 65.4 / 65.4 ms, 3058 / 3126 MB).
  int64_t buffers;
};
static StackSpace stack_space(const BlockDims& d, int64_t blocks, int64_t C_s, int64_t H_s, int64_t D_s, int64_t HID_s) {
  StackSpace w;
  const int64_t attn = of3_attn_pair_bias_workspace_bytes_for(d.dtype, d.B, d.N, C_s, H_s, D_s);
  const int64_t rows = of3_transition_rows_fast_workspace_bytes(d.dtype, d.B * d.N, C_s, HID_s);
  w.module = pair_block_module_bytes(d.dtype, d.B, d.N, d.C, d.CH, d.H, d.D, d.HID);
  w.total = OF3_EINVAL;
  if (w.module < 0 || attn < 0 || rows < 0 || d.HID < 1 || H_s > (d.wide() ? 64 : 32) || blocks < 1) return w;
  w.module = align256(w.module);
  w.prepared = d.prepared_bytes() * (blocks < kPrepared ? blocks : kPrepared);
  w.bias = align256(d.B * H_s * d.N * d.N * (d.wide() ? 4 : 2));
  w.buffers = (64ll << 20) / w.bias;
  if (w.buffers < 1) w.buffers = 1;
  if (w.buffers > blocks) w.buffers = blocks;
  w.single = align256(attn > rows ? attn : rows);
  w.total = w.module + w.prepared + w.buffers * w.bias + w.single;
  return w;
}

int64_t of3_pairformer_stack_workspace_bytes(int dtype, int64_t blocks, int64_t B, int64_t N, int64_t C, int64_t CH,
                                             int64_t H, int64_t D, int64_t HID, int64_t C_s, int64_t H_s, int64_t D_s,
                                             int64_t HID_s) {
  const BlockDims d = {dtype, B, N, C, CH, H, D, HID, 0.f};
  return stack_space(d, blocks, C_s, H_s, D_s, HID_s).total;
}

int of3_pairformer_stack_fwd(const void* const* const* weights, int64_t blocks, const void* s, const void* z,
                             const int64_t z_strides[3], const float* single_mask, const float* pair_mask,
                             const int64_t mask_strides[3], void* s_out, void* z_out, int64_t B, int64_t N, int64_t C,
                             int64_t CH, int64_t H, int64_t D, int64_t HID, int64_t C_s, int64_t H_s, int64_t D_s,
                             int64_t HID_s, float inf, float inf_s, int flags, void* workspace, int64_t workspace_bytes,
                             int dtype, void* stream, void* side_stream) {
  BlockDims d = {dtype, B, N, C, CH, H, D, HID, inf};
  const StackSpace w = stack_space(d, blocks, C_s, H_s, D_s, HID_s);
  if (w.total < 0 || B > 65535 || N > (1 << 16) || !weights) return OF3_EINVAL;
  for (int64_t i = 0; i < blocks; ++i)
    if (!pair_block_args_ok(d, weights[i], z, z_strides, pair_mask, mask_strides, z_out, workspace) ||
        !single_args_ok(d, weights[i] + OF3_PAIR_BLOCK_WEIGHTS, s, s_out, single_mask))
      return OF3_EINVAL;
  if (workspace_bytes < w.total) return OF3_ENOSPC;
  d.rows16 = rows16(z, z_out, z_strides);
  char* const prepared = static_cast<char*>(workspace) + w.module;
  char* const bias0 = prepared + w.prepared;
  char* const single = bias0 + w.buffers * w.bias;

  // block j overwrites the bias that attention j - buffers reads, and waits for attention j - ahead or the one after it
  const int64_t ahead = w.buffers < 2 ? w.buffers : 2;
  StreamPair streams(static_cast<hipStream_t>(stream), static_cast<hipStream_t>(side_stream));
  // Where every block has a bias of its own, s of two blocks goes to the side stream together, behind one wait in place of two, as long as two more pair
  // updates follow: beside one alone it may end later (three blocks, waited for, one wait a block / for two, us: N = 40 310 / 329, 200 678 / 696).  Pair
  // updates take longer than s of their block (68 us against 33 at 40 tokens), so behind two of them nothing is left over.  One wait a block / for two, us, calls one after
  // the other, bf16, where the host sets the pace: four blocks N = 16 343 / 331, 40 349 / 331, 64 350 / 332, eight at 40 657 / 614; further up no difference
  // (four at 130 557 / 558, at 200 802 / 804); fp32, four blocks, 16 437 / 434, 24 445 / 440.
  const bool pairs = streams.main != streams.side && w.buffers >= blocks;
  auto attention = [&](int64_t j, int phases, hipStream_t on) {
    const void* const* ws_ = weights[j] + OF3_PAIR_BLOCK_WEIGHTS;
    return attn_pair_bias(phases, j ? s_out : s, bias0 + (j % w.buffers) * w.bias, single_mask, ws_[3], ws_[4], ws_[5], ws_[6], ws_[7],
                          ws_[8], ws_[9], ws_[10], s_out, B, N, C_s, H_s, D_s, inf_s, 1, single, w.single, dtype, on);
  };
  auto transition = [&](int64_t j, hipStream_t on) {
    const void* const* ws_ = weights[j] + OF3_PAIR_BLOCK_WEIGHTS;
    return of3_transition_rows_fwd(s_out, flags & OF3_BLOCK_TRANSITION_UNMASKED ? nullptr : single_mask, ws_[11], ws_[12],
                                   ws_[13], ws_[14], ws_[15], s_out, B * N, C_s, HID_s, 1, single, w.single, dtype, on);
  };
  BlockWeights k[kPrepared];
  int64_t next = 0;  // the first block whose s has not been issued
  int st = OF3_OK;
  for (int64_t i = 0; i < blocks && st == OF3_OK; ++i) {
    const int q = (int)(i % kPrepared);
    const bool hold = pairs && i % 2 == 0 && i + 3 < blocks;  // s goes with the next block's
    const bool last = i + 1 == blocks;
    if (q == 0) {
      const int n = (int)(blocks - i < kPrepared ? blocks - i : kPrepared);
      const hipError_t e = prepare_blocks(weights + i, n, d, pair_mask, mask_strides, prepared, k, streams.main);
      if (e != hipSuccess) return fail_hip(e);
    }
    const void* const* ws_ = weights[i] + OF3_PAIR_BLOCK_WEIGHTS;
    void* const bias = bias0 + (i % w.buffers) * w.bias;
    BlockBias bias_args;
    bool bias_done = false;
    const bool with_bias = i < w.buffers && block_bias_args(d, ws_, H_s, z_out, z_strides, bias, &bias_args);  // else its buffer has to be waited for
    // the projections of s need no pair bias; those of the first block have nothing to wait behind on the side stream
    const bool projected = i > 0 && next == i && !hold;
    if (projected && (st = attention(i, of3::kSingleProject, streams.side)) != OF3_OK) break;
    st = run_pair_block(k[q], d, i ? z_out : z, z_strides, pair_mask, mask_strides, z_out, flags, workspace, w.module, streams.main,
                        with_bias ? &bias_args : nullptr, &bias_done);
    if (st != OF3_OK) break;
    // a buffer is used again: the attentions issued so far have read theirs
    if (i >= w.buffers && (st = streams.wait(streams.main, StreamPair::kFree)) != OF3_OK) break;
    if (!bias_done) st = of3_pair_bias_fwd(z_out, z_strides, ws_[0], ws_[1], ws_[2], bias, B, N, C, H_s, dtype, streams.main);
    if (st != OF3_OK) break;
    if (hold) continue;
    // the last block has nothing beside it: it goes on where its bias was written
    st = last ? streams.join() : streams.order(streams.main, streams.side, StreamPair::kBias);
    const hipStream_t on = last ? streams.main : streams.side;
    for (; st == OF3_OK && next <= i; ++next) {
      st = attention(next, next == i && projected ? of3::kSingleAttend : of3::kSingleProject | of3::kSingleAttend, on);
      if (st == OF3_OK && next + ahead < blocks && next + ahead >= w.buffers) st = streams.record(on, StreamPair::kFree);
      if (st == OF3_OK) st = transition(next, on);
    }
  }
  return st;
}

int of3_side_stream_create(void** stream) {
  if (!stream) return OF3_EINVAL;
  hipStream_t s = nullptr;
  const hipError_t e = hipStreamCreateWithFlags(&s, hipStreamNonBlocking);
  if (e != hipSuccess) {
    (void)hipGetLastError();  // the caller goes on with one stream
    return fail_hip(e);
  }
  *stream = s;
  return OF3_OK;
}

int of3_side_stream_destroy(void* stream) {
  if (!stream) return OF3_EINVAL;
  hipError_t e = hipStreamSynchronize(static_cast<hipStream_t>(stream));
  if (e == hipSuccess) e = hipStreamDestroy(static_cast<hipStream_t>(stream));
  return e == hipSuccess ? OF3_OK : fail_hip(e);
}

}  // extern "C"
