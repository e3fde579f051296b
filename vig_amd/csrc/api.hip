// C ABI of the library (declared in include/vig_gla.h): argument validation and
// dispatch only.  Nothing here allocates, frees or synchronises.
#include "../../include/vig_gla.h"
#include "launch.h"
#include <algorithm>
#include <mutex>

namespace vig {
int launch_dirgate(const void* in, void* out, int B, int L, int H, int Dk, float inv_norm, float clamp_min,
                   int in_dtype, int out_dtype, hipStream_t stream);
int launch_dirgate_bwd(const void* in, const void* d_out, void* d_in, int B, int L, int H, int Dk, float inv_norm,
                       float clamp_min, int in_dtype, int out_dtype, hipStream_t stream);
int launch_merge_heads(const void* dq, const void* dk, const void* dv, void* dqkv, int B, int L, int H, int Dk, int Dv,
                       long long ld, int io_dtype, hipStream_t stream);
size_t dwconv3x3_wgrad_workspace(int B, int C);
size_t dwconv3x3_wgrad_least_workspace(int B, int C);
int launch_dwconv3x3_bwd(const void* x, const void* dy, const void* pre, const float* wt, void* dx, float* dw_db,
                         void* workspace, size_t workspace_bytes, int B, int h, int w, int C, int io_dtype, vig_sum_jobs* later, hipStream_t stream);
int launch_dirgate_lowrank_bwd(const void* low, long long ld, const void* w1, const void* w1t, const void* b1,
                               const void* d_out, void* dx, void* d_low, long long ldd, int B, int L, int H, int Dk,
                               float inv_norm, float clamp_min, int out_dtype, hipStream_t stream);
bool linear_preferred(long long M, int N, int K);
int launch_linear(const void* x, long long ldx, const void* w, const void* bias, void* y, long long ldy, long long M, int N, int K,
                  hipStream_t stream);
int launch_conv3x3s2(const void* x, const void* w, void* y, int B, int H, int W, int Cin, int Cout, hipStream_t stream);
size_t rmsnorm_pool_workspace(int B, int L, int C);
int launch_rmsnorm_pool(const void* x, const void* residual, const float* weight, void* out, void* workspace, int B, int L, int C,
                        float eps, hipStream_t stream);
int launch_cast_many(const void* const* src, void* const* dst, const int* n, const int* cols, const int* src_dtype,
                     const int* dst_dtype, int count, hipStream_t stream);
int launch_dwconv3x3(const void* x, const float* wt, const float* bias, void* y, void* pre, int B, int h, int w, int C,
                     int silu, int io_dtype, hipStream_t stream);
int launch_dirgate_lowrank(const void* low, long long ld, const void* w1, const void* b1, void* out, int B, int L,
                           int H, int Dk, int rank, float inv_norm, float clamp_min, int in_dtype, int out_dtype,
                           hipStream_t stream);
int launch_locality_gate(const void* o, const float* wt, void* y, int B, int H, int h, int w, int Dv, int io_dtype,
                         hipStream_t stream);
int launch_locality_blend(const void* o, const void* loc, const void* glin, const float* wg, const float* wl, void* y,
                          int B, int H, int L, int Dv, long long ldg, float eps, int silu_out, int io_dtype,
                          hipStream_t stream);
size_t locality_blend_bwd_workspace(int B, int L, int Dv);
size_t locality_blend_bwd_least_workspace(int B, int L, int Dv);
int launch_locality_blend_bwd(const void* o, const void* loc, const void* glin, const float* wg, const float* wl,
                              const void* dy, void* d_o, void* d_loc, void* d_glin, float* dw, void* workspace, long long workspace_rows, int B,
                              int H, int L, int Dv, long long ldg, long long ldd, float eps, int silu_out, int io_dtype,
                              vig_sum_jobs* later, hipStream_t stream);
bool rmsnorm_types_ok(int x_dtype, int sum_dtype, int y_dtype);
int launch_rmsnorm(const void* x, const void* residual, const float* weight, void* y, void* residual_out, int rows,
                   int C, float eps, int round_sum, int x_dtype, int sum_dtype, int y_dtype, hipStream_t stream);
int launch_layernorm(const void* x, const float* weight, const float* bias, void* y, long long rows, int C, float eps,
                     int silu, const float* pre_bias, const void* post_add, int post_rows, int io_dtype,
                     hipStream_t stream);
int launch_split_heads(const void* qkv, void* q, void* k, void* v, int B, int L, int H, int Dk, int Dv, long long ld,
                       int io_dtype, hipStream_t stream);
int launch_swiglu(const void* in, void* out, long long rows, int I, int io_dtype, hipStream_t stream);
int launch_swiglu_bwd(const void* in, const void* dy, void* din, long long rows, int I, int io_dtype,
                      hipStream_t stream);
size_t rmsnorm_bwd_workspace(long long rows, int C);
int launch_rmsnorm_bwd(const void* s, const float* weight, const void* dy, const void* d_sum, void* ds, void* dx, float* dweight,
                       void* workspace, long long rows, int C, float eps, int sum_dtype, int y_dtype, vig_sum_jobs* later, hipStream_t stream);
bool blend_linear_supported(int H, int Dv, int C);
int launch_blend_linear(const void* o, const void* loc, const void* glin, const float* w_g, const float* w_l,
                        const void* W, void* out, void* kept, int B, int H, int L, int Dv, int C, long long ldg, float eps,
                        int silu_out, hipStream_t stream);
bool linear_swiglu_supported(int K, int I);
int launch_linear_swiglu(const void* A, const void* W, void* out, void* kept, long long T, int K, int I, hipStream_t stream);
bool patch_conv_supported(int Cin, int H, int W, int KH, int KW, int stride, int padding, int Cout);
int launch_patch_conv(const void* x, const void* w_packed, void* y, int B, int Cin, int H, int W, int KH, int KW,
                      int Cout, hipStream_t stream);
bool stem_norm_supported(long long rows, int C, int x_dtype, int y_dtype);
size_t stem_norm_bwd_workspace(long long rows, int C);
int launch_stem_norm(const void* x, const float* pre, const float* w, const float* b, void* y, long long rows, int C, float eps, int silu,
                     int x_dtype, int y_dtype, hipStream_t stream);
int launch_stem_norm_bwd(const void* x, const float* pre, const float* w, const float* b, const void* dy, void* dx, float* dparams, void* workspace,
                         long long rows, int C, float eps, int silu, int x_dtype, int y_dtype, hipStream_t stream);
int launch_patch_conv_norm(const void* x, const void* w_packed, const float* weight, const float* bias, const float* pre_bias, void* y, int B,
                           int Cin, int H, int W, int KH, int KW, int Cout, float eps, int silu, hipStream_t stream);
int launch_pad_channels(const void* src, void* dst, long long rows, int src_c, int dst_c, hipStream_t stream);
int launch_pad_channels_multi(const void* const* src, void* const* dst, const int* src_c, const int* dst_c, int n,
                              long long rows, hipStream_t stream);
int launch_gla_backward(const void* q, const void* k, const void* v, const void* g_fwd, const void* g_bwd,
                        const void* d_o, void* dq, void* dk, void* dv, void* dg_fwd, void* dg_bwd, void* workspace,
                        int B, int H, int L, int Dk, int Dv, float scale, float out_scale, int io_dtype,
                        int gate_dtype, bool exact, size_t beyond, hipStream_t stream, long long ld_in = 0, long long ld_out = 0);
bool gla_backward_in_place(int L, int Dk, int Dv, int io_dtype, int gate_dtype, bool bidir);
size_t gla_backward_workspace(int B, int H, int L, int Dk, int Dv, int bidir);  // (launch_gla_backward's; `beyond`: bytes behind it)
bool linear_wgrad_supported(long long T, int N, int K);
size_t matmul_f32_workspace(long long M, int N, long long K);
bool matmul_f32_supported(long long lda, bool ta, long long ldb, bool tb, long long M, int N, long long K);
int launch_matmul_f32(const float* a, long long lda, bool ta, const float* b, long long ldb, bool tb, const float* bias, const float* add,
                      long long ldadd, float* out, long long ldo, float* a_sums, long long M, int N, long long K, void* workspace,
                      hipStream_t stream);
}  // namespace vig

static bool dtype_ok(int d) { return d == VIG_F32 || d == VIG_BF16; }

// rows read with 16-byte vector loads: the base and the distance between rows have to keep that alignment
static bool strided_rows_ok(const void* base, long long ld_elems, int dtype) {
  const long long elem = dtype == VIG_BF16 ? 2 : 4;
  return (reinterpret_cast<uintptr_t>(base) % 16) == 0 && (ld_elems * elem) % 16 == 0;
}
// whether a list of sums put off (none: they run at once) takes n more
static bool room_for(const vig_sum_jobs* later, int n) { return !later || (later->count >= 0 && later->count <= VIG_SUM_JOBS - n); }
// every tensor is moved 16 bytes per access: a pointer off that boundary is refused (null, for an optional tensor, passes)
template <typename... P>
static bool aligned16(P... p) {
  return ((reinterpret_cast<uintptr_t>(static_cast<const void*>(p)) % 16 == 0) && ...);
}
static bool dk_ok(int d) { return d == 16 || d == 32 || d == 64 || d == 128; }
static bool dv_ok(int d) { return d == 32 || d == 64 || d == 128; }

extern "C" {

const char* vig_gla_version(void) { return "vig_gla 0.1 gfx950"; }

const char* vig_gla_strerror(int code) {
  switch (code) {
    case VIG_OK: return "ok";
    case VIG_EINVAL: return "invalid argument";
    case VIG_ENOTSUP: return "shape or dtype combination not built";
    case VIG_ENOSPC: return "workspace too small";
    case VIG_ELAUNCH: return "HIP launch error";
    default: return "unknown error";
  }
}

static int fill_args(vig::GlaArgs& a, const void* q, const void* k, const void* v, const void* g_fwd,
                     const void* g_bwd, void* o, void* workspace, size_t workspace_bytes, int B, int H, int L,
                     int Dk, int Dv, float scale, float out_scale, int io_dtype, int gate_dtype, void* stream) {
  if (!q || !k || !v || !g_fwd || !o) return VIG_EINVAL;
  if (!aligned16(q, k, v, g_fwd, g_bwd, o, workspace)) return VIG_EINVAL;
  if (B <= 0 || H <= 0 || L <= 0) return VIG_EINVAL;
  if ((long long)B * H > 2147483647LL) return VIG_EINVAL;
  if (!dtype_ok(io_dtype) || !dtype_ok(gate_dtype)) return VIG_ENOTSUP;
  if (!dk_ok(Dk) || !dv_ok(Dv)) return VIG_ENOTSUP;
  a = vig::GlaArgs{q, k, v, g_fwd, g_bwd, o, workspace, workspace_bytes, B, H, L, Dk, Dv,
                   scale, out_scale, io_dtype, gate_dtype, (hipStream_t)stream};
  return VIG_OK;
}

// HierViG's head shape (Dk 16, Dv 32) rides the matrix-core kernel zero-padded to Dk 32 / Dv 64 once the sequence is
// long enough for that to beat the token-recurrent kernel (measured: 1.5x at L = 196, 10x at L = 3136).
constexpr int kPadMinL = 128;
static bool padded_shape(int L, int Dk, int Dv, int io_dtype, int gate_dtype, bool bidir) {
  return bidir && io_dtype == VIG_BF16 && gate_dtype == VIG_BF16 && Dk == 16 && Dv == 32 && L >= kPadMinL;
}
static size_t padded_elems_qk(int B, int H, int L) { return (size_t)B * H * L * 32; }
static size_t padded_elems_v(int B, int H, int L) { return (size_t)B * H * L * 64; }
static size_t padded_workspace(int B, int H, int L) {
  // q, k, g_fwd, g_bwd padded to 32 channels, v and o to 64, then the matrix-core kernel's own workspace
  return (4 * padded_elems_qk(B, H, L) + 2 * padded_elems_v(B, H, L)) * sizeof(uint16_t) +
         vig::gla_mfma_workspace(B, H, L, 32, 64);
}

// What the path vig_gla_bidir_fwd dispatches to for exactly these arguments needs.
static size_t fwd_workspace_exact(int B, int H, int L, int Dk, int Dv, int io_dtype, int gate_dtype, bool bidir) {
  if (io_dtype == VIG_BF16 && gate_dtype == VIG_BF16 && (Dk == 64 || Dk == 32) && Dv == 64)
    return vig::gla_mfma_workspace(B, H, L, Dk, Dv);
  if (io_dtype == VIG_F32 && gate_dtype == VIG_F32) return vig::gla_f32_workspace(B, H, L, Dk, Dv, bidir);
  if (padded_shape(L, Dk, Dv, io_dtype, gate_dtype, bidir)) return padded_workspace(B, H, L);
  return bidir ? vig::gla_recurrent_workspace(B, H, L, Dv, io_dtype) : 0;
}

size_t vig_gla_bidir_fwd_workspace_for(int B, int H, int L, int Dk, int Dv, int io_dtype, int gate_dtype,
                                       int bidirectional) {
  if (B <= 0 || H <= 0 || L <= 0 || !dtype_ok(io_dtype) || !dtype_ok(gate_dtype)) return 0;
  return fwd_workspace_exact(B, H, L, Dk, Dv, io_dtype, gate_dtype, bidirectional != 0);
}

size_t vig_gla_bidir_fwd_workspace(int B, int H, int L, int Dk, int Dv, int io_dtype) {
  if (B <= 0 || H <= 0 || L <= 0) return 0;
  // The largest requirement over the paths the dispatcher may take for this shape.
  size_t need = vig::gla_recurrent_workspace(B, H, L, Dv, io_dtype);
  if (padded_shape(L, Dk, Dv, io_dtype, VIG_BF16, true)) {
    const size_t p = padded_workspace(B, H, L);
    if (p > need) need = p;
  }
  if (io_dtype == VIG_BF16) {
    const size_t m = vig::gla_mfma_workspace(B, H, L, Dk, Dv);
    if (m > need) need = m;
  } else {
    // (without the room for the directions' halves of leftover whole sequences, a quicker form that no call needs)
    const size_t m = vig::gla_f32_workspace(B, H, L, Dk, Dv, false);
    if (m > need) need = m;
  }
  return need;
}

static int gla_bidir_fwd(const void* q, const void* k, const void* v, const void* g_fwd, const void* g_bwd, void* o,
                         void* workspace, size_t workspace_bytes, int B, int H, int L, int Dk, int Dv, float scale,
                         float out_scale, int io_dtype, int gate_dtype, void* stream, int wide_gates) {
  vig::GlaArgs a;
  const int rc = fill_args(a, q, k, v, g_fwd, g_bwd, o, workspace, workspace_bytes, B, H, L, Dk, Dv, scale,
                           out_scale, io_dtype, gate_dtype, stream);
  if (rc != VIG_OK) return rc;
  a.wide_gates = wide_gates;
  if (vig::gla_mfma_supported(a)) {
    // (the segment scan of long sequences puts sequence x direction on grid.y)
    if (L > 256 && (long long)B * H * (g_bwd ? 2 : 1) > 65535) return VIG_ENOTSUP;
    if (vig::gla_mfma_workspace(B, H, L, Dk, Dv) > workspace_bytes) return VIG_ENOSPC;
    if (vig::gla_mfma_workspace(B, H, L, Dk, Dv) > 0 && !workspace) return VIG_EINVAL;
    return vig::launch_gla_mfma(a);
  }
  if (padded_shape(L, Dk, Dv, io_dtype, gate_dtype, g_bwd != nullptr) && workspace &&
      workspace_bytes >= padded_workspace(B, H, L)) {
    // (a caller that sized the workspace for the recurrent kernel only still gets that kernel below)
    const size_t nqk = padded_elems_qk(B, H, L), nv = padded_elems_v(B, H, L);
    uint16_t* p = static_cast<uint16_t*>(workspace);
    uint16_t *qp = p, *kp = p + nqk, *gfp = p + 2 * nqk, *gbp = p + 3 * nqk, *vp = p + 4 * nqk, *op = vp + nv;
    const long long rows = (long long)B * H * L;
    hipStream_t st = (hipStream_t)stream;
    const void* srcs[5] = {q, k, g_fwd, g_bwd, v};
    void* dsts[5] = {qp, kp, gfp, gbp, vp};
    const int src_c[5] = {16, 16, 16, 16, 32}, dst_c[5] = {32, 32, 32, 32, 64};
    int e = vig::launch_pad_channels_multi(srcs, dsts, src_c, dst_c, 5, rows, st);
    if (e) return e;
    vig::GlaArgs b = a;
    b.q = qp, b.k = kp, b.v = vp, b.g_fwd = gfp, b.g_bwd = gbp, b.o = op;
    b.Dk = 32, b.Dv = 64;
    b.workspace = op + nv;
    b.workspace_bytes = vig::gla_mfma_workspace(B, H, L, 32, 64);
    e = vig::launch_gla_mfma(b);
    if (e) return e;
    return vig::launch_pad_channels(op, o, rows, 64, 32, st);
  }
  // fp32 on the matrix cores; a caller that brought no room for a long sequence's states gets the recurrent kernel
  if (vig::gla_f32_supported(a)) {
    const size_t n = vig::gla_f32_least_workspace(B, H, L, Dk, Dv);
    if (n == 0 || (workspace && workspace_bytes >= n)) return vig::launch_gla_f32(a);
  }
  const size_t need = g_bwd ? vig::gla_recurrent_workspace(B, H, L, Dv, io_dtype) : 0;
  if (need > workspace_bytes) return VIG_ENOSPC;
  if (need > 0 && !workspace) return VIG_EINVAL;
  return vig::launch_gla_recurrent(a);
}

int vig_gla_bidir_fwd(const void* q, const void* k, const void* v, const void* g_fwd, const void* g_bwd, void* o,
                      void* workspace, size_t workspace_bytes, int B, int H, int L, int Dk, int Dv, float scale,
                      float out_scale, int io_dtype, int gate_dtype, void* stream) {
  return gla_bidir_fwd(q, k, v, g_fwd, g_bwd, o, workspace, workspace_bytes, B, H, L, Dk, Dv, scale, out_scale,
                       io_dtype, gate_dtype, stream, 0);
}

// q, k, v read in place from wider rows (e.g. the column blocks of a stacked projection's output): the matrix-core slab
// kernel with the rows' pitches in scalar registers; no workspace.
int vig_gla_bidir_fwd_strided(const void* q, const void* k, const void* v, const void* g_fwd, const void* g_bwd, void* o,
                              int B, int H, int L, int Dk, int Dv, const long long* q_strides,
                              const long long* k_strides, const long long* v_strides, float scale, float out_scale,
                              int io_dtype, int gate_dtype, void* stream) {
  if (!q_strides || !k_strides || !v_strides) return VIG_EINVAL;
  vig::GlaArgs a;
  const int rc = fill_args(a, q, k, v, g_fwd, g_bwd, o, nullptr, 0, B, H, L, Dk, Dv, scale, out_scale, io_dtype,
                           gate_dtype, stream);
  if (rc != VIG_OK) return rc;
  if (!vig::gla_mfma_supported(a) || L > 256) return VIG_ENOTSUP;
  a.q_strides = q_strides, a.k_strides = k_strides, a.v_strides = v_strides;
  return vig::launch_gla_mfma(a);
}

// The one-launch kernel at every length it takes, with q, k, v in place and the locality gate as options; no workspace.
int vig_gla_slab_tokens(int Dk) { return Dk == 64 || Dk == 32 ? vig::gla_slab_tokens(Dk) : 0; }

int vig_gla_slab_fwd(const void* q, const void* k, const void* v, const void* g_fwd, const void* g_bwd, const float* gate_weight,
                     void* o, int B, int H, int L, int Dk, int Dv, const long long* q_strides, const long long* k_strides,
                     const long long* v_strides, int grid_h, int grid_w, float scale, float out_scale, int io_dtype,
                     int gate_dtype, void* stream) {
  vig::GlaArgs a;
  const int rc = fill_args(a, q, k, v, g_fwd, g_bwd, o, nullptr, 0, B, H, L, Dk, Dv, scale, out_scale, io_dtype, gate_dtype, stream);
  if (rc != VIG_OK) return rc;
  a.q_strides = q_strides, a.k_strides = k_strides, a.v_strides = v_strides;
  if (gate_weight) {
    if (!g_bwd || grid_h <= 0 || grid_w <= 0 || (long long)grid_h * grid_w != L || !aligned16(gate_weight)) return VIG_EINVAL;
    if (grid_w > 126) return VIG_ENOTSUP;  // (grids that vig_locality_gate_fwd takes: one op, whichever way it runs)
    a.gate_w = gate_weight, a.gate_rows = grid_h, a.gate_cols = grid_w;
  }
  return vig::gla_tiles_supported(a) ? vig::launch_gla_tiles(a) : VIG_ENOTSUP;
}

// The op with the gates made on the way from their rank-16 rows, q, k, v in place.
size_t vig_gla_lowrank_fwd_workspace(int B, int H, int L, int Dk, int Dv) {
  return B <= 0 || H <= 0 || L <= 0 || Dk != 32 || Dv != 64 || L <= vig::gla_slab_tokens(Dk) ? 0 : vig::gla_mfma_workspace(B, H, L, Dk, Dv);
}

int vig_gla_lowrank_fwd(const void* q, const void* k, const void* v, const void* low, long long low_row_stride, const void* up_w,
                        const void* up_b, void* o, void* workspace, size_t workspace_bytes, int B, int H, int L, int Dk, int Dv,
                        const long long* q_strides, const long long* k_strides, const long long* v_strides, float inv_norm,
                        float clamp_min, float scale, float out_scale, int io_dtype, void* stream) {
  vig::GlaArgs a;
  const int rc = fill_args(a, q, k, v, low, low, o, workspace, workspace_bytes, B, H, L, Dk, Dv, scale, out_scale, io_dtype, io_dtype, stream);
  if (rc != VIG_OK) return rc;
  if (!up_w || !up_b || !aligned16(up_w) || low_row_stride < 16 || !strided_rows_ok(low, low_row_stride, io_dtype)) return VIG_EINVAL;
  a.q_strides = q_strides, a.k_strides = k_strides, a.v_strides = v_strides;
  a.low = low, a.up_w = up_w, a.up_b = up_b, a.low_ld = low_row_stride, a.inv_norm = inv_norm, a.clamp = clamp_min;
  return vig::launch_gla_lowrank(a);
}

// The causal op with a state carried in and / or out.
static size_t causal_state_workspace(int B, int H, int L, int Dk, int Dv, int io_dtype, int gate_dtype) {
  if (io_dtype == VIG_BF16 && gate_dtype == VIG_BF16 && (Dk == 64 || Dk == 32) && Dv == 64)
    return vig::gla_mfma_state_workspace(B, H, L, Dk, Dv);
  return 0;  // the token-recurrent kernel keeps the state in registers
}

size_t vig_gla_causal_state_fwd_workspace(int B, int H, int L, int Dk, int Dv, int io_dtype, int gate_dtype) {
  if (B <= 0 || H <= 0 || L <= 0 || !dtype_ok(io_dtype) || !dtype_ok(gate_dtype)) return 0;
  return causal_state_workspace(B, H, L, Dk, Dv, io_dtype, gate_dtype);
}

static int causal_state_fwd(const void* q, const void* k, const void* v, const void* g, void* o,
                            const float* initial_state, float* final_state, void* workspace, size_t workspace_bytes,
                            int B, int H, int L, int Dk, int Dv, float scale, float out_scale, int io_dtype,
                            int gate_dtype, void* stream, bool exact) {
  vig::GlaArgs a;
  const int rc = fill_args(a, q, k, v, g, nullptr, o, workspace, workspace_bytes, B, H, L, Dk, Dv, scale, out_scale,
                           io_dtype, gate_dtype, stream);
  if (rc != VIG_OK) return rc;
  if (!aligned16(initial_state, final_state)) return VIG_EINVAL;
  a.init_state = initial_state;
  a.final_state = final_state;
  if (!exact && vig::gla_mfma_supported(a)) {
    if ((long long)B * H > 65535) return VIG_ENOTSUP;  // (the segment scan puts the sequences on grid.y)
    const size_t need = vig::gla_mfma_state_workspace(B, H, L, Dk, Dv);
    if (need > workspace_bytes) return VIG_ENOSPC;
    if (!workspace) return VIG_EINVAL;
    return vig::launch_gla_mfma(a);
  }
  return vig::launch_gla_recurrent(a);
}

int vig_gla_causal_state_fwd(const void* q, const void* k, const void* v, const void* g, void* o,
                             const float* initial_state, float* final_state, void* workspace, size_t workspace_bytes,
                             int B, int H, int L, int Dk, int Dv, float scale, float out_scale, int io_dtype,
                             int gate_dtype, void* stream) {
  return causal_state_fwd(q, k, v, g, o, initial_state, final_state, workspace, workspace_bytes, B, H, L, Dk, Dv, scale,
                          out_scale, io_dtype, gate_dtype, stream, false);
}

// Same contract, always the fp32-arithmetic token-recurrent kernel (no workspace).
int vig_gla_causal_state_fwd_exact(const void* q, const void* k, const void* v, const void* g, void* o,
                                   const float* initial_state, float* final_state, int B, int H, int L, int Dk, int Dv,
                                   float scale, float out_scale, int io_dtype, int gate_dtype, void* stream) {
  return causal_state_fwd(q, k, v, g, o, initial_state, final_state, nullptr, 0, B, H, L, Dk, Dv, scale, out_scale,
                          io_dtype, gate_dtype, stream, true);
}

// Same contract and results to the same bar; for callers whose gates are known to be strong (see the header).
int vig_gla_bidir_fwd_wide(const void* q, const void* k, const void* v, const void* g_fwd, const void* g_bwd, void* o,
                           void* workspace, size_t workspace_bytes, int B, int H, int L, int Dk, int Dv, float scale,
                           float out_scale, int io_dtype, int gate_dtype, void* stream) {
  return gla_bidir_fwd(q, k, v, g_fwd, g_bwd, o, workspace, workspace_bytes, B, H, L, Dk, Dv, scale, out_scale,
                       io_dtype, gate_dtype, stream, 1);
}

// ---- vig_gla_bidir_fwd for callers that cannot allocate: the workspace is a device array of this library ----
// One copy per GPU, held from the first launch of the library on that GPU until the process ends.
constexpr size_t kScratchBytes = VIG_GLA_NOALLOC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];
// The array's name is only a host-side handle: its address on each device is looked up once, with that device current.
constexpr int kScratchMaxDevices = 64;
static void* scratch_ptr[kScratchMaxDevices] = {};
static std::mutex scratch_mutex;

// `owned`: a device pointer of the call (q).  The array that serves a call is the one of the GPU that holds the
// call's tensors, which has to be the current device (the kernels are launched there, and the symbol lookup answers
// for the current device only): a caller on another device is refused instead of being handed the wrong GPU's array.
static int scratch_for_current_device(void** out, const void* owned) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kScratchMaxDevices) return VIG_ELAUNCH;
  hipPointerAttribute_t attr;
  if (hipPointerGetAttributes(&attr, owned) == hipSuccess) {
    if (attr.type == hipMemoryTypeDevice && attr.device != dev) return VIG_EINVAL;
  } else {
    (void)hipGetLastError();  // (an unregistered pointer: the launch itself will report it)
  }
  std::lock_guard<std::mutex> lock(scratch_mutex);
  if (!scratch_ptr[dev]) {
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return VIG_ELAUNCH;
    scratch_ptr[dev] = p;
  }
  *out = scratch_ptr[dev];
  return VIG_OK;
}

size_t vig_gla_bidir_fwd_noalloc_max_workspace(void) { return kScratchBytes; }

int vig_gla_bidir_fwd_noalloc(const void* q, const void* k, const void* v, const void* g_fwd, const void* g_bwd,
                              void* o, int B, int H, int L, int Dk, int Dv, float scale, float out_scale,
                              int io_dtype, int gate_dtype, void* stream) {
  if (B <= 0 || H <= 0 || L <= 0) return VIG_EINVAL;
  if (!dtype_ok(io_dtype) || !dtype_ok(gate_dtype)) return VIG_ENOTSUP;
  // what the dispatched path of vig_gla_bidir_fwd needs; shapes whose need exceeds the array are refused, not shrunk
  size_t need = fwd_workspace_exact(B, H, L, Dk, Dv, io_dtype, gate_dtype, g_bwd != nullptr);
  if (io_dtype == VIG_F32 && need > kScratchBytes) need = 0;  // (fp32 tensors: the recurrent kernel keeps its state in registers)
  if (need > kScratchBytes) return VIG_ENOSPC;
  void* ws = nullptr;
  if (need > 0) {
    const int rc = scratch_for_current_device(&ws, q);
    if (rc != VIG_OK) return rc;
  }
  // Every kernel behind vig_gla_bidir_fwd writes the part of the workspace it later reads (segment states, padded
  // copies, the reverse direction's partial outputs) before reading it: nothing has to start at zero.
  return gla_bidir_fwd(q, k, v, g_fwd, g_bwd, o, ws, need, B, H, L, Dk, Dv, scale, out_scale, io_dtype, gate_dtype,
                       stream, 0);
}

// vig_gla_bidir_fwd followed by vig_locality_gate_fwd in one kernel: y = o * sigmoid(conv3x3(o)) with o the rounded
// GLA output, never written to memory (but for few sequences: gla_tiles.hip, spread_gate_kernel).  Only shapes of the bf16 MFMA path with the whole sequence in one slab.
int vig_gla_bidir_locgate_fwd(const void* q, const void* k, const void* v, const void* g_fwd, const void* g_bwd,
                              const float* gate_weight, void* y, int B, int H, int L, int Dk, int Dv, int grid_h,
                              int grid_w, float scale, float out_scale, int io_dtype, int gate_dtype, void* stream) {
  vig::GlaArgs a;
  const int rc = fill_args(a, q, k, v, g_fwd, g_bwd, y, nullptr, 0, B, H, L, Dk, Dv, scale, out_scale, io_dtype,
                           gate_dtype, stream);
  if (rc != VIG_OK) return rc;
  if (!gate_weight || !g_bwd || grid_h <= 0 || grid_w <= 0 || (long long)grid_h * grid_w != L) return VIG_EINVAL;
  if (!aligned16(gate_weight)) return VIG_EINVAL;
  if (!vig::gla_mfma_supported(a) || vig::gla_mfma_workspace(B, H, L, Dk, Dv) > 0 ||
      !vig::gla_mfma_gate_grid_ok(grid_h, grid_w))
    return VIG_ENOTSUP;
  a.gate_w = gate_weight;
  a.gate_rows = grid_h;
  a.gate_cols = grid_w;
  return vig::launch_gla_mfma(a);
}

// Same contract as vig_gla_bidir_fwd, but always takes the fp32-arithmetic
// token-recurrent kernel (the exact path), whatever the dtypes.
int vig_gla_bidir_fwd_exact(const void* q, const void* k, const void* v, const void* g_fwd, const void* g_bwd,
                            void* o, void* workspace, size_t workspace_bytes, int B, int H, int L, int Dk, int Dv,
                            float scale, float out_scale, int io_dtype, int gate_dtype, void* stream) {
  vig::GlaArgs a;
  const int rc = fill_args(a, q, k, v, g_fwd, g_bwd, o, workspace, workspace_bytes, B, H, L, Dk, Dv, scale,
                           out_scale, io_dtype, gate_dtype, stream);
  if (rc != VIG_OK) return rc;
  const size_t need = g_bwd ? vig::gla_recurrent_workspace(B, H, L, Dv, io_dtype) : 0;
  if (need > workspace_bytes) return VIG_ENOSPC;
  if (need > 0 && !workspace) return VIG_EINVAL;
  return vig::launch_gla_recurrent(a);
}

int vig_dirgate_fwd(const void* gk_lin, void* g_out, int B, int L, int H, int Dk, float inv_normalizer,
                    float clamp_min, int in_dtype, int out_dtype, void* stream) {
  if (!gk_lin || !g_out || B <= 0 || L <= 0 || H <= 0 || Dk <= 0) return VIG_EINVAL;
  if (!aligned16(gk_lin, g_out)) return VIG_EINVAL;
  if (!dtype_ok(in_dtype) || !dtype_ok(out_dtype) || (Dk % 8) != 0) return VIG_ENOTSUP;
  return vig::launch_dirgate(gk_lin, g_out, B, L, H, Dk, inv_normalizer, clamp_min, in_dtype, out_dtype,
                             (hipStream_t)stream);
}

int vig_dirgate_bwd(const void* gk_lin, const void* d_g, void* d_gk_lin, int B, int L, int H, int Dk,
                    float inv_normalizer, float clamp_min, int in_dtype, int out_dtype, void* stream) {
  if (!gk_lin || !d_g || !d_gk_lin || B <= 0 || L <= 0 || H <= 0 || Dk <= 0) return VIG_EINVAL;
  if (!aligned16(gk_lin, d_g, d_gk_lin)) return VIG_EINVAL;
  if (!dtype_ok(in_dtype) || !dtype_ok(out_dtype) || (Dk % 8) != 0) return VIG_ENOTSUP;
  return vig::launch_dirgate_bwd(gk_lin, d_g, d_gk_lin, B, L, H, Dk, inv_normalizer, clamp_min, in_dtype, out_dtype,
                                 (hipStream_t)stream);
}

int vig_split_heads_bwd_strided(const void* dq, const void* dk, const void* dv, void* d_qkv, long long d_qkv_row_stride,
                                int B, int L, int H, int Dk, int Dv, int io_dtype, void* stream) {
  if (!dq || !dk || !dv || !d_qkv || B <= 0 || L <= 0 || H <= 0 || Dk <= 0 || Dv <= 0) return VIG_EINVAL;
  if (!aligned16(dq, dk, dv, d_qkv)) return VIG_EINVAL;
  if (!dtype_ok(io_dtype) || (Dk % 8) != 0 || (Dv % 8) != 0 || B > 65535) return VIG_ENOTSUP;
  const long long packed = (long long)H * (2 * Dk + Dv);
  const long long ld = d_qkv_row_stride > 0 ? d_qkv_row_stride : packed;
  if (ld < packed || !strided_rows_ok(d_qkv, ld, io_dtype)) return VIG_EINVAL;
  return vig::launch_merge_heads(dq, dk, dv, d_qkv, B, L, H, Dk, Dv, ld, io_dtype, (hipStream_t)stream);
}

int vig_split_heads_bwd(const void* dq, const void* dk, const void* dv, void* d_qkv, int B, int L, int H, int Dk,
                        int Dv, int io_dtype, void* stream) {
  return vig_split_heads_bwd_strided(dq, dk, dv, d_qkv, 0, B, L, H, Dk, Dv, io_dtype, stream);
}

int vig_dirgate_lowrank_fwd(const void* gk_low, long long low_row_stride, const void* w_up, const void* b_up,
                            void* g_out, int B, int L, int H, int Dk, int rank, float inv_normalizer, float clamp_min,
                            int in_dtype, int out_dtype, void* stream) {
  if (!gk_low || !w_up || !b_up || !g_out || B <= 0 || L <= 0 || H <= 0 || Dk <= 0 || rank <= 0) return VIG_EINVAL;
  if (!dtype_ok(in_dtype) || !dtype_ok(out_dtype) || (Dk % 8) != 0 || rank != 16) return VIG_ENOTSUP;
  const long long ld = low_row_stride > 0 ? low_row_stride : rank;
  if (ld < rank || !strided_rows_ok(gk_low, ld, in_dtype) || !strided_rows_ok(w_up, rank, in_dtype) ||
      !strided_rows_ok(b_up, 8, in_dtype) || !aligned16(g_out))
    return VIG_EINVAL;
  return vig::launch_dirgate_lowrank(gk_low, ld, w_up, b_up, g_out, B, L, H, Dk, rank, inv_normalizer, clamp_min,
                                     in_dtype, out_dtype, (hipStream_t)stream);
}

int vig_dirgate_lowrank_bwd(const void* gk_low, long long low_row_stride, const void* w_up, const void* w_up_t,
                            const void* b_up, const void* d_g, void* d_x, void* d_low, long long d_low_row_stride, int B,
                            int L, int H, int Dk, int rank, float inv_normalizer, float clamp_min, int in_dtype,
                            int out_dtype, void* stream) {
  if (!gk_low || !w_up || !w_up_t || !b_up || !d_g || !d_x || !d_low || B <= 0 || L <= 0 || H <= 0 || Dk <= 0) return VIG_EINVAL;
  if (in_dtype != VIG_BF16 || !dtype_ok(out_dtype) || (Dk % 16) != 0 || rank != 16) return VIG_ENOTSUP;
  const long long ld = low_row_stride > 0 ? low_row_stride : rank, ldd = d_low_row_stride > 0 ? d_low_row_stride : rank;
  if (ld < rank || ldd < rank || !strided_rows_ok(gk_low, ld, in_dtype) || !strided_rows_ok(d_low, ldd, in_dtype) ||
      !aligned16(w_up, w_up_t, b_up, d_g, d_x))
    return VIG_EINVAL;
  return vig::launch_dirgate_lowrank_bwd(gk_low, ld, w_up, w_up_t, b_up, d_g, d_x, d_low, ldd, B, L, H, Dk, inv_normalizer,
                                         clamp_min, out_dtype, (hipStream_t)stream);
}

int vig_linear_preferred(long long rows, int N, int K) { return vig::linear_preferred(rows, N, K); }

int vig_linear_fwd(const void* x, long long x_row_stride, const void* weight, const void* bias, void* y, long long y_row_stride,
                   long long rows, int N, int K, void* stream) {
  if (!x || !weight || !y || rows <= 0 || N <= 0 || K <= 0 || x_row_stride < K || y_row_stride < N) return VIG_EINVAL;
  if (N % 8 || K % 32) return VIG_ENOTSUP;
  if (!strided_rows_ok(x, x_row_stride, VIG_BF16) || !strided_rows_ok(y, y_row_stride, VIG_BF16) || !aligned16(weight, bias))
    return VIG_EINVAL;
  return vig::launch_linear(x, x_row_stride, weight, bias, y, y_row_stride, rows, N, K, (hipStream_t)stream);
}

int vig_norm_swiglu_preferred(long long rows, int K, int I) { return vig::norm_swiglu_supported(rows, K, I); }

int vig_norm_swiglu_fwd(const void* x, const void* residual, const float* norm_weight, const void* weight, void* sum, void* y,
                        long long rows, int K, int I, float eps, void* stream) {
  if (!x || !residual || !norm_weight || !weight || !sum || !y || rows <= 0 || K <= 0 || I <= 0 || sum == x || sum == residual ||
      y == x || y == residual || y == sum)
    return VIG_EINVAL;
  if (!aligned16(x, residual, norm_weight, weight, sum, y)) return VIG_EINVAL;
  if (!vig::norm_swiglu_supported(rows, K, I)) return VIG_ENOTSUP;
  return vig::launch_norm_swiglu(x, residual, norm_weight, weight, sum, y, rows, K, I, eps, (hipStream_t)stream);
}

// (16384 rows 14.3 us against 19.6 of a product and a norm; 8192 13.0 / 13.3, 4096 12.5 / 10.9)
int vig_linear_norm_preferred(long long rows, int N, int K) { return rows >= 16384 && vig::linear_norm_supported(rows, N, K); }

int vig_linear_norm_fwd(const void* x, const void* weight, const void* residual, const float* norm_weight, void* y, void* sum,
                        long long rows, int N, int K, float eps, void* stream) {
  if (!x || !weight || !residual || !norm_weight || !y || !sum || rows <= 0 || N <= 0 || K <= 0) return VIG_EINVAL;
  if (!vig::linear_norm_supported(rows, N, K)) return VIG_ENOTSUP;
  if (!aligned16(x, weight, residual, norm_weight, y, sum)) return VIG_EINVAL;
  return vig::launch_linear_norm(x, weight, residual, norm_weight, y, sum, rows, N, K, eps, (hipStream_t)stream);
}

int vig_conv3x3s2_fwd(const void* x, const void* weight, void* y, int B, int H, int W, int Cin, int Cout, void* stream) {
  if (!x || !weight || !y || B <= 0 || H <= 0 || W <= 0 || Cin <= 0 || Cout <= 0) return VIG_EINVAL;
  if (!aligned16(x, weight, y)) return VIG_EINVAL;
  return vig::launch_conv3x3s2(x, weight, y, B, H, W, Cin, Cout, (hipStream_t)stream);
}

size_t vig_matmul_f32_workspace(long long M, int N, long long K) {
  return M <= 0 || N <= 0 || K <= 0 ? 0 : vig::matmul_f32_workspace(M, N, K);
}

int vig_matmul_f32(const float* a, long long lda, int a_across, const float* b, long long ldb, int b_across, const float* bias,
                   const float* add, long long ldadd, float* out, long long ldo, float* a_sums, long long M, int N, long long K,
                   void* workspace, size_t workspace_bytes, void* stream) {
  if (!a || !b || !out || M <= 0 || N <= 0 || K <= 0 || !aligned16(a, b, workspace)) return VIG_EINVAL;
  const bool ta = a_across != 0, tb = b_across != 0;
  if (lda < (ta ? M : K) || ldb < (tb ? N : K) || ldo < N || (add && ldadd < N) || (a_sums && !ta)) return VIG_EINVAL;
  if (!vig::matmul_f32_supported(lda, ta, ldb, tb, M, N, K)) return VIG_ENOTSUP;
  const size_t need = vig::matmul_f32_workspace(M, N, K);
  if (need > workspace_bytes || (need && !workspace)) return VIG_ENOSPC;
  return vig::launch_matmul_f32(a, lda, ta, b, ldb, tb, bias, add, ldadd, out, ldo, a_sums, M, N, K, workspace, (hipStream_t)stream);
}

size_t vig_rmsnorm_pool_workspace(int B, int L, int C) {
  return B <= 0 || L <= 0 || C <= 0 ? 0 : vig::rmsnorm_pool_workspace(B, L, C);
}

int vig_rmsnorm_pool_fwd(const void* x, const void* residual, const float* weight, void* out, void* workspace,
                         size_t workspace_bytes, int B, int L, int C, float eps, void* stream) {
  if (!x || !residual || !weight || !out || B <= 0 || L <= 0 || C <= 0) return VIG_EINVAL;
  if (!aligned16(x, residual, weight, out, workspace)) return VIG_EINVAL;
  if (!workspace || workspace_bytes < vig::rmsnorm_pool_workspace(B, L, C)) return VIG_ENOSPC;
  return vig::launch_rmsnorm_pool(x, residual, weight, out, workspace, B, L, C, eps, (hipStream_t)stream);
}

int vig_cast_many(const void* const* src, void* const* dst, const int* n, const int* transposed_cols, const int* src_dtype,
                  const int* dst_dtype, int count, void* stream) {
  if (!src || !dst || !n || !transposed_cols || !src_dtype || !dst_dtype || count <= 0) return VIG_EINVAL;
  if (count > vig::kMaxCastJobs) return VIG_ENOTSUP;
  for (int j = 0; j < count; ++j) {
    if (!dst[j] || n[j] <= 0 || transposed_cols[j] < 0 || (transposed_cols[j] && n[j] % transposed_cols[j])) return VIG_EINVAL;
    if (!aligned16(src[j], dst[j]) || src[j] == dst[j]) return VIG_EINVAL;
    if (!dtype_ok(src_dtype[j]) || !dtype_ok(dst_dtype[j])) return VIG_ENOTSUP;
  }
  return vig::launch_cast_many(src, dst, n, transposed_cols, src_dtype, dst_dtype, count, (hipStream_t)stream);
}

int vig_dwconv3x3_fwd_pre(const void* x, const float* weight, const float* bias, void* y, void* pre, int B, int h, int w,
                          int C, int silu, int io_dtype, void* stream) {
  if (!x || !weight || !y || B <= 0 || h <= 0 || w <= 0 || C <= 0 || x == y || (pre && (pre == y || pre == x || !silu)))
    return VIG_EINVAL;
  if (!aligned16(x, weight, bias, y, pre)) return VIG_EINVAL;
  if (!dtype_ok(io_dtype) || (C % 8) != 0) return VIG_ENOTSUP;
  return vig::launch_dwconv3x3(x, weight, bias, y, pre, B, h, w, C, silu, io_dtype, (hipStream_t)stream);
}

int vig_dwconv3x3_fwd(const void* x, const float* weight, const float* bias, void* y, int B, int h, int w, int C,
                      int silu, int io_dtype, void* stream) {
  return vig_dwconv3x3_fwd_pre(x, weight, bias, y, nullptr, B, h, w, C, silu, io_dtype, stream);
}

int vig_norm_dwconv3x3_preferred(int B, int h, int w, int C) {
  return B > 0 && h > 0 && w > 0 && vig::norm_dwconv3x3_supported(B, h, w, C);
}

int vig_norm_dwconv3x3_fwd(const void* x, const void* residual, const float* norm_weight, const float* weight, const float* bias,
                           void* sum, void* y, int B, int h, int w, int C, float eps, int silu, void* stream) {
  if (!x || !norm_weight || !weight || !y || B <= 0 || h <= 0 || w <= 0 || C <= 0) return VIG_EINVAL;
  // (a workgroup reads its neighbours' rows: nothing may be written over an input)
  if (y == x || y == residual || y == sum || (sum && (sum == x || sum == residual))) return VIG_EINVAL;
  if (!aligned16(x, residual, norm_weight, weight, sum, y) || !aligned16(bias)) return VIG_EINVAL;
  if (!vig::norm_dwconv3x3_supported(B, h, w, C)) return VIG_ENOTSUP;
  return vig::launch_norm_dwconv3x3(x, residual, norm_weight, weight, bias, sum, y, B, h, w, C, eps, silu, (hipStream_t)stream);
}

int vig_norm_dwconv3x3_linear_preferred(int B, int h, int w, int C, int N) {
  return B > 0 && h > 0 && w > 0 && N > 0 && vig::norm_conv_linear_supported(B, h, w, C, N);
}

int vig_norm_dwconv3x3_linear_fwd(const void* x, const void* residual, const float* norm_weight, const float* conv_weight,
                                  const float* conv_bias, const void* weight, const void* bias, void* sum, void* conv, void* y, int B,
                                  int h, int w, int C, int N, float eps, int silu, void* stream) {
  if (!x || !norm_weight || !conv_weight || !weight || !conv || !y || B <= 0 || h <= 0 || w <= 0 || C <= 0 || N <= 0) return VIG_EINVAL;
  // (a workgroup reads its neighbours' rows: nothing may be written over an input)
  for (const void* out : {(const void*)sum, (const void*)conv, (const void*)y})
    if (out && (out == x || out == residual || out == weight)) return VIG_EINVAL;
  if (conv == y || conv == sum || y == sum) return VIG_EINVAL;
  if (!aligned16(x, residual, norm_weight, conv_weight, sum, conv) || !aligned16(conv_bias, weight, bias, y)) return VIG_EINVAL;
  if (!vig::norm_conv_linear_supported(B, h, w, C, N)) return VIG_ENOTSUP;
  return vig::launch_norm_conv_linear(x, residual, norm_weight, conv_weight, conv_bias, weight, bias, sum, conv, y, B, h, w, C, N, eps, silu,
                                      (hipStream_t)stream);
}

size_t vig_dwconv3x3_bwd_weight_workspace(int B, int C) {
  if (B <= 0 || C <= 0) return 0;
  return vig::dwconv3x3_wgrad_workspace(B, C);
}

int vig_dwconv3x3_bwd_later(const void* x, const void* dy, const void* pre, const float* weight, void* dx, float* dw_db,
                      void* workspace, size_t workspace_bytes, int B, int h, int w, int C, int io_dtype, vig_sum_jobs* later, void* stream) {
  if (!x || !dy || (!dx && !dw_db) || (dx && !weight) || B <= 0 || h <= 0 || w <= 0 || C <= 0 || dx == dy || (dx && dx == x))
    return VIG_EINVAL;
  if (!aligned16(x, dy, pre, dx, dw_db, workspace)) return VIG_EINVAL;
  if (!dtype_ok(io_dtype) || (C % 8) != 0) return VIG_ENOTSUP;
  if (dw_db && (!workspace || workspace_bytes < vig::dwconv3x3_wgrad_least_workspace(B, C))) return VIG_ENOSPC;
  if (!room_for(later, dw_db ? 1 : 0)) return VIG_EINVAL;
  return vig::launch_dwconv3x3_bwd(x, dy, pre, weight, dx, dw_db, workspace, workspace_bytes, B, h, w, C, io_dtype, later, (hipStream_t)stream);
}
int vig_dwconv3x3_bwd(const void* x, const void* dy, const void* pre, const float* weight, void* dx, float* dw_db,
                      void* workspace, size_t workspace_bytes, int B, int h, int w, int C, int io_dtype, void* stream) {
  return vig_dwconv3x3_bwd_later(x, dy, pre, weight, dx, dw_db, workspace, workspace_bytes, B, h, w, C, io_dtype, nullptr, stream);
}

int vig_dwconv3x3_bwd_weight(const void* x, const void* dy, float* dw_db, void* workspace, size_t workspace_bytes,
                             int B, int h, int w, int C, int io_dtype, void* stream) {
  if (!dw_db) return VIG_EINVAL;
  return vig_dwconv3x3_bwd(x, dy, nullptr, nullptr, nullptr, dw_db, workspace, workspace_bytes, B, h, w, C, io_dtype, stream);
}

int vig_locality_gate_fwd(const void* o, const float* weight, void* y, int B, int H, int h, int w, int Dv,
                          int io_dtype, void* stream) {
  if (!o || !weight || !y || B <= 0 || H <= 0 || h <= 0 || w <= 0 || o == y) return VIG_EINVAL;
  if (!aligned16(o, weight, y)) return VIG_EINVAL;
  if (!dtype_ok(io_dtype) || (Dv % 8) != 0 || Dv <= 0) return VIG_ENOTSUP;
  return vig::launch_locality_gate(o, weight, y, B, H, h, w, Dv, io_dtype, (hipStream_t)stream);
}

int vig_locality_blend_fwd(const void* o, const void* local, const void* g_lin, const float* w_g, const float* w_l,
                           void* y, int B, int H, int L, int Dv, long long g_row_stride, float eps, int silu_out,
                           int io_dtype, void* stream) {
  if (!o || !local || !g_lin || !w_g || !w_l || !y || B <= 0 || H <= 0 || L <= 0) return VIG_EINVAL;
  if (!aligned16(o, local, w_g, w_l, y)) return VIG_EINVAL;
  if (!dtype_ok(io_dtype) || !(Dv == 32 || Dv == 64)) return VIG_ENOTSUP;
  const long long ldg = g_row_stride > 0 ? g_row_stride : (long long)H * Dv;
  if (ldg < (long long)H * Dv || !strided_rows_ok(g_lin, ldg, io_dtype)) return VIG_EINVAL;
  return vig::launch_locality_blend(o, local, g_lin, w_g, w_l, y, B, H, L, Dv, ldg, eps, silu_out, io_dtype,
                                    (hipStream_t)stream);
}

size_t vig_locality_blend_bwd_workspace(int B, int L, int Dv) {
  if (B <= 0 || L <= 0 || !(Dv == 32 || Dv == 64)) return 0;
  return vig::locality_blend_bwd_workspace(B, L, Dv);
}

int vig_locality_blend_bwd_strided_later(const void* o, const void* local, const void* g_lin, const float* w_g, const float* w_l,
                                   const void* dy, void* d_o, void* d_local, void* d_glin, float* dw, void* workspace,
                                   size_t workspace_bytes, int B, int H, int L, int Dv, long long g_row_stride,
                                   long long d_glin_row_stride, float eps, int silu_out, int io_dtype, vig_sum_jobs* later, void* stream) {
  if (!o || !local || !g_lin || !w_g || !w_l || !dy || !d_o || !d_local || !d_glin || !dw || B <= 0 || H <= 0 ||
      L <= 0)
    return VIG_EINVAL;
  if (!aligned16(o, local, w_g, w_l, dy, d_o, d_local, d_glin, dw, workspace)) return VIG_EINVAL;
  if (!dtype_ok(io_dtype) || !(Dv == 32 || Dv == 64)) return VIG_ENOTSUP;
  const long long row = (long long)H * Dv;
  const long long ldg = g_row_stride > 0 ? g_row_stride : row, ldd = d_glin_row_stride > 0 ? d_glin_row_stride : row;
  if (ldg < row || !strided_rows_ok(g_lin, ldg, io_dtype) || ldd < row || !strided_rows_ok(d_glin, ldd, io_dtype))
    return VIG_EINVAL;
  if (!workspace || workspace_bytes < vig::locality_blend_bwd_least_workspace(B, L, Dv)) return VIG_ENOSPC;
  const long long rows = (long long)(std::min(workspace_bytes, vig::locality_blend_bwd_workspace(B, L, Dv)) / (2 * Dv * sizeof(float)));
  if (!room_for(later, 1)) return VIG_EINVAL;
  return vig::launch_locality_blend_bwd(o, local, g_lin, w_g, w_l, dy, d_o, d_local, d_glin, dw, workspace, rows, B, H, L, Dv,
                                        ldg, ldd, eps, silu_out, io_dtype, later, (hipStream_t)stream);
}
int vig_locality_blend_bwd_strided(const void* o, const void* local, const void* g_lin, const float* w_g, const float* w_l,
                                   const void* dy, void* d_o, void* d_local, void* d_glin, float* dw, void* workspace,
                                   size_t workspace_bytes, int B, int H, int L, int Dv, long long g_row_stride,
                                   long long d_glin_row_stride, float eps, int silu_out, int io_dtype, void* stream) {
  return vig_locality_blend_bwd_strided_later(o, local, g_lin, w_g, w_l, dy, d_o, d_local, d_glin, dw, workspace, workspace_bytes, B, H, L,
                                              Dv, g_row_stride, d_glin_row_stride, eps, silu_out, io_dtype, nullptr, stream);
}

int vig_locality_blend_bwd(const void* o, const void* local, const void* g_lin, const float* w_g, const float* w_l,
                           const void* dy, void* d_o, void* d_local, void* d_glin, float* dw, void* workspace,
                           size_t workspace_bytes, int B, int H, int L, int Dv, long long g_row_stride, float eps,
                           int silu_out, int io_dtype, void* stream) {
  return vig_locality_blend_bwd_strided(o, local, g_lin, w_g, w_l, dy, d_o, d_local, d_glin, dw, workspace, workspace_bytes,
                                        B, H, L, Dv, g_row_stride, 0, eps, silu_out, io_dtype, stream);
}

int vig_rmsnorm_mixed_fwd(const void* x, const void* residual, const float* weight, void* y, void* residual_out,
                          long long rows, int C, float eps, int round_sum, int x_dtype, int sum_dtype, int y_dtype,
                          void* stream) {
  if (!x || !weight || !y || rows <= 0 || C <= 0 || rows > 0x7fffffffLL) return VIG_EINVAL;
  if (!aligned16(x, residual, weight, y, residual_out)) return VIG_EINVAL;
  if (!dtype_ok(x_dtype) || !dtype_ok(sum_dtype) || !dtype_ok(y_dtype) || (C % 8) != 0 || C > 4096 ||
      !vig::rmsnorm_types_ok(x_dtype, sum_dtype, y_dtype))
    return VIG_ENOTSUP;
  return vig::launch_rmsnorm(x, residual, weight, y, residual_out, (int)rows, C, eps, round_sum, x_dtype, sum_dtype, y_dtype,
                             (hipStream_t)stream);
}

int vig_rmsnorm_fwd(const void* x, const void* residual, const float* weight, void* y, void* residual_out,
                    long long rows, int C, float eps, int round_sum, int io_dtype, void* stream) {
  return vig_rmsnorm_mixed_fwd(x, residual, weight, y, residual_out, rows, C, eps, round_sum, io_dtype, io_dtype, io_dtype,
                               stream);
}

int vig_layernorm_fwd(const void* x, const float* weight, const float* bias, void* y, long long rows, int C,
                      float eps, int silu, const float* pre_bias, const void* post_add, int post_rows, int io_dtype,
                      void* stream) {
  if (!x || !weight || !bias || !y || rows <= 0 || C <= 0 || (post_add && post_rows <= 0)) return VIG_EINVAL;
  if (!aligned16(x, weight, bias, y, pre_bias, post_add)) return VIG_EINVAL;
  if (!dtype_ok(io_dtype) || (C % 8) != 0 || C > 4096) return VIG_ENOTSUP;
  return vig::launch_layernorm(x, weight, bias, y, rows, C, eps, silu, pre_bias, post_add, post_rows, io_dtype,
                               (hipStream_t)stream);
}

int vig_stem_norm_fwd(const void* x, const float* pre_bias, const float* weight, const float* bias, void* y, long long rows, int C, float eps,
                      int silu, int x_dtype, int y_dtype, void* stream) {
  if (!x || !weight || !bias || !y || rows <= 0 || C <= 0) return VIG_EINVAL;
  if (!aligned16(x, pre_bias, weight, bias, y)) return VIG_EINVAL;
  if (!dtype_ok(x_dtype) || !dtype_ok(y_dtype) || !vig::stem_norm_supported(rows, C, x_dtype, y_dtype)) return VIG_ENOTSUP;
  return vig::launch_stem_norm(x, pre_bias, weight, bias, y, rows, C, eps, silu, x_dtype, y_dtype, (hipStream_t)stream);
}

size_t vig_stem_norm_bwd_workspace(long long rows, int C) { return rows <= 0 || C <= 0 ? 0 : vig::stem_norm_bwd_workspace(rows, C); }

int vig_stem_norm_bwd(const void* x, const float* pre_bias, const float* weight, const float* bias, const void* dy, void* dx, float* dparams,
                      void* workspace, size_t workspace_bytes, long long rows, int C, float eps, int silu, int x_dtype, int y_dtype,
                      void* stream) {
  if (!x || !weight || !bias || !dy || !dparams || rows <= 0 || C <= 0) return VIG_EINVAL;
  if (!aligned16(x, pre_bias, weight, bias, dy, dx) || !aligned16(dparams, workspace)) return VIG_EINVAL;
  if (!dtype_ok(x_dtype) || !dtype_ok(y_dtype) || !vig::stem_norm_supported(rows, C, x_dtype, y_dtype)) return VIG_ENOTSUP;
  if (!workspace || workspace_bytes < vig::stem_norm_bwd_workspace(rows, C)) return VIG_ENOSPC;
  return vig::launch_stem_norm_bwd(x, pre_bias, weight, bias, dy, dx, dparams, workspace, rows, C, eps, silu, x_dtype, y_dtype, (hipStream_t)stream);
}

int vig_split_heads_fwd(const void* qkv, void* q, void* k, void* v, int B, int L, int H, int Dk, int Dv,
                        long long qkv_row_stride, int io_dtype, void* stream) {
  if (!qkv || !q || !k || !v || B <= 0 || L <= 0 || H <= 0 || Dk <= 0 || Dv <= 0) return VIG_EINVAL;
  if (!aligned16(q, k, v)) return VIG_EINVAL;
  if (!dtype_ok(io_dtype) || (Dk % 8) != 0 || (Dv % 8) != 0 || B > 65535) return VIG_ENOTSUP;
  const long long packed = (long long)H * (2 * Dk + Dv);
  const long long ld = qkv_row_stride > 0 ? qkv_row_stride : packed;
  if (ld < packed || !strided_rows_ok(qkv, ld, io_dtype)) return VIG_EINVAL;
  return vig::launch_split_heads(qkv, q, k, v, B, L, H, Dk, Dv, ld, io_dtype, (hipStream_t)stream);
}

int vig_patch_conv_fwd(const void* x, const void* w_packed, void* y, int B, int Cin, int H, int W, int KH, int KW,
                       int stride, int padding, int Cout, int io_dtype, void* stream) {
  if (!x || !w_packed || !y || B <= 0 || Cin <= 0 || H <= 0 || W <= 0 || KH <= 0 || KW <= 0 || Cout <= 0) return VIG_EINVAL;
  if (io_dtype != VIG_BF16 || !vig::patch_conv_supported(Cin, H, W, KH, KW, stride, padding, Cout)) return VIG_ENOTSUP;
  if (!strided_rows_ok(x, W, io_dtype) || !strided_rows_ok(w_packed, 16, io_dtype) || !strided_rows_ok(y, Cout, io_dtype))
    return VIG_EINVAL;
  return vig::launch_patch_conv(x, w_packed, y, B, Cin, H, W, KH, KW, Cout, (hipStream_t)stream);
}

int vig_patch_conv_norm_fwd(const void* x, const void* w_packed, const float* norm_weight, const float* norm_bias, const float* pre_bias, void* y,
                            int B, int Cin, int H, int W, int KH, int KW, int stride, int padding, int Cout, float eps, int silu, void* stream) {
  if (!x || !w_packed || !norm_weight || !norm_bias || !y || B <= 0 || Cin <= 0 || H <= 0 || W <= 0 || KH <= 0 || KW <= 0 || Cout <= 0)
    return VIG_EINVAL;
  if (!vig::patch_conv_supported(Cin, H, W, KH, KW, stride, padding, Cout)) return VIG_ENOTSUP;
  if (!strided_rows_ok(x, W, VIG_BF16) || !strided_rows_ok(w_packed, 16, VIG_BF16) || !strided_rows_ok(y, Cout, VIG_BF16)) return VIG_EINVAL;
  return vig::launch_patch_conv_norm(x, w_packed, norm_weight, norm_bias, pre_bias, y, B, Cin, H, W, KH, KW, Cout, eps, silu, (hipStream_t)stream);
}

int vig_locality_blend_linear_fwd(const void* o, const void* local, const void* g_lin, const float* w_g,
                                  const float* w_l, const void* weight, void* out, int B, int H, int L, int Dv, int C,
                                  long long g_row_stride, float eps, int silu_out, int io_dtype, void* stream) {
  if (!o || !local || !g_lin || !w_g || !w_l || !weight || !out || B <= 0 || H <= 0 || L <= 0) return VIG_EINVAL;
  if (!aligned16(o, local, w_g, w_l, weight, out)) return VIG_EINVAL;
  if (io_dtype != VIG_BF16 || !vig::blend_linear_supported(H, Dv, C)) return VIG_ENOTSUP;
  const long long ldg = g_row_stride > 0 ? g_row_stride : (long long)H * Dv;
  if (ldg < (long long)H * Dv || !strided_rows_ok(g_lin, ldg, io_dtype)) return VIG_EINVAL;
  return vig::launch_blend_linear(o, local, g_lin, w_g, w_l, weight, out, nullptr, B, H, L, Dv, C, ldg, eps, silu_out,
                                  (hipStream_t)stream);
}

int vig_locality_blend_linear_kept_fwd(const void* o, const void* local, const void* g_lin, const float* w_g,
                                  const float* w_l, const void* weight, void* blended, void* out, int B, int H, int L, int Dv, int C,
                                  long long g_row_stride, float eps, int silu_out, int io_dtype, void* stream) {
  if (!o || !local || !g_lin || !w_g || !w_l || !weight || !blended || !out || B <= 0 || H <= 0 || L <= 0) return VIG_EINVAL;
  if (!aligned16(o, local, w_g, w_l, weight, blended, out)) return VIG_EINVAL;
  if (io_dtype != VIG_BF16 || !vig::blend_linear_supported(H, Dv, C)) return VIG_ENOTSUP;
  const long long ldg = g_row_stride > 0 ? g_row_stride : (long long)H * Dv;
  if (ldg < (long long)H * Dv || !strided_rows_ok(g_lin, ldg, io_dtype)) return VIG_EINVAL;
  return vig::launch_blend_linear(o, local, g_lin, w_g, w_l, weight, out, blended, B, H, L, Dv, C, ldg, eps, silu_out,
                                  (hipStream_t)stream);
}

int vig_locality_blend_swiglu_preferred(long long rows, int C, int I) { return vig::blend_swiglu_supported(rows, C, I); }

int vig_locality_blend_swiglu_fwd(const void* o, const void* local, const void* g_lin, const float* w_g, const float* w_l,
                                  const void* out_weight, const void* residual, const float* norm_weight, const void* weight, void* sum,
                                  void* y, int B, int H, int L, int Dv, int C, int I, long long g_row_stride, float eps, int silu_out,
                                  float norm_eps, void* stream) {
  if (!o || !local || !g_lin || !w_g || !w_l || !out_weight || !residual || !norm_weight || !weight || !sum || !y || B <= 0 || H <= 0 || L <= 0)
    return VIG_EINVAL;
  // (a row is read by every workgroup of its tile: nothing may be written over an input)
  for (const void* in : {o, local, g_lin, out_weight, residual, weight})
    if (in == sum || in == y) return VIG_EINVAL;
  if (sum == y) return VIG_EINVAL;
  if (!aligned16(o, local, w_g, w_l, out_weight, residual) || !aligned16(norm_weight, weight, sum, y)) return VIG_EINVAL;
  if (Dv != 64 || (long long)H * Dv != C || !vig::blend_swiglu_supported((long long)B * L, C, I)) return VIG_ENOTSUP;
  const long long ldg = g_row_stride > 0 ? g_row_stride : C;
  if (ldg < C || !strided_rows_ok(g_lin, ldg, VIG_BF16)) return VIG_EINVAL;
  return vig::launch_blend_swiglu(o, local, g_lin, w_g, w_l, out_weight, residual, norm_weight, weight, sum, y, (long long)B * L, L, C, I, ldg,
                                  eps, silu_out, norm_eps, (hipStream_t)stream);
}

int vig_linear_swiglu_fwd(const void* x, const void* weight, void* y, long long rows, int K, int I, int io_dtype,
                          void* stream) {
  if (!x || !weight || !y || rows <= 0 || K <= 0 || I <= 0) return VIG_EINVAL;
  if (io_dtype != VIG_BF16 || !vig::linear_swiglu_supported(K, I)) return VIG_ENOTSUP;
  if (!strided_rows_ok(x, K, io_dtype) || !strided_rows_ok(weight, K, io_dtype) || !strided_rows_ok(y, I, io_dtype))
    return VIG_EINVAL;
  return vig::launch_linear_swiglu(x, weight, y, nullptr, rows, K, I, (hipStream_t)stream);
}

int vig_linear_swiglu_kept_fwd(const void* x, const void* weight, void* gate_up, void* y, long long rows, int K, int I,
                               int io_dtype, void* stream) {
  if (!x || !weight || !gate_up || !y || rows <= 0 || K <= 0 || I <= 0) return VIG_EINVAL;
  if (io_dtype != VIG_BF16 || !vig::linear_swiglu_supported(K, I)) return VIG_ENOTSUP;
  if (!strided_rows_ok(x, K, io_dtype) || !strided_rows_ok(weight, K, io_dtype) || !strided_rows_ok(gate_up, 2LL * I, io_dtype) ||
      !strided_rows_ok(y, I, io_dtype))
    return VIG_EINVAL;
  return vig::launch_linear_swiglu(x, weight, y, gate_up, rows, K, I, (hipStream_t)stream);
}

int vig_linear_swiglu_bwd(const void* d_out, const void* w_down, const void* gate_up, void* d_gate_up, long long rows, int K, int I,
                          int io_dtype, void* stream) {
  if (!d_out || !w_down || !gate_up || !d_gate_up || rows <= 0 || K <= 0 || I <= 0) return VIG_EINVAL;
  if (io_dtype != VIG_BF16 || !vig::linear_swiglu_supported(K, I)) return VIG_ENOTSUP;
  if (!strided_rows_ok(d_out, K, io_dtype) || !strided_rows_ok(w_down, I, io_dtype) || !strided_rows_ok(gate_up, 2LL * I, io_dtype) ||
      !strided_rows_ok(d_gate_up, 2LL * I, io_dtype))
    return VIG_EINVAL;
  return vig::launch_linear_swiglu_bwd(d_out, w_down, gate_up, d_gate_up, rows, K, I, (hipStream_t)stream);
}

int vig_linear_bwd_input_preferred(long long rows, int N, int K) { return rows >= 16384 && vig::linear_regs_supported(N, K); }

int vig_linear_bwd_input(const void* dy, const void* weight, void* dx, long long rows, int N, int K, int io_dtype, void* stream) {
  if (!dy || !weight || !dx || rows <= 0 || N <= 0 || K <= 0) return VIG_EINVAL;
  if (io_dtype != VIG_BF16 || !vig::linear_regs_supported(N, K)) return VIG_ENOTSUP;
  if (!strided_rows_ok(dy, N, io_dtype) || !strided_rows_ok(weight, K, io_dtype) || !strided_rows_ok(dx, K, io_dtype)) return VIG_EINVAL;
  return vig::launch_linear_columns(dy, weight, dx, rows, K, N, (hipStream_t)stream);
}

int vig_swiglu_fwd(const void* gate_up, void* out, long long rows, int I, int io_dtype, void* stream) {
  if (!gate_up || !out || rows <= 0 || I <= 0) return VIG_EINVAL;
  if (!aligned16(gate_up, out)) return VIG_EINVAL;
  if (!dtype_ok(io_dtype) || (I % 8) != 0) return VIG_ENOTSUP;
  return vig::launch_swiglu(gate_up, out, rows, I, io_dtype, (hipStream_t)stream);
}

int vig_swiglu_bwd(const void* gate_up, const void* dy, void* d_gate_up, long long rows, int I, int io_dtype,
                   void* stream) {
  if (!gate_up || !dy || !d_gate_up || rows <= 0 || I <= 0) return VIG_EINVAL;
  if (!aligned16(gate_up, dy, d_gate_up)) return VIG_EINVAL;
  if (!dtype_ok(io_dtype) || (I % 8) != 0) return VIG_ENOTSUP;
  return vig::launch_swiglu_bwd(gate_up, dy, d_gate_up, rows, I, io_dtype, (hipStream_t)stream);
}

size_t vig_rmsnorm_bwd_workspace(long long rows, int C) {
  if (rows <= 0 || C <= 0) return 0;
  return vig::rmsnorm_bwd_workspace(rows, C);
}

int vig_rmsnorm_mixed_bwd_later(const void* sum, const float* weight, const void* dy, const void* d_sum, void* ds, void* dx,
                          float* dweight, void* workspace, size_t workspace_bytes, long long rows, int C, float eps,
                          int sum_dtype, int y_dtype, vig_sum_jobs* later, void* stream) {
  if (!sum || !weight || !dy || !ds || rows <= 0 || C <= 0 || rows > 0x7fffffffLL) return VIG_EINVAL;
  if (!aligned16(sum, weight, dy, d_sum, ds, dx, dweight, workspace)) return VIG_EINVAL;
  if (!dtype_ok(sum_dtype) || !dtype_ok(y_dtype) || (C % 8) != 0 || C > 1024 ||
      !vig::rmsnorm_types_ok(sum_dtype, sum_dtype, y_dtype))
    return VIG_ENOTSUP;
  if (dweight && (!workspace || workspace_bytes < vig::rmsnorm_bwd_workspace(rows, C))) return VIG_ENOSPC;
  if (!room_for(later, dweight ? 1 : 0)) return VIG_EINVAL;
  return vig::launch_rmsnorm_bwd(sum, weight, dy, d_sum, ds, dx, dweight, workspace, rows, C, eps, sum_dtype, y_dtype,
                                 later, (hipStream_t)stream);
}
int vig_rmsnorm_mixed_bwd(const void* sum, const float* weight, const void* dy, const void* d_sum, void* ds, void* dx,
                          float* dweight, void* workspace, size_t workspace_bytes, long long rows, int C, float eps,
                          int sum_dtype, int y_dtype, void* stream) {
  return vig_rmsnorm_mixed_bwd_later(sum, weight, dy, d_sum, ds, dx, dweight, workspace, workspace_bytes, rows, C, eps, sum_dtype, y_dtype, nullptr, stream);
}

int vig_rmsnorm_bwd(const void* sum, const float* weight, const void* dy, const void* d_sum, void* ds, float* dweight,
                    void* workspace, size_t workspace_bytes, long long rows, int C, float eps, int io_dtype,
                    void* stream) {
  return vig_rmsnorm_mixed_bwd(sum, weight, dy, d_sum, ds, nullptr, dweight, workspace, workspace_bytes, rows, C, eps, io_dtype,
                               io_dtype, stream);
}

static bool bwd_shape_ok(int Dk, int Dv) {
  return (Dk == 16 && Dv == 32) || (Dk == 32 && (Dv == 32 || Dv == 64)) || (Dk == 64 && (Dv == 32 || Dv == 64));
}

size_t vig_gla_bidir_bwd_workspace(int B, int H, int L, int Dk, int Dv, int bidirectional) {
  if (B <= 0 || H <= 0 || L <= 0 || !bwd_shape_ok(Dk, Dv)) return 0;
  return vig::gla_backward_workspace(B, H, L, Dk, Dv, bidirectional);
}

// The backward of HierViG's head shape rides the matrix-core kernels the way its forward does: q, k, both gates and
// their four gradients padded to 32 channels, v, d_o and dv to 64, then the backward's own workspace at 32 / 64.
static size_t padded_bwd_tensors(int B, int H, int L) {
  const size_t n = (8 * padded_elems_qk(B, H, L) + 3 * padded_elems_v(B, H, L)) * sizeof(uint16_t);
  return (n + 255) / 256 * 256;
}
static size_t padded_bwd_workspace(int B, int H, int L) {
  return padded_bwd_tensors(B, H, L) + vig::gla_backward_workspace(B, H, L, 32, 64, 1);
}

size_t vig_gla_bidir_bwd_workspace_for(int B, int H, int L, int Dk, int Dv, int io_dtype, int gate_dtype,
                                       int bidirectional) {
  if (B <= 0 || H <= 0 || L <= 0 || !bwd_shape_ok(Dk, Dv) || !dtype_ok(io_dtype) || !dtype_ok(gate_dtype)) return 0;
  if (padded_shape(L, Dk, Dv, io_dtype, gate_dtype, bidirectional != 0)) return padded_bwd_workspace(B, H, L);
  const size_t beyond = io_dtype == VIG_F32 && gate_dtype == VIG_F32 && bidirectional ? vig::gla_backward_f32_extra(B, H, L, Dk, Dv) : 0;
  return vig::gla_backward_workspace(B, H, L, Dk, Dv, bidirectional) + beyond;
}

static int gla_bidir_bwd(const void* q, const void* k, const void* v, const void* g_fwd, const void* g_bwd,
                         const void* d_o, void* dq, void* dk, void* dv, void* dg_fwd, void* dg_bwd, void* workspace,
                         size_t workspace_bytes, int B, int H, int L, int Dk, int Dv, float scale, float out_scale,
                         int io_dtype, int gate_dtype, bool exact, void* stream) {
  if (!q || !k || !v || !g_fwd || !d_o || !dq || !dk || !dv || !dg_fwd || (g_bwd && !dg_bwd) || B <= 0 || H <= 0 ||
      L <= 0)
    return VIG_EINVAL;
  if (!aligned16(q, k, v, g_fwd, g_bwd, d_o, dq, dk, dv, dg_fwd, dg_bwd, workspace)) return VIG_EINVAL;
  if ((long long)B * H > 2147483647LL) return VIG_EINVAL;
  if (!dtype_ok(io_dtype) || !dtype_ok(gate_dtype) || !bwd_shape_ok(Dk, Dv)) return VIG_ENOTSUP;
  if (!exact && padded_shape(L, Dk, Dv, io_dtype, gate_dtype, g_bwd != nullptr) && workspace &&
      workspace_bytes >= padded_bwd_workspace(B, H, L)) {
    // (a caller that sized the workspace with vig_gla_bidir_bwd_workspace gets the recurrent kernel below)
    const size_t nqk = padded_elems_qk(B, H, L), nv = padded_elems_v(B, H, L);
    uint16_t* p = static_cast<uint16_t*>(workspace);
    uint16_t *qp = p, *kp = p + nqk, *gfp = p + 2 * nqk, *gbp = p + 3 * nqk, *dqp = p + 4 * nqk, *dkp = p + 5 * nqk,
             *dgfp = p + 6 * nqk, *dgbp = p + 7 * nqk, *vp = p + 8 * nqk, *dop = vp + nv, *dvp = dop + nv;
    const long long rows = (long long)B * H * L;
    hipStream_t st = (hipStream_t)stream;
    {
      const void* srcs[6] = {q, k, g_fwd, g_bwd, v, d_o};
      void* dsts[6] = {qp, kp, gfp, gbp, vp, dop};
      const int src_c[6] = {16, 16, 16, 16, 32, 32}, dst_c[6] = {32, 32, 32, 32, 64, 64};
      const int e = vig::launch_pad_channels_multi(srcs, dsts, src_c, dst_c, 6, rows, st);
      if (e) return e;
    }
    const int e = vig::launch_gla_backward(qp, kp, vp, gfp, gbp, dop, dqp, dkp, dvp, dgfp, dgbp,
                                           (char*)workspace + padded_bwd_tensors(B, H, L), B, H, L, 32, 64, scale,
                                           out_scale, io_dtype, gate_dtype, false, 0, st);
    if (e) return e;
    const void* srcs[5] = {dqp, dkp, dgfp, dgbp, dvp};
    void* dsts[5] = {dq, dk, dg_fwd, dg_bwd, dv};
    const int src_c[5] = {32, 32, 32, 32, 64}, dst_c[5] = {16, 16, 16, 16, 32};
    return vig::launch_pad_channels_multi(srcs, dsts, src_c, dst_c, 5, rows, st);
  }
  const size_t need = vig::gla_backward_workspace(B, H, L, Dk, Dv, g_bwd != nullptr);
  if (!workspace || workspace_bytes < need) return VIG_ENOSPC;
  return vig::launch_gla_backward(q, k, v, g_fwd, g_bwd, d_o, dq, dk, dv, dg_fwd, dg_bwd, workspace, B, H, L, Dk, Dv,
                                  scale, out_scale, io_dtype, gate_dtype, exact, workspace_bytes - need, (hipStream_t)stream);
}

int vig_gla_bidir_bwd(const void* q, const void* k, const void* v, const void* g_fwd, const void* g_bwd,
                      const void* d_o, void* dq, void* dk, void* dv, void* dg_fwd, void* dg_bwd, void* workspace,
                      size_t workspace_bytes, int B, int H, int L, int Dk, int Dv, float scale, float out_scale,
                      int io_dtype, int gate_dtype, void* stream) {
  return gla_bidir_bwd(q, k, v, g_fwd, g_bwd, d_o, dq, dk, dv, dg_fwd, dg_bwd, workspace, workspace_bytes, B, H, L, Dk,
                       Dv, scale, out_scale, io_dtype, gate_dtype, false, stream);
}

int vig_gla_bidir_bwd_rows(const void* q, const void* k, const void* v, long long row_stride, const void* g_fwd, const void* g_bwd, const void* d_o,
                           void* dq, void* dk, void* dv, long long d_row_stride, void* dg_fwd, void* dg_bwd, void* workspace, size_t workspace_bytes,
                           int B, int H, int L, int Dk, int Dv, float scale, float out_scale, int io_dtype, int gate_dtype, void* stream) {
  if (!q || !k || !v || !g_fwd || !g_bwd || !d_o || !dq || !dk || !dv || !dg_fwd || !dg_bwd || B <= 0 || H <= 0 || L <= 0) return VIG_EINVAL;
  if (!aligned16(q, k, v, g_fwd, g_bwd, d_o, dq, dk, dv, dg_fwd, dg_bwd, workspace)) return VIG_EINVAL;
  if (!vig::gla_backward_in_place(L, Dk, Dv, io_dtype, gate_dtype, true) || (long long)B * H > 2147483647LL) return VIG_ENOTSUP;
  for (const long long ld : {row_stride, d_row_stride})
    if (ld < (long long)H * std::max(Dk, Dv) || ld % 8 != 0 || ld > (1 << 20)) return VIG_EINVAL;
  const size_t need = vig::gla_backward_workspace(B, H, L, Dk, Dv, 1);
  if (!workspace || workspace_bytes < need) return VIG_ENOSPC;
  return vig::launch_gla_backward(q, k, v, g_fwd, g_bwd, d_o, dq, dk, dv, dg_fwd, dg_bwd, workspace, B, H, L, Dk, Dv, scale, out_scale, io_dtype,
                                  gate_dtype, false, workspace_bytes - need, (hipStream_t)stream, row_stride, d_row_stride);
}

// Same contract, always the fp32-arithmetic token-recurrent kernel.
int vig_gla_bidir_bwd_exact(const void* q, const void* k, const void* v, const void* g_fwd, const void* g_bwd,
                            const void* d_o, void* dq, void* dk, void* dv, void* dg_fwd, void* dg_bwd,
                            void* workspace, size_t workspace_bytes, int B, int H, int L, int Dk, int Dv, float scale,
                            float out_scale, int io_dtype, int gate_dtype, void* stream) {
  return gla_bidir_bwd(q, k, v, g_fwd, g_bwd, d_o, dq, dk, dv, dg_fwd, dg_bwd, workspace, workspace_bytes, B, H, L, Dk,
                       Dv, scale, out_scale, io_dtype, gate_dtype, true, stream);
}

size_t vig_linear_bwd_weight_workspace(long long rows, int N, int K) {
  return vig_linear_bwd_weight_many_workspace(rows, &N, &K, 1);
}

size_t vig_linear_bwd_weight_many_workspace(long long rows, const int* N, const int* K, int count) {
  if (!N || !K || count < 1 || count > vig::kWgradLayers) return 0;
  vig::LinearWgrad l[vig::kWgradLayers] = {};
  for (int i = 0; i < count; ++i) {
    if (!vig::linear_wgrad_supported(rows, N[i], K[i])) return 0;
    l[i].N = N[i], l[i].K = K[i];
  }
  return vig::linear_wgrad_workspace(rows, l, count);
}

int vig_linear_bwd_weight(const void* dy, long long dy_row_stride, const void* x, long long x_row_stride, float* dweight,
                          float* dbias, void* workspace, size_t workspace_bytes, long long rows, int N, int K, void* stream) {
  return vig_linear_bwd_weight_many(&dy, &dy_row_stride, &x, &x_row_stride, &dweight, &dbias, workspace, workspace_bytes, rows, &N, &K, 1,
                                    stream);
}

int vig_linear_bwd_weight_many_later(const void* const* dy, const long long* dy_row_stride, const void* const* x, const long long* x_row_stride,
                               float* const* dweight, float* const* dbias, void* workspace, size_t workspace_bytes, long long rows,
                               const int* N, const int* K, int count, vig_sum_jobs* later, void* stream) {
  if (!dy || !dy_row_stride || !x || !x_row_stride || !dweight || !N || !K || count < 1 || count > vig::kWgradLayers) return VIG_EINVAL;
  vig::LinearWgrad l[vig::kWgradLayers] = {};
  for (int i = 0; i < count; ++i)
    if (!dy[i] || !x[i] || !dweight[i] || rows <= 0 || N[i] <= 0 || K[i] <= 0 || dy_row_stride[i] < N[i] || x_row_stride[i] < K[i])
      return VIG_EINVAL;
  for (int i = 0; i < count; ++i)
    if (!vig::linear_wgrad_supported(rows, N[i], K[i])) return VIG_ENOTSUP;
  for (int i = 0; i < count; ++i) {
    float* const db = dbias ? dbias[i] : nullptr;
    if (!strided_rows_ok(dy[i], dy_row_stride[i], VIG_BF16) || !strided_rows_ok(x[i], x_row_stride[i], VIG_BF16) ||
        !aligned16(dweight[i], workspace) || (db && reinterpret_cast<uintptr_t>(db) % 4))
      return VIG_EINVAL;
    l[i] = {dy[i], x[i], dy_row_stride[i], x_row_stride[i], dweight[i], db, N[i], K[i]};
  }
  if (!workspace || workspace_bytes < vig::linear_wgrad_workspace(rows, l, count)) return VIG_ENOSPC;
  if (!room_for(later, 2 * count)) return VIG_EINVAL;
  return vig::launch_linear_wgrad(l, count, rows, workspace, later, (hipStream_t)stream);
}
int vig_linear_bwd_weight_many(const void* const* dy, const long long* dy_row_stride, const void* const* x, const long long* x_row_stride,
                               float* const* dweight, float* const* dbias, void* workspace, size_t workspace_bytes, long long rows,
                               const int* N, const int* K, int count, void* stream) {
  return vig_linear_bwd_weight_many_later(dy, dy_row_stride, x, x_row_stride, dweight, dbias, workspace, workspace_bytes, rows, N, K, count, nullptr, stream);
}

int vig_sum_jobs_run(vig_sum_jobs* jobs, void* stream) {
  if (!jobs || jobs->count < 0 || jobs->count > VIG_SUM_JOBS) return VIG_EINVAL;
  const int rc = vig::launch_sum_jobs(*jobs, (hipStream_t)stream);
  if (rc == VIG_OK) jobs->count = 0;
  return rc;
}

}  // extern "C"
