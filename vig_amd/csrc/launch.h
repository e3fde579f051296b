// Host-side argument block and launcher prototypes shared by the C ABI and the kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>

#include "../../include/vig_gla.h"

namespace vig {

struct GlaArgs {
  const void* q;
  const void* k;
  const void* v;
  const void* g_fwd;
  const void* g_bwd;  // may be null: forward direction only
  void* o;
  void* workspace;
  size_t workspace_bytes;
  int B, H, L, Dk, Dv;
  float scale, out_scale;
  int io_dtype, gate_dtype;  // 0 = f32, 1 = bf16
  hipStream_t stream;
  // fused locality gate (bf16 MFMA path only): o * sigmoid(conv3x3(o)) on the gate_rows x gate_cols token grid is
  // stored instead of o; weights [H*Dv, 9] f32.  Null: plain output.
  const float* gate_w = nullptr;
  int gate_rows = 0, gate_cols = 0;
  // bf16 MFMA path: the caller expects gates beyond the fp16 score variant's range (|chunk total| > ~8 nat in some
  // channel): start with the split-bf16 variant instead of finding out on the first segment of every workgroup
  int wide_gates = 0;
  // causal op only (g_bwd null): fp32 [B, H, Dk, Dv] state before the first token / after the last one; null: zero / not wanted
  const float* init_state = nullptr;
  float* final_state = nullptr;
  // bf16 MFMA path, Dk 64, both directions, any L: run the backward's state passes alone into `workspace`, per (sequence,
  // segment, direction) kGlaStateFloats floats, no scan, no outputs: the forward's pass on (k, v, gates) and, behind its slots,
  // the gradient-state pass on (q for k, `o` read as the output gradient for v, the two directions' gates exchanged,
  // cumulative gates exclusive of each token's own gate).
  int state_pass = 0;
  int state_segments = 0, state_seg_len = 0;  // the segmentation (at most 256 tokens each)
  // bf16 MFMA path: q, k, v that are not plain [B, H, L, D] tensors: element strides (batch, head, token) with the
  // channels of a (token, head) contiguous, e.g. column blocks of a projection output [B, L, H*(2*Dk + Dv)] read in
  // place.  Null (or token stride 0): plain layout.  Strides are multiples of 8 elements.
  const long long* q_strides = nullptr;
  const long long* k_strides = nullptr;
  const long long* v_strides = nullptr;
  // tile-pair and state kernels, Dk 32, both directions, strided q, k, v: gates made from rank-16 rows [B, L, 16] (low_ld elements apart) and
  // their second layer up_w [2 * H * Dk, 16], up_b, all bf16 (g_fwd, g_bwd are not read)
  const void *low = nullptr, *up_w = nullptr, *up_b = nullptr;
  long long low_ld = 0;
  float inv_norm = 0.f, clamp = 0.f;  // (clamp NaN: none)
};

// Per (sequence, segment, direction) slot of a state pass: the 64 x 64 state contribution in the matrix cores' register
// order (element ((u*64 + lane)*4 + m): unit u = (pk*2 + pv)*4 + cq), then the segment's 64 per-channel decays.
constexpr int kGlaStateFloats = 64 * 64 + 64;
// Segments of a long sequence: ceil(L / 256) of them, ceil(L / nseg) tokens each (the last one possibly fewer).
inline int gla_segments(int L) { return (L + 255) / 256; }
inline int gla_segment_len(int L) { return (L + gla_segments(L) - 1) / gla_segments(L); }
// The forward of a long sequence, when its output pass is the tile-pair kernel: segments of whole 32-token tiles, at
// most 7 of them (one wave each, two workgroups per CU); the last segment of a sequence may hold fewer tokens, down to
// none in its trailing tiles.
inline int gla_tile_segments(int L) { return (L + 223) / 224; }
inline int gla_tile_segment_tiles(int L) { return ((L + gla_tile_segments(L) - 1) / gla_tile_segments(L) + 31) / 32; }
// Behind the state slots of a scanned workspace: per (sequence, direction) 16 partial maxima of |state entering a
// segment| (one per block of the scan), for consumers that read the states as fp16.
constexpr int kGlaScanMaxima = 16;

// fp32 tensors and gates on the matrix cores (operands in three bf16 pieces): segments of up to seven 32-token tiles, as
// the tile-pair kernel cuts them, or, where those leave compute units idle (256 of them), of as few tiles as one workgroup a
// unit allows: a workgroup's time grows faster than its tiles.  us, segments of seven
// tiles / these: forward Dk 32 12 sequences of 1031 44.8 / 28.0, 36 of 1024 46.6 / 39.2, Dk 64 66 / 38.5 and 72 / 61.6; backward
// Dk 32 105 / 64 and 124 / 102, Dk 64 196 / 114 and 220 / 185.  (One tile more a segment than fits 256 units: 36 of 1024, Dk 64,
// backward 276.)  Whole sequences of seven tiles stay whole: 120 of 196, Dk 64, backward 141 / 153.
inline int gla_f32_segments(int L) { return gla_tile_segments(L); }
inline int gla_f32_segment_tiles(int L) { return gla_tile_segment_tiles(L); }
inline int gla_f32_fine_tiles(long long nseq, int L) {
  const int tiles = (L + 31) / 32;
  for (int NT = 2; tiles > 7 && NT < 7; ++NT)
    if (nseq * ((tiles + NT - 1) / NT) <= 256) return NT;
  return gla_f32_segment_tiles(L);
}
bool gla_f32_supported(const GlaArgs& a);
size_t gla_f32_workspace(int B, int H, int L, int Dk, int Dv, bool bidir);
size_t gla_f32_least_workspace(int B, int H, int L, int Dk, int Dv);
int launch_gla_f32(const GlaArgs& a);
// both sets of segment contributions of an fp32 backward: the states (k, v) and the gradient states (q, d_o)
// (flags, one int per sequence, are cleared on the way)
int launch_gla_f32_states(int NG, const float* k, const float* v, const float* q, const float* d_o, const float* gf,
                          const float* gb, float* slots, float* grad_slots, int* flags, int nseq, int L, int NT, int nseg, hipStream_t stream);
// fp32 backward on the matrix cores; one flag per sequence marks what it left to the recurrent kernel; the two sets of states go
// to two pieces of memory, either of which may be empty; a third one takes what else there may be room for
size_t gla_backward_f32_extra(int B, int H, int L, int Dk, int Dv);  // memory beyond gla_backward_workspace that speeds it up
bool gla_backward_f32_supported(int B, int H, int L, int Dk, int Dv, int io_dtype, int gate_dtype, bool bidir);
int launch_gla_backward_f32(const void* q, const void* k, const void* v, const void* gf, const void* gb, const void* d_o,
                            void* dq, void* dk, void* dv, void* dgf, void* dgb, int* flags, void* room0, size_t bytes0,
                            void* room1, size_t bytes1, void* room2, size_t bytes2, int B, int H, int L, int Dk, float s, hipStream_t stream);
// bf16: contributions and decays of every segment of seg_len tokens, and with q and d_o the gradient states (gla_states.hip)
int launch_gla_states(const GlaArgs& a, int seg_len, int nseg, float* slots, const void* q, const void* d_o, float* grad_slots);
// chains the slots of a state pass in place (gla_segment_scan_kernel, no state in or out), and those of another if there is one
int launch_gla_segment_scan(float* slots, float* more, int nseq, int nseg, int ndir, int ng, hipStream_t stream);

// Sums that kernels put off (wgrad.hip): false where the list is full.
inline bool put_off(vig_sum_jobs& jobs, const float* part, float* out, int rows, long long cols, bool fours) {
  if (jobs.count < 0 || jobs.count >= VIG_SUM_JOBS) return false;
  jobs.job[jobs.count++] = {part, out, cols, rows, fours};
  return true;
}
int launch_sum_jobs(const vig_sum_jobs& jobs, hipStream_t stream);

// Weight and bias gradients of up to kWgradLayers linear layers over the same T bf16 rows (wgrad.hip).
constexpr int kWgradLayers = 4;
struct LinearWgrad {
  const void *dy, *x;
  long long ldy, ldx;
  float *dw, *db;  // db may be null
  int N, K;
};
size_t linear_wgrad_workspace(long long T, const LinearWgrad* layers, int count);
int launch_linear_wgrad(const LinearWgrad* layers, int count, long long T, void* workspace, vig_sum_jobs* later, hipStream_t stream);

// Most tensors one launch_cast_many takes.
constexpr int kMaxCastJobs = 16;

// fp32-arithmetic token-recurrent path (any supported dtype combination).
int launch_gla_recurrent(const GlaArgs& a);
size_t gla_recurrent_workspace(int B, int H, int L, int Dv, int io_dtype);

// bf16 MFMA chunked path (bf16 io and gates).
bool gla_mfma_supported(const GlaArgs& a);
int launch_gla_mfma(const GlaArgs& a);
int launch_gla_lowrank(const GlaArgs& a);
int gla_strides(const GlaArgs& a, long long (&q)[3], long long (&k)[3], long long (&v)[3]);  // what q, k, v are read with; -22: none such
// bf16 tile-pair path for whole sequences (up to gla_slab_tokens): one wave per 32-token tile, both directions per wave.
bool gla_tiles_supported(const GlaArgs& a);
int gla_slab_tokens(int Dk);  // longest sequence that one workgroup takes whole
int launch_gla_tiles(const GlaArgs& a);
// the same kernel as the output pass of a longer sequence: one workgroup per (sequence, segment), the states
// entering the segments (scanned slots, kGlaStateFloats floats per (sequence, segment, direction)) and their maxima
// (kGlaScanMaxima floats per (sequence, direction)) in `states` / `maxima`
bool gla_tiles_chain_supported(const GlaArgs& a);
int launch_gla_tiles_chain(const GlaArgs& a, const float* states, const float* maxima);
bool gla_mfma_gate_grid_ok(int rows, int cols);  // token grids the fused locality gate takes
size_t gla_mfma_workspace(int B, int H, int L, int Dk, int Dv);
size_t gla_mfma_state_workspace(int B, int H, int L, int Dk, int Dv);  // causal op with an initial / final state

// bf16 matrix-core backward (quadratic form per slab, or per <= 256-token segment of a longer sequence with the
// segments chained through states); flags[b*H + h] = 1 marks sequences it left to the recurrent kernel.
// seg_workspace: gla_backward_mfma_workspace() bytes (seg_bytes), used for L > 256 only, and with it `scratch`, if there is room.
bool gla_backward_mfma_supported(int B, int H, int L, int Dk, int Dv, int io_dtype, int gate_dtype, bool bidir);
size_t gla_backward_mfma_workspace(int B, int H, int L, int Dk, int Dv);
int launch_gla_backward_mfma(const void* q, const void* k, const void* v, const void* gf, const void* gb,
                             const void* d_o, void* dq, void* dk, void* dv, void* dgf, void* dgb, int* flags,
                             void* scratch, size_t scratch_bytes, void* seg_workspace, size_t seg_bytes, int B, int H, int L,
                             int Dk, float s, long long ld_in, long long ld_out, hipStream_t stream);

// allows a kernel its LDS, once per device (concurrent first calls only repeat an idempotent setting)
inline bool allow_lds(const void* kernel, size_t bytes, bool (&done)[64]) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return false;
  if (!done[dev]) done[dev] = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) == hipSuccess;
  return done[dev];
}

// bf16 row products (gemm.hip, linear.hip): a layer whose weights stay in registers, and SwiGLU of a layer over few rows
bool linear_regs_supported(int K, int N);
int launch_linear_regs(const void* x, const void* w, const void* bias, void* y, long long T, int N, int K, hipStream_t stream);
int launch_linear_columns(const void* x, const void* w, void* y, long long T, int N, int K, hipStream_t stream);
int launch_linear_swiglu_bwd(const void* d_out, const void* w_down, const void* kept, void* d_kept, long long T, int K, int I,
                             hipStream_t stream);
bool norm_dwconv3x3_supported(int B, int h, int w, int C);
int launch_norm_dwconv3x3(const void* x, const void* residual, const float* norm, const float* wt, const float* bias, void* sum, void* y,
                          int B, int h, int w, int C, float eps, int silu, hipStream_t stream);
bool few_blend_linear(long long T, int C);
int launch_few_blend_linear(const void* o, const void* loc, const void* glin, const float* w_g, const float* w_l, const void* W, void* out,
                            void* kept, long long T, int L, int C, long long ldg, float eps, int silu_out, hipStream_t stream);
bool norm_conv_linear_supported(int B, int h, int w, int C, int N);
int launch_norm_conv_linear(const void* x, const void* residual, const float* norm, const float* taps, const float* conv_bias, const void* w,
                            const void* bias, void* sum, void* conv, void* y, int B, int h, int width, int C, int N, float eps, int silu,
                            hipStream_t stream);
bool blend_swiglu_supported(long long T, int C, int N);
int launch_blend_swiglu(const void* o, const void* loc, const void* glin, const float* w_g, const float* w_l, const void* w_out,
                        const void* residual, const float* norm, const void* w, void* sum, void* y, long long T, int L, int C, int N,
                        long long ldg, float eps, int silu_out, float norm_eps, hipStream_t stream);
bool norm_swiglu_supported(long long T, int K, int I);
int launch_norm_swiglu(const void* x, const void* residual, const float* norm, const void* w, void* sum, void* y, long long T, int K, int I,
                       float eps, hipStream_t stream);
bool linear_norm_supported(long long M, int N, int K);
int launch_linear_norm(const void* x, const void* w, const void* residual, const float* norm, void* y, void* sum, long long M, int N,
                       int K, float eps, hipStream_t stream);
bool few_swiglu(long long T, int K, int I);
int launch_few_swiglu(const void* x, const void* w, void* y, long long T, int K, int I, hipStream_t stream);

// Tokens a workgroup of 256 threads owns where every thread takes `each` octets of rows of nv octets (OctetRows).
inline int octet_tokens(int nv, int each) { return nv >= 256 * each ? 1 : 256 * each / nv; }
// ... and their workgroups, as many as one launch takes threads for (a workgroup of more tokens goes round more often); token rows are
// numbered in 32 bits
inline bool octet_rows_ok(int B, int L) { return (long long)B * L <= 0xffffffffLL; }
inline unsigned octet_grid(long long rows, int& tokens) {
  while ((rows + tokens - 1) / tokens > 0xffffff) tokens *= 2;
  return (unsigned)((rows + tokens - 1) / tokens);
}
// Octets a thread takes at once: four, whose loads are under way together, once that leaves four workgroups a compute unit.
inline int octets_each(long long rows, int nv) { return rows / octet_tokens(nv, 4) >= 1024 ? 4 : 1; }

}  // namespace vig
