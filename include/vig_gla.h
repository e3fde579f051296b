/*
 * vig_gla.h -- C ABI of the MI355X (gfx950) bidirectional gated-linear-attention
 * forward path of ViG and its two neighbours (direction-wise gate preparation,
 * 2D locality gate).
 *
 * Conventions shared by every entry point
 *   - every pointer is DEVICE memory owned by the caller; nothing is allocated,
 *     freed or synchronised inside; work is enqueued on `stream`
 *     (a hipStream_t passed as void*; NULL = the null stream);
 *   - tensors are dense row-major with the innermost dimension contiguous;
 *   - every tensor, weight vector and workspace starts on a 16-byte boundary
 *     (the kernels move 16 bytes per access); a pointer off it is VIG_EINVAL;
 *   - return value: 0 on success, a negative VIG_E* code otherwise
 *     (vig_gla_strerror() gives the text); a failed call enqueues nothing;
 *   - dtype codes: VIG_F32 = 0, VIG_BF16 = 1.
 *
 * Citations name the reference (hustvl/ViG) interface each entry point replaces.
 */
#ifndef VIG_GLA_H_
#define VIG_GLA_H_

#include <stddef.h>

#ifdef __cplusplus
extern "C" {
#endif

#define VIG_F32 0
#define VIG_BF16 1

#define VIG_OK 0
#define VIG_EINVAL (-22)  /* bad argument (null or misaligned pointer, non-positive size) */
#define VIG_ENOTSUP (-95) /* shape / dtype combination not built */
#define VIG_ENOSPC (-28)  /* workspace too small */
#define VIG_ELAUNCH (-5)  /* HIP reported a launch error */

/* Library identification: "vig_gla <version> gfx950". */
const char* vig_gla_version(void);
const char* vig_gla_strerror(int code);

/*
 * Bidirectional GLA forward, both directions in one call, natural token order.
 *
 *   S_i  = diag(exp(gf_i)) S_{i-1} + k_i v_i^T      (i = 0..L-1)
 *   S'_i = diag(exp(gb_i)) S'_{i+1} + k_i v_i^T     (i = L-1..0)
 *   o_i  = out_scale * (scale*q_i)^T (S_i + S'_i)
 *
 * q, k, g_fwd, g_bwd: [B, H, L, Dk]; v, o: [B, H, L, Dv].  g_* are natural-log
 * decays (<= 0).  g_bwd == NULL computes the forward direction only (the causal
 * op).  io_dtype is the type of q, k, v, o; gate_dtype the type of g_*.
 * `workspace` must hold vig_gla_bidir_fwd_workspace(...) bytes (may be NULL when
 * that is 0).
 *
 * Replaces: bid_fused_recurrent_gla (flash-linear-attention/fla/ops/gla/
 * recurrent_fuse.py:659-676, kernel :19-148; out_scale 1/2 from :442),
 * batch_bid_fused_chunk_gla (fla/ops/gla/chunk_fuse.py:574-596) and, with
 * g_bwd == NULL, fused_chunk_gla (chunk_fuse.py:554-572).
 *
 * Built shapes: Dk in {16, 32, 64, 128}, Dv in {32, 64, 128}, any L >= 1.
 *
 * Numeric range of the matrix-core paths (bf16 tensors and gates, Dk in {32, 64},
 * Dv = 64).  q, k and v may hold any finite bf16 values; the kernels check
 * magnitudes and gate totals themselves and switch arithmetic where needed:
 *   L <= 512 at Dk 32, 416 at Dk 64 (one workgroup per sequence, one wave per 32-token tile): fp16
 *   operands while every tile's gate total stays within about 7 (natural log
 *   units) per channel and rows of q / k / v have sums of squares below 2^15 /
 *   2^10 / 10^8; a sequence outside that is redone by the same workgroup with
 *   power-of-two input scales and split-bf16 diagonal tiles, good for gates down
 *   to about -5 per token (beyond: exponents are clamped, far tokens count as 0).
 *   longer (from 257 on for vig_gla_bidir_fwd_wide; segments of <= 224 tokens, seven tiles each, chained through states
 *   in the workspace: a state pass, a scan, then the kernel above once more per
 *   segment with the entering states; refused with VIG_ENOTSUP when
 *   B*H*directions > 65535): the same per-tile behaviour for the outputs, and for
 *   the state pass the sum of |g| over any 56 consecutive tokens of one channel
 *   must stay below about 80 (beyond it results may be inf / NaN, never silently
 *   wrong finite numbers).
 * HierViG's head shape (bf16, Dk = 16, Dv = 32, both directions) takes the same
 * paths from L = 128 on, zero-padded to Dk 32 / Dv 64 in the workspace
 * (classification/models/vig_h.py:377-385 with EXPAND_K 0.5, EXPAND_V 1.0).
 * fp32 tensors and gates with Dk in {32, 64}, Dv = 64: matrix-core kernels too, every operand in three bf16 pieces
 * (fp32 precision), any gates and magnitudes; sequences longer than 224 tokens as segments linked by states in the
 * workspace.  Other combinations run on the fp32-arithmetic token-recurrent kernel, which has no limit either.
 */
int vig_gla_bidir_fwd(const void* q, const void* k, const void* v,
                      const void* g_fwd, const void* g_bwd, void* o,
                      void* workspace, size_t workspace_bytes,
                      int B, int H, int L, int Dk, int Dv,
                      float scale, float out_scale,
                      int io_dtype, int gate_dtype, void* stream);

/*
 * vig_gla_bidir_fwd on q, k, v that are not plain [B, H, L, D] tensors: element (b, h, l, d) of q lies at
 * q + b*q_strides[0] + h*q_strides[1] + l*q_strides[2] + d (likewise k, v; the channels of one (token, head) are
 * contiguous).  For the column blocks of a projection output [B, L, H*(2*Dk + Dv)] read in place that is
 * {L*row, Dk (or Dv), row} with row = H*(2*Dk + Dv), so no head-major copies of q, k, v are made.  g_fwd, g_bwd and o
 * stay plain [B, H, L, D].  Strides are positive multiples of 8 elements (16-byte rows), the token stride at most 2^20.
 * Built for the matrix-core slab kernel only: bf16 tensors and gates, Dk in {32, 64}, Dv = 64, L <= 256 (no workspace);
 * VIG_ENOTSUP otherwise.  Same arithmetic and results as vig_gla_bidir_fwd on contiguous copies.
 *
 * Replaces: the stride arguments of the reference's kernels (s_qk_h, s_qk_t, s_qk_d, s_vo_h, s_vo_t, s_vo_d,
 * flash-linear-attention/fla/ops/gla/chunk_fuse.py:23-38), which its wrapper feeds with contiguous copies
 * (@contiguous, chunk_fuse.py:315) of the head-split views made at classification/models/vig.py:402-406 and :436-438.
 */
int vig_gla_bidir_fwd_strided(const void* q, const void* k, const void* v,
                              const void* g_fwd, const void* g_bwd, void* o,
                              int B, int H, int L, int Dk, int Dv,
                              const long long* q_strides, const long long* k_strides, const long long* v_strides,
                              float scale, float out_scale,
                              int io_dtype, int gate_dtype, void* stream);

/* Longest sequence that one workgroup takes whole, tensors in LDS (0: no such kernel for this Dk). */
int vig_gla_slab_tokens(int Dk);

/*
 * The kernel behind vig_gla_bidir_fwd, _strided and vig_gla_bidir_locgate_fwd at every length one launch takes
 * (L <= vig_gla_slab_tokens(Dk); those two stop at 256): strides as for _strided, each NULL for a plain tensor; with
 * gate_weight [H*Dv, 3, 3] f32 (NULL: none) the locality gate of vig_gla_bidir_locgate_fwd on a grid_h x grid_w token grid
 * (both directions, plain tensors, grid_w <= 126, a grid whose padded rows fit LDS).  VIG_ENOTSUP for anything else.  No workspace.
 */
int vig_gla_slab_fwd(const void* q, const void* k, const void* v, const void* g_fwd, const void* g_bwd,
                     const float* gate_weight, void* o, int B, int H, int L, int Dk, int Dv,
                     const long long* q_strides, const long long* k_strides, const long long* v_strides,
                     int grid_h, int grid_w, float scale, float out_scale, int io_dtype, int gate_dtype, void* stream);

/*
 * The bidirectional op with q, k, v read in place and the gates made on the way, as vig_dirgate_lowrank_fwd makes them (same
 * roundings), instead of read: low [B, L, 16] (rows low_row_stride elements apart), up_w [2*H*Dk, 16], up_b [2*H*Dk], clamp_min NaN
 * for none; all bf16.  Dk 32, Dv 64, all three strides given (as for _strided; token stride 0: that tensor is plain); VIG_ENOTSUP for
 * anything else.  Any length; past vig_gla_slab_tokens(32) tokens the workspace (vig_gla_lowrank_fwd_workspace bytes) holds the states
 * that link the segments, and 2*B*H > 65535 is refused with VIG_ENOTSUP.
 *
 * Replaces: classification/models/vig.py:401-435 (head split, gate up-projection, log-sigmoid, direction split, the op).
 */
size_t vig_gla_lowrank_fwd_workspace(int B, int H, int L, int Dk, int Dv);
int vig_gla_lowrank_fwd(const void* q, const void* k, const void* v, const void* low, long long low_row_stride,
                        const void* up_w, const void* up_b, void* o, void* workspace, size_t workspace_bytes,
                        int B, int H, int L, int Dk, int Dv,
                        const long long* q_strides, const long long* k_strides, const long long* v_strides,
                        float inv_norm, float clamp_min, float scale, float out_scale, int io_dtype, void* stream);

/* Workspace that is enough for every gate dtype and for one or two directions (the largest over the kernels the
 * call may dispatch to for this shape and io_dtype). */
size_t vig_gla_bidir_fwd_workspace(int B, int H, int L, int Dk, int Dv, int io_dtype);
/* Workspace of exactly the kernel vig_gla_bidir_fwd / _wide dispatch to for these arguments (bidirectional: g_bwd
 * given): 0 for bf16 tensors and gates with Dk in {32, 64}, Dv = 64, L <= 256 (between 257 tokens and the one-launch
 * kernel's limit only _wide uses it, but both ask for it).  fp32 tensors take quicker forms in this much than in less: shorter
 * segments, or whole sequences as two halves, the sums in another order (equal within fp32 rounding); with the same
 * number of bytes a call gives the same bits. */
size_t vig_gla_bidir_fwd_workspace_for(int B, int H, int L, int Dk, int Dv, int io_dtype, int gate_dtype,
                                       int bidirectional);

/*
 * The causal op (one direction) with a state carried in and / or out:
 *   S_{-1} = initial_state (zero when NULL);  S_i = diag(exp(g_i)) S_{i-1} + k_i v_i^T;  o_i = out_scale * (scale*q_i)^T S_i;
 *   final_state = S_{L-1} (not written when NULL).
 * initial_state, final_state: fp32 [B, H, Dk, Dv], row-major (k channel, then v channel); same tensors, dtypes and
 * shapes as vig_gla_bidir_fwd with g_bwd == NULL.  bf16 tensors and gates with Dk in {32, 64}, Dv = 64 run on the
 * matrix cores as chained segments of up to 256 tokens (state contributions, a scan that starts from initial_state
 * and ends in final_state, outputs); everything else on the fp32-arithmetic token-recurrent kernel.
 * `workspace` must hold vig_gla_causal_state_fwd_workspace(...) bytes (may be NULL when that is 0).
 *
 * Replaces: fused_chunk_gla with initial_state / output_final_state (flash-linear-attention/fla/ops/gla/
 * chunk_fuse.py:554-572; the state enters at :70-72 and leaves at :99-101) and fused_recurrent_gla with the same
 * arguments (fla/ops/gla/recurrent_fuse.py:631-657, kernel :213-218,240-246).
 */
int vig_gla_causal_state_fwd(const void* q, const void* k, const void* v, const void* g, void* o,
                             const float* initial_state, float* final_state,
                             void* workspace, size_t workspace_bytes,
                             int B, int H, int L, int Dk, int Dv,
                             float scale, float out_scale,
                             int io_dtype, int gate_dtype, void* stream);
size_t vig_gla_causal_state_fwd_workspace(int B, int H, int L, int Dk, int Dv, int io_dtype, int gate_dtype);
/* Same contract, always the fp32-arithmetic token-recurrent kernel whatever the dtypes (no workspace): the counterpart
 * of fused_recurrent_gla's state arguments (fla/ops/gla/recurrent_fuse.py:631-657). */
int vig_gla_causal_state_fwd_exact(const void* q, const void* k, const void* v, const void* g, void* o,
                                   const float* initial_state, float* final_state,
                                   int B, int H, int L, int Dk, int Dv,
                                   float scale, float out_scale,
                                   int io_dtype, int gate_dtype, void* stream);

/*
 * Same contract, workspace and accuracy bar as vig_gla_bidir_fwd, for callers who know their gates to be strong.
 * The matrix-core kernel computes on fp16 operands while every 32-token tile's gate total stays within about 7
 * (natural log units) in every channel, and in its wider-range form beyond; it finds out per sequence (or segment),
 * after preparing the fp16 operands in vain, and redoes it at about four times the cost.  This entry point runs the
 * wider-range form alone, in a kernel of its own with twice the registers: about 1.65 times the fp16 form's time
 * whatever the gates (60 against 37 us at B128 H6 L196 Dk64), against 3.8 times through the default entry point when
 * every sequence refuses.  No counterpart
 * in the reference, whose kernels have one arithmetic (fla/ops/gla/chunk_fuse.py:25-101,212-254).
 */
int vig_gla_bidir_fwd_wide(const void* q, const void* k, const void* v,
                           const void* g_fwd, const void* g_bwd, void* o,
                           void* workspace, size_t workspace_bytes,
                           int B, int H, int L, int Dk, int Dv,
                           float scale, float out_scale,
                           int io_dtype, int gate_dtype, void* stream);

/*
 * vig_gla_bidir_fwd without a workspace argument, for callers that cannot allocate device memory: code under
 * HIP graph capture, tight serving loops, harnesses that forbid hipMalloc.  Same tensors, dispatch, kernels and
 * results (bit for bit) as vig_gla_bidir_fwd with vig_gla_bidir_fwd_workspace_for(...) bytes; the workspace is a device array inside the library,
 * VIG_GLA_NOALLOC_SCRATCH_BYTES per GPU, held from the first call on that GPU until the process ends.  A shape whose
 * vig_gla_bidir_fwd_workspace_for(...) exceeds that size returns VIG_ENOSPC and launches nothing (then use
 * vig_gla_bidir_fwd with a workspace of the caller's).  Calls no hipMalloc / hipFree and nothing else that allocates.
 * All calls on one GPU share the one array, fp32 calls on whole sequences too: calls that overlap in time on the same GPU (two
 * streams, two threads) race on it; serialise them.  The tensors must live on the current device (another device's pointers: VIG_EINVAL).
 * Under HIP graph capture: make one call per device and shape class outside the capture first.  The first call on a
 * device looks up the array's address and sets the kernels' shared-memory attribute (no stream work, but not capturable
 * either); every later call is kernel launches on `stream` only.  It has no counterpart in the reference, whose ops
 * allocate their temporaries through torch (flash-linear-attention/fla/ops/gla/chunk_fuse.py:325-345).
 */
#define VIG_GLA_NOALLOC_SCRATCH_BYTES (16u << 20)
int vig_gla_bidir_fwd_noalloc(const void* q, const void* k, const void* v,
                              const void* g_fwd, const void* g_bwd, void* o,
                              int B, int H, int L, int Dk, int Dv,
                              float scale, float out_scale,
                              int io_dtype, int gate_dtype, void* stream);
size_t vig_gla_bidir_fwd_noalloc_max_workspace(void);

/*
 * Same contract as vig_gla_bidir_fwd, but always runs the fp32-arithmetic
 * token-recurrent kernel whatever the dtypes (bf16 tensors are widened on load,
 * the state and all sums stay fp32).  This is the op-level counterpart of the
 * reference's recurrent kernels (fla/ops/gla/recurrent_fuse.py:19-148,152-246),
 * kept callable for callers that want fp32 state arithmetic on bf16 tensors.
 * Workspace: B*H*L*Dv*4 bytes when io_dtype is bf16 and g_bwd != NULL, else 0.
 */
int vig_gla_bidir_fwd_exact(const void* q, const void* k, const void* v,
                            const void* g_fwd, const void* g_bwd, void* o,
                            void* workspace, size_t workspace_bytes,
                            int B, int H, int L, int Dk, int Dv,
                            float scale, float out_scale,
                            int io_dtype, int gate_dtype, void* stream);

/*
 * Backward of vig_gla_bidir_fwd: given d_o = dL/do [B, H, L, Dv], writes
 *   dq, dk [B, H, L, Dk], dv [B, H, L, Dv] (summed over the directions) in io_dtype and
 *   dg_fwd, dg_bwd [B, H, L, Dk] in gate_dtype (dg_bwd only when g_bwd != NULL).
 * `workspace` must hold vig_gla_bidir_bwd_workspace(...) bytes.
 * Built shapes: (Dk, Dv) in {(16,32), (32,32), (32,64), (64,32), (64,64)}, any L >= 1.
 * Dispatch: bf16 tensors + bf16 gates + Dk in {32, 64} + Dv = 64 (both directions, or the causal op with
 * g_bwd == NULL) -> matrix-core kernel (bf16 operands, fp32 accumulation; gradients within ~1e-2 of their largest
 * magnitude): one quadratic form per (batch, head) for L <= 256; a longer sequence as segments of <= 256 tokens linked
 * by their states (two state passes of the forward kernel, a segment scan, then one quadratic form per segment;
 * B*H*directions <= 65535).  fp32 tensors and gates with the same head widths -> matrix-core kernel on operands in
 * three bf16 pieces (fp32 precision).  A sequence with a segment whose gate total exceeds ~83 in some channel (fp32: a
 * 32-token tile with a total beyond ~28, or values beyond 1e12), and every other case -> fp32-arithmetic token-recurrent
 * kernel.
 *
 * Replaces: FusedChunkGLAFunction.backward (flash-linear-attention/fla/ops/gla/chunk_fuse.py:413-518; gate
 * gradient :505-518) under the flip-concat glue of classification/models/vig.py:407-426, for both directions in
 * natural token order.
 */
int vig_gla_bidir_bwd(const void* q, const void* k, const void* v,
                      const void* g_fwd, const void* g_bwd, const void* d_o,
                      void* dq, void* dk, void* dv, void* dg_fwd, void* dg_bwd,
                      void* workspace, size_t workspace_bytes,
                      int B, int H, int L, int Dk, int Dv,
                      float scale, float out_scale,
                      int io_dtype, int gate_dtype, void* stream);

size_t vig_gla_bidir_bwd_workspace(int B, int H, int L, int Dk, int Dv, int bidirectional);

/*
 * Workspace of the path vig_gla_bidir_bwd takes for exactly these dtypes.  It differs from the query above for
 * HierViG's head shape (Dk 16, Dv 32; classification/models/vig_h.py:521-527) with bf16 tensors and gates, both
 * directions and L >= 128: given this many bytes, the backward runs zero-padded to 32 / 64 channels on the matrix-core
 * kernels (inputs padded, gradients cropped; 20x faster than the token-recurrent kernel at L = 3136); given only the
 * smaller amount of the query above, it runs on the token-recurrent kernel.
 */
size_t vig_gla_bidir_bwd_workspace_for(int B, int H, int L, int Dk, int Dv, int io_dtype, int gate_dtype,
                                       int bidirectional);

/*
 * vig_gla_bidir_bwd for q, k, v in the columns of a matrix [B * L, row_stride], head h's channels at q + h*Dk, k + h*Dk and v + h*Dv of a token's
 * row, and dq, dk, dv likewise in one of d_row_stride; the other tensors and the workspace as there, and the same results.  Both directions,
 * bf16 tensors and gates, Dk in {32, 64}, Dv = 64, L <= 256; VIG_ENOTSUP otherwise.  Row strides are multiples of 8 up to 2^20 elements.
 *
 * Replaces: the backward of the head split (classification/models/vig.py:401-409) around that of the op.
 */
int vig_gla_bidir_bwd_rows(const void* q, const void* k, const void* v, long long row_stride, const void* g_fwd, const void* g_bwd, const void* d_o,
                           void* dq, void* dk, void* dv, long long d_row_stride, void* dg_fwd, void* dg_bwd, void* workspace, size_t workspace_bytes,
                           int B, int H, int L, int Dk, int Dv, float scale, float out_scale, int io_dtype, int gate_dtype, void* stream);

/* Same contract as vig_gla_bidir_bwd, always the fp32-arithmetic token-recurrent kernel (the exact path). */
int vig_gla_bidir_bwd_exact(const void* q, const void* k, const void* v,
                            const void* g_fwd, const void* g_bwd, const void* d_o,
                            void* dq, void* dk, void* dv, void* dg_fwd, void* dg_bwd,
                            void* workspace, size_t workspace_bytes,
                            int B, int H, int L, int Dk, int Dv,
                            float scale, float out_scale,
                            int io_dtype, int gate_dtype, void* stream);

/*
 * Direction-wise gate preparation.
 *   gk_lin [B, L, 2*H*Dk]  ->  g_out [2, B, H, L, Dk]
 *   g_out[dir,b,h,l,d] = max(logsigmoid(gk_lin[b,l,dir*H*Dk + h*Dk + d]) * inv_normalizer, clamp_min)
 * clamp_min = NaN disables the clamp.  g_out[0] / g_out[1] are the g_fwd / g_bwd
 * arguments of vig_gla_bidir_fwd.
 *
 * Replaces: classification/models/vig.py:432-441 (chunk(2), cat, rearrange,
 * logsigmoid / gate_logit_normalizer, clamp_min).
 */
int vig_dirgate_fwd(const void* gk_lin, void* g_out, int B, int L, int H, int Dk,
                    float inv_normalizer, float clamp_min,
                    int in_dtype, int out_dtype, void* stream);

/*
 * Backward of vig_dirgate_fwd: d_g [2, B, H, L, Dk] (type out_dtype) -> d_gk_lin [B, L, 2*H*Dk] (type in_dtype),
 *   d_gk_lin = d_g * inv_normalizer * sigmoid(-gk_lin), zero where the forward clamped.
 *
 * Replaces: what autograd derives for classification/models/vig.py:368-371,411-414 (logsigmoid, division, clamp,
 * the direction split and the head rearrange).
 */
int vig_dirgate_bwd(const void* gk_lin, const void* d_g, void* d_gk_lin, int B, int L, int H, int Dk,
                    float inv_normalizer, float clamp_min, int in_dtype, int out_dtype, void* stream);

/*
 * Direction-wise gate preparation with the second layer of the low-rank gate projection inside:
 *   gk_low [B, L, rank] (token rows low_row_stride elements apart, 0 = packed), w_up [2*H*Dk, rank], b_up [2*H*Dk]
 *   x = gk_low . w_up^T + b_up, rounded to in_dtype (what the separate layer would have stored);
 *   g_out [2, B, H, L, Dk] as in vig_dirgate_fwd.  gk_low, w_up and b_up share in_dtype; rank must be 16; bases and
 *   row strides in bytes must be multiples of 16.  The [B, L, 2*H*Dk] intermediate never goes to memory.
 *
 * Replaces: the second nn.Linear of gk_proj (classification/models/vig.py:296-297, applied at vig.py:432) together
 * with vig.py:432-441.
 */
int vig_dirgate_lowrank_fwd(const void* gk_low, long long low_row_stride, const void* w_up, const void* b_up,
                            void* g_out, int B, int L, int H, int Dk, int rank, float inv_normalizer, float clamp_min,
                            int in_dtype, int out_dtype, void* stream);
/*
 * Backward of vig_dirgate_lowrank_fwd for bf16 rows: d_g [2, B, H, L, Dk] (type out_dtype) ->
 *   d_x [B*L, 2*H*Dk] bf16, the gradient at the up-projection's result (its weight gradient is d_x^T gk_low),
 *   d_low [B*L, rank] bf16, rows d_low_row_stride elements apart (0 = packed) = d_x w_up.
 * w_up_t is w_up transposed, [rank, 2*H*Dk].  Dk % 16 == 0, rank 16, in_dtype VIG_BF16.
 *
 * Replaces: what autograd derives for classification/models/vig.py:432-441 and the second gk_proj layer in front.
 */
int vig_dirgate_lowrank_bwd(const void* gk_low, long long low_row_stride, const void* w_up, const void* w_up_t,
                            const void* b_up, const void* d_g, void* d_x, void* d_low, long long d_low_row_stride, int B,
                            int L, int H, int Dk, int rank, float inv_normalizer, float clamp_min, int in_dtype,
                            int out_dtype, void* stream);

/*
 * Up to 16 small tensors converted in one launch: dst[j] (type dst_dtype[j]) gets the n[j] elements of src[j] (type
 * src_dtype[j]); zeros where src[j] is NULL; transposed where transposed_cols[j] > 0 (src is [n/cols, cols], dst
 * [cols, n/cols]).  What a training step needs of a block's weights after the optimiser has changed them.
 */
int vig_cast_many(const void* const* src, void* const* dst, const int* n, const int* transposed_cols, const int* src_dtype,
                  const int* dst_dtype, int count, void* stream);


/*
 * 3x3 depthwise convolution on the token grid, channels-last, zero padding 1.
 *   x [B, L=h*w, C], weight [C, 3, 3] (f32), bias [C] (f32) or NULL -> y [B, L, C]
 *   optional SiLU on the result.
 *
 * Replaces: the in_proj of GatedLinearAttention (classification/models/vig.py:
 * 291-294 applied at :428-430 with the two permutes around it).
 */
int vig_dwconv3x3_fwd(const void* x, const float* weight, const float* bias, void* y,
                      int B, int h, int w, int C, int silu, int io_dtype, void* stream);
/* The same; with silu, `pre` (may be NULL) also receives the stored result in front of the activation, and the activation
 * reads that stored value (what a backward needs). */
int vig_dwconv3x3_fwd_pre(const void* x, const float* weight, const float* bias, void* y, void* pre, int B, int h, int w,
                          int C, int silu, int io_dtype, void* stream);


/*
 * Weight and bias gradients of vig_dwconv3x3_fwd (without its SiLU) from x and dy [B, h*w, C]:
 *   dw_db fp32 [C*9 + C]: dw[c, ky, kx] = sum dy[b, y, x, c] * x[b, y+ky-1, x+kx-1, c], then db[c] = sum dy[b, y, x, c].
 * `workspace` holds vig_dwconv3x3_bwd_weight_workspace(B, C) bytes
 * (per-workgroup partial sums, added in a fixed order: no atomics).
 *
 * Replaces: the convolution library's depthwise weight-gradient call behind classification/models/vig.py:291-294.
 */
size_t vig_dwconv3x3_bwd_weight_workspace(int B, int C);
int vig_dwconv3x3_bwd_weight(const void* x, const void* dy, float* dw_db, void* workspace, size_t workspace_bytes,
                             int B, int h, int w, int C, int io_dtype, void* stream);
/* Both gradients in one pass over x and dy: dx (NULL to skip it) and dw_db (NULL to skip it, then no workspace).  With
 * `pre` (see vig_dwconv3x3_fwd_pre) dy is the gradient behind the SiLU and is taken through it first, rounded to the
 * storage type. */
int vig_dwconv3x3_bwd(const void* x, const void* dy, const void* pre, const float* weight, void* dx, float* dw_db,
                      void* workspace, size_t workspace_bytes, int B, int h, int w, int C, int io_dtype, void* stream);


/*
 * Synthetic locality gate of the ViG-B benchmark shape:
 *   y[b,hd,l,d] = o[b,hd,l,d] * sigmoid( dwconv3x3(o on the h x w grid, channel c = hd*Dv+d) )
 * o, y: [B, H, L=h*w, Dv]; weight [H*Dv, 3, 3] f32.  In-place (y == o) is NOT allowed.
 */
int vig_locality_gate_fwd(const void* o, const float* weight, void* y,
                          int B, int H, int h, int w, int Dv, int io_dtype, void* stream);

/*
 * vig_gla_bidir_fwd and vig_locality_gate_fwd in one call: the GLA output o = out_scale * (o_fwd + o_bwd) is
 * rounded to bf16, staged on chip, and y = o * sigmoid(dwconv3x3(o)) is what reaches memory (bit-identical to the
 * two calls in a row); of few sequences of 129 to 256 tokens, which the op spreads over the chip, the op's output does, and a second
 * launch gates it in place.  Same tensors as vig_gla_bidir_fwd; weight [H*Dv, 3, 3] f32; L = grid_h * grid_w.
 * Built for bf16 tensors and gates, Dk in {32, 64}, Dv = 64, L <= 256, both directions, and token grids with
 * grid_w <= 62 and grid_h + 2 <= 8 * floor(64 / (grid_w + 2)) (14x14 and 16x16 are); VIG_ENOTSUP otherwise
 * (the caller then makes the two calls).  No workspace.
 *
 * Replaces: the GLA call of classification/models/vig.py:442 followed by the benchmark's sigmoid locality gate
 * (the synthetic restatement of vig.py:291-294,447-454 on the op's own output).
 */
int vig_gla_bidir_locgate_fwd(const void* q, const void* k, const void* v, const void* g_fwd, const void* g_bwd,
                              const float* gate_weight, void* y, int B, int H, int L, int Dk, int Dv,
                              int grid_h, int grid_w, float scale, float out_scale, int io_dtype, int gate_dtype,
                              void* stream);

/*
 * Block epilogue before o_proj:
 *   y[b,l,hd*Dv+d] = rms(o[b,hd,l,:])*w_g * s + rms(local[b,l,hd,:])*w_l * (1-s),  s = sigmoid(g_lin[b,l,hd*Dv+d])
 *   rms(x) = x * rsqrt(mean(x^2) + eps); optional SiLU on y.
 * o [B,H,L,Dv]; local, g_lin, y [B, L, H*Dv]; w_g, w_l [Dv] f32.
 * g_row_stride: elements between consecutive token rows of g_lin (0 = packed, H*Dv), so that g_lin may be a block
 * of columns of a wider projection output; the base and the stride in bytes must be multiples of 16.
 *
 * Replaces: classification/models/vig.py:444-457 (two RMSNorm launches
 * fla/modules/rmsnorm.py:69-125, three rearranges, sigmoid blend, out_act).
 */
int vig_locality_blend_fwd(const void* o, const void* local, const void* g_lin,
                           const float* w_g, const float* w_l, void* y,
                           int B, int H, int L, int Dv, long long g_row_stride, float eps, int silu_out,
                           int io_dtype, void* stream);

/*
 * Backward of vig_locality_blend_fwd from the forward's inputs and dy [B, L, H*Dv]:
 *   d_o [B, H, L, Dv], d_local and d_glin [B, L, H*Dv] (packed), dw fp32 [2, Dv] = (gradient of w_g | of w_l).
 * With s = sigmoid(g_lin), on = rms(o) * w_g, ln = rms(local) * w_l, y0 = on * s + ln * (1 - s):
 *   dy0 = dy * d(y)/d(y0) (SiLU derivative when silu_out), d_on = dy0 * s, d_ln = dy0 * (1 - s),
 *   d_glin = dy0 * (on - ln) * s * (1 - s); d_o and d_local are the RMS-norm backward of d_on and d_ln per
 *   (token, head) row; dw sums d_on * o * r_o and d_ln * local * r_l over batch, tokens and heads.
 * `workspace` holds vig_locality_blend_bwd_workspace(B, L, Dv) bytes (per-workgroup partial sums of dw, added in a
 * fixed order: no atomics).
 *
 * Replaces: what autograd derives for classification/models/vig.py:447-457 in the reference (two fused RMS-norm
 * backward launches, rmsnorm.py:203-296, and the elementwise chain of the blend).
 */
size_t vig_locality_blend_bwd_workspace(int B, int L, int Dv);
int vig_locality_blend_bwd(const void* o, const void* local, const void* g_lin, const float* w_g, const float* w_l,
                           const void* dy, void* d_o, void* d_local, void* d_glin, float* dw, void* workspace,
                           size_t workspace_bytes, int B, int H, int L, int Dv, long long g_row_stride, float eps,
                           int silu_out, int io_dtype, void* stream);
/* The same with d_glin's rows d_glin_row_stride elements apart (0 = packed). */
int vig_locality_blend_bwd_strided(const void* o, const void* local, const void* g_lin, const float* w_g, const float* w_l,
                                   const void* dy, void* d_o, void* d_local, void* d_glin, float* dw, void* workspace,
                                   size_t workspace_bytes, int B, int H, int L, int Dv, long long g_row_stride,
                                   long long d_glin_row_stride, float eps, int silu_out, int io_dtype, void* stream);


/*
 * Residual-add + RMS norm over the last dimension (rows x C, C % 8 == 0, C <= 4096):
 *   s = x (+ residual) in fp32;  residual_out = s (if not NULL);  y = s * rsqrt(mean(s^2) + eps) * weight
 * residual and residual_out may be NULL; weight [C] f32.  round_sum != 0 first rounds s to the storage
 * type and normalises the rounded value (what `norm(a + b)` on stored tensors computes); round_sum == 0
 * is the fused kernel's arithmetic (the unrounded sum is normalised).
 *
 * Replaces: flash-linear-attention/fla/modules/rmsnorm.py:69-125 (_layer_norm_fwd_1pass_kernel with
 * IS_RMS_NORM, HAS_RESIDUAL, STORE_RESIDUAL_OUT) as used at classification/models/vig.py:598,602-606,896.
 */
int vig_rmsnorm_fwd(const void* x, const void* residual, const float* weight, void* y, void* residual_out,
                    long long rows, int C, float eps, int round_sum, int io_dtype, void* stream);
/* The same with a type for each role: residual and sum of sum_dtype, x of x_dtype, y of y_dtype.  One type throughout, or an
 * fp32 sum with a bf16 y (a bf16 branch meeting the fp32 stream under autocast). */
int vig_rmsnorm_mixed_fwd(const void* x, const void* residual, const float* weight, void* y, void* residual_out,
                          long long rows, int C, float eps, int round_sum, int x_dtype, int sum_dtype, int y_dtype,
                          void* stream);


/*
 * LayerNorm over the last dimension (rows x C, C % 8 == 0, C <= 4096), optional SiLU behind it:
 *   y = (x - mean) * rsqrt(var + eps) * weight + bias   (biased variance, fp32 arithmetic; weight, bias [C] f32)
 *   silu != 0:  y = r * sigmoid(r) with r the normalised value rounded to the storage type
 *   pre_bias [C] f32 or NULL: x + pre_bias, rounded to the storage type, is what gets normalised (the bias of the
 *     convolution in front of the norm);
 *   post_add [post_rows, C] (io dtype) or NULL: row r of the (rounded) result gets post_add[r % post_rows] added
 *     (the position table behind the last norm, post_rows = tokens per image).
 * x and y may be the same buffer.
 *
 * Replaces: LayerNorm2d of the v2 patch embedding on a channels-last feature map with the bias add of the
 * convolution before it, the swish that follows the first one (classification/models/vig.py:619-624, 650-655) and
 * the position-table add behind the second (vig.py:858-865).
 */
int vig_layernorm_fwd(const void* x, const float* weight, const float* bias, void* y, long long rows, int C,
                      float eps, int silu, const float* pre_bias, const void* post_add, int post_rows, int io_dtype,
                      void* stream);

/*
 * Head-major split of the fused q/k/v projection:
 *   qkv [B, L, H*Dk | H*Dk | H*Dv]  ->  q, k [B, H, L, Dk],  v [B, H, L, Dv]   (Dk, Dv multiples of 8)
 * qkv_row_stride: elements between consecutive token rows of qkv (0 = packed), so that qkv may be the leading
 * columns of a wider projection output; the base and the stride in bytes must be multiples of 16.
 *
 * Replaces: classification/models/vig.py:401-409 (torch.split and the three 'b l (h d) -> b h l d'
 * rearranges in front of the GLA op).
 */
int vig_split_heads_fwd(const void* qkv, void* q, void* k, void* v, int B, int L, int H, int Dk, int Dv,
                        long long qkv_row_stride, int io_dtype, void* stream);

/*
 * Backward of vig_split_heads_fwd: dq, dk [B, H, L, Dk] and dv [B, H, L, Dv] gathered into d_qkv
 * [B, L, H*(2*Dk+Dv)] (packed rows), one pass.
 *
 * Replaces: what autograd derives for classification/models/vig.py:401-409 (three rearranges back and a concat).
 */
int vig_split_heads_bwd(const void* dq, const void* dk, const void* dv, void* d_qkv, int B, int L, int H, int Dk,
                        int Dv, int io_dtype, void* stream);
/* The same with d_qkv's rows d_qkv_row_stride elements apart (0 = packed): the columns of a wider matrix. */
int vig_split_heads_bwd_strided(const void* dq, const void* dk, const void* dv, void* d_qkv, long long d_qkv_row_stride,
                                int B, int L, int H, int Dk, int Dv, int io_dtype, void* stream);


/*
 * SwiGLU product of the MLP:  gate_up [rows, 2*I] = (gate | up)  ->  out [rows, I] = gate * up / (1 + exp(-gate))
 *
 * Replaces: swiglu_fwd (flash-linear-attention/fla/modules/activations.py:109-113) on the two halves of
 * gate_proj's output (classification/models/vig.py:492-495).
 */
int vig_swiglu_fwd(const void* gate_up, void* out, long long rows, int I, int io_dtype, void* stream);

/*
 * Backward of vig_swiglu_fwd: d_gate_up [rows, 2*I] = (d_gate | d_up) from the forward's input and dy [rows, I]:
 *   d_gate = dy * up * sig(gate) * (1 + gate * (1 - sig(gate))),  d_up = dy * gate * sig(gate).
 *
 * Replaces: swiglu_bwd (flash-linear-attention/fla/modules/activations.py:113-119, used by SwiGLUFunction :137-148).
 */
int vig_swiglu_bwd(const void* gate_up, const void* dy, void* d_gate_up, long long rows, int I, int io_dtype,
                   void* stream);

/*
 * Backward of vig_rmsnorm_fwd.  `sum` [rows, C] is the tensor the forward normalised (x, or the x + residual it
 * returned), dy the gradient of y, d_sum (may be NULL) the gradient that arrives at the returned sum:
 *   r = rsqrt(mean(sum^2) + eps),  g = dy * weight,
 *   ds = r * (g - sum * r^2 * mean(g * sum)) + d_sum     -- the gradient of x and of the residual alike
 *   dweight[c] = sum over rows of dy[c] * sum[c] * r     -- fp32 [C]; NULL skips it (and needs no workspace)
 * `workspace` holds vig_rmsnorm_bwd_workspace(rows, C) bytes of per-workgroup partial sums; the result does not
 * depend on scheduling (no atomics).  C % 8 == 0, C <= 1024.
 *
 * Replaces: _layer_norm_bwd_kernel in its RMS mode with residual
 * (flash-linear-attention/fla/modules/rmsnorm.py:203-296, driver :300-387).
 */
size_t vig_rmsnorm_bwd_workspace(long long rows, int C);
int vig_rmsnorm_bwd(const void* sum, const float* weight, const void* dy, const void* d_sum, void* ds, float* dweight,
                    void* workspace, size_t workspace_bytes, long long rows, int C, float eps, int io_dtype,
                    void* stream);
/* The same with a type for each role (see vig_rmsnorm_mixed_fwd); dx (may be NULL) receives ds in y_dtype, for a branch of
 * that type. */
int vig_rmsnorm_mixed_bwd(const void* sum, const float* weight, const void* dy, const void* d_sum, void* ds, void* dx,
                          float* dweight, void* workspace, size_t workspace_bytes, long long rows, int C, float eps,
                          int sum_dtype, int y_dtype, void* stream);


/*
 * gate_proj and the SwiGLU product in one kernel, for a short contraction (K = 384 or 192, the hidden sizes of
 * ViG-S / ViG-T), bf16, fp32 accumulation:
 *   y [rows, I] = swiglu(gate, up) with (gate | up) = x [rows, K] . weight [2*I, K]^T, the product taken on gate and
 *   up rounded to bf16 (what the separate layer stores); I % 32 == 0; x, weight and y packed row-major.
 * Other K or dtypes return VIG_ENOTSUP (use a GEMM library and vig_swiglu_fwd).
 *
 * Replaces: gate_proj followed by swiglu (classification/models/vig.py:492-495,
 * flash-linear-attention/fla/modules/activations.py:109-113) without the [rows, 2*I] intermediate.
 */
int vig_linear_swiglu_fwd(const void* x, const void* weight, void* y, long long rows, int K, int I, int io_dtype,
                          void* stream);
/* The same, leaving gate | up as well: gate_up [rows, 2*I], what the backward of the product reads. */
int vig_linear_swiglu_kept_fwd(const void* x, const void* weight, void* gate_up, void* y, long long rows, int K, int I,
                               int io_dtype, void* stream);
/*
 * The input gradient of down_proj and the backward of the SwiGLU product in one kernel: d = d_out [rows, K] . w_down [K, I] rounded
 * to bf16, d_gate_up [rows, 2*I] as vig_swiglu_bwd gives it for (gate_up, d).  K = 384 or 192, I % 32 == 0, bf16.
 */
int vig_linear_swiglu_bwd(const void* d_out, const void* w_down, const void* gate_up, void* d_gate_up, long long rows, int K, int I,
                          int io_dtype, void* stream);
/*
 * The input gradient of a linear layer, dx [rows, K] = dy [rows, N] . weight [N, K], bf16, fp32 accumulation; N = 384 or 192,
 * K % 64 == 0 (else VIG_ENOTSUP).  _preferred: whether it is the better choice next to a BLAS library.
 */
int vig_linear_bwd_input_preferred(long long rows, int N, int K);
int vig_linear_bwd_input(const void* dy, const void* weight, void* dx, long long rows, int N, int K, int io_dtype, void* stream);

/*
 * vig_locality_blend_fwd and o_proj in one kernel, for square blocks with 64-channel heads at the widths whose weight
 * tiles fit the registers (C = H*Dv = 384 or 192, the hidden sizes of ViG-S / ViG-T), bf16, fp32 accumulation:
 *   out [B*L, C] = y . weight [C, H*Dv]^T with y the blend above, rounded to bf16 as vig_locality_blend_fwd stores
 *   it; y itself is never written.  Arguments as in vig_locality_blend_fwd (Dv = 64, g_row_stride likewise);
 *   weight and out packed row-major.  Other shapes or dtypes return VIG_ENOTSUP (make the two calls).
 *
 * Replaces: classification/models/vig.py:444-463 (head norms, sigmoid blend, out_act, o_proj) without the
 * [B, L, H*Dv] intermediate.
 */
int vig_locality_blend_linear_fwd(const void* o, const void* local, const void* g_lin,
                                  const float* w_g, const float* w_l, const void* weight, void* out,
                                  int B, int H, int L, int Dv, int C, long long g_row_stride, float eps, int silu_out,
                                  int io_dtype, void* stream);
/* The same, leaving the blended rows as well: blended [B*L, H*Dv], what a backward reads. */
int vig_locality_blend_linear_kept_fwd(const void* o, const void* local, const void* g_lin, const float* w_g,
                                       const float* w_l, const void* weight, void* blended, void* out, int B, int H, int L, int Dv,
                                       int C, long long g_row_stride, float eps, int silu_out, int io_dtype, void* stream);

/*
 * First convolution of the v2 patch embedding, without its bias (vig_layernorm_fwd's pre_bias takes that):
 *   x [B, Cin, H, W] (bf16, the layout images arrive in)  ->  y [B, OH, OW, Cout] (bf16, channels-last rows),
 *   OH = (H + 2*padding - KH) / stride + 1, OW likewise.
 *   w_packed [Cout, Cin*KH, 16] bf16: the kernel rows of the [Cout, Cin, KH, KW] weight, each padded with zeros to
 *   16 columns.
 * Built for the reference's stem: stride 8, padding 1, KW <= 16 (9 where W > 248), Cin*KH = 27 (3 channels x 9 rows),
 * W % 8 == 0, Cout a multiple of 32 from 64 to 256, or 384; anything else returns VIG_ENOTSUP (use a library convolution).
 *
 * Replaces: the first nn.Conv2d of V2PatchEmbed (classification/models/vig.py:651) and the layout change a
 * channels-last convolution library needs in front of it.
 */
int vig_patch_conv_fwd(const void* x, const void* w_packed, void* y, int B, int Cin, int H, int W, int KH, int KW,
                       int stride, int padding, int Cout, int io_dtype, void* stream);

/*
 * vig_patch_conv_fwd and vig_layernorm_fwd on its rows (pre_bias [Cout] or NULL, silu, no post_add) in one kernel, bit for bit; the
 * convolution's own result is not stored.  Built for the same shapes up to Cout = 256, bf16.
 *
 * Replaces: the first nn.Conv2d, LayerNorm2d and SiLU of V2PatchEmbed (classification/models/vig.py:651-653).
 */
int vig_patch_conv_norm_fwd(const void* x, const void* w_packed, const float* norm_weight, const float* norm_bias, const float* pre_bias, void* y,
                            int B, int Cin, int H, int W, int KH, int KW, int stride, int padding, int Cout, float eps, int silu, void* stream);

/*
 * y [rows, N] = x [rows, K] . weight [N, K]^T (+ bias [N]), bf16, fp32 accumulation, the bias added before the one rounding;
 * rows of x and y x_row_stride / y_row_stride elements apart.  N % 8 == 0, K % 32 == 0.
 * vig_linear_preferred: whether this entry point is the better choice for a size (short of large products, where the BLAS
 * library's kernels win).
 *
 * Replaces: the nn.Linear layers of the block and the classifier (classification/models/vig.py:286-312,492-497,826).
 */
int vig_linear_preferred(long long rows, int N, int K);
int vig_linear_fwd(const void* x, long long x_row_stride, const void* weight, const void* bias, void* y, long long y_row_stride,
                   long long rows, int N, int K, void* stream);

/*
 * The middle of a block in one kernel, bf16, few rows of C = 192 channels (vig_locality_blend_swiglu_preferred), else VIG_ENOTSUP: what
 * vig_locality_blend_linear_fwd (out_weight [C, C]; its result is not stored) and vig_norm_swiglu_fwd (weight [2*I, C], I % 64 == 0) give one
 * after the other, bit for bit: sum [B*L, C], y [B*L, I].  No output may be an input.
 *
 * Replaces: classification/models/vig.py:444-463,606-608 and :492-497 (head norms, sigmoid blend, out_act, o_proj, mlp_norm, SwiGLU layer).
 */
int vig_locality_blend_swiglu_preferred(long long rows, int C, int I);
int vig_locality_blend_swiglu_fwd(const void* o, const void* local, const void* g_lin, const float* w_g, const float* w_l,
                                  const void* out_weight, const void* residual, const float* norm_weight, const void* weight, void* sum,
                                  void* y, int B, int H, int L, int Dv, int C, int I, long long g_row_stride, float eps, int silu_out,
                                  float norm_eps, void* stream);

/*
 * Residual add, RMS norm and the depthwise 3x3 convolution behind it in one kernel, bf16:
 *   sum [B, h*w, C] = x + residual (rounded; residual NULL: x),  y = conv3x3(rms(sum) * norm_weight) (+ bias, SiLU): what
 * vig_rmsnorm_fwd (round_sum 1) and vig_dwconv3x3_fwd give one after the other.  weight [C, 9], bias [C] or NULL; sum may be NULL.
 * C = 192 or 384 and sizes where it is quicker than those (vig_norm_dwconv3x3_preferred), else VIG_ENOTSUP.  No output may be an input.
 *
 * Replaces: classification/models/vig.py:291-294,364-366,598-606 (attn_norm, local convolution).
 */
int vig_norm_dwconv3x3_preferred(int B, int h, int w, int C);
int vig_norm_dwconv3x3_fwd(const void* x, const void* residual, const float* norm_weight, const float* weight, const float* bias,
                           void* sum, void* y, int B, int h, int w, int C, float eps, int silu, void* stream);

/*
 * The same with a row product behind the convolution: sum as above (may be NULL), conv [B, h*w, C] the convolution's result,
 * y [B, h*w, N] = conv . weight [N, C]^T (+ bias [N] bf16, or NULL), as vig_norm_dwconv3x3_fwd and vig_linear_fwd give one after the other.
 * C = 192 or 384, N % 128 == 0 and few images (vig_norm_dwconv3x3_linear_preferred), else VIG_ENOTSUP.  No output may be an input.
 *
 * Replaces: classification/models/vig.py:291-294,364-369,598-606 (attn_norm, local convolution, projections).
 */
int vig_norm_dwconv3x3_linear_preferred(int B, int h, int w, int C, int N);
int vig_norm_dwconv3x3_linear_fwd(const void* x, const void* residual, const float* norm_weight, const float* conv_weight,
                                  const float* conv_bias, const void* weight, const void* bias, void* sum, void* conv, void* y, int B,
                                  int h, int w, int C, int N, float eps, int silu, void* stream);

/*
 * Residual add, RMS norm and the SwiGLU layer behind it in one kernel, bf16, packed rows:
 *   sum [rows, K] = x + residual (stored rounded; the norm is of the sum in fp32),  y [rows, I] = SwiGLU of rms(sum) * norm_weight . weight^T,
 * weight [2*I, K] with the gate rows first: what vig_rmsnorm_fwd (round_sum 0) and vig_linear_swiglu_fwd give one after the other.
 * K = 192 or 384, I % 32 == 0 and few rows (vig_norm_swiglu_preferred), else VIG_ENOTSUP.  No output may be an input.
 *
 * Replaces: classification/models/vig.py:486-496,604-606 (prenorm add, mlp_norm, gate_proj, up_proj and their product).
 */
int vig_norm_swiglu_preferred(long long rows, int K, int I);
int vig_norm_swiglu_fwd(const void* x, const void* residual, const float* norm_weight, const void* weight, void* sum, void* y,
                        long long rows, int K, int I, float eps, void* stream);

/*
 * A linear layer without bias, the residual add and the RMS norm behind it in one kernel, bf16, packed rows:
 *   sum [rows, N] = residual + x [rows, K] . weight [N, K]^T (the product rounded to bf16, then the sum),  y = rms(sum) * norm_weight
 * N = 192, K % 64 == 0, else VIG_ENOTSUP.  sum and y are not the inputs.  _preferred: whether it is the better
 * choice next to a product and vig_rmsnorm_fwd with round_sum, which give the same values.
 *
 * Replaces: down_proj, the block's closing add and the next block's attn_norm (classification/models/vig.py:497,598,606).
 */
int vig_linear_norm_preferred(long long rows, int N, int K);
int vig_linear_norm_fwd(const void* x, const void* weight, const void* residual, const float* norm_weight, void* y, void* sum,
                        long long rows, int N, int K, float eps, void* stream);

/*
 * 3x3 convolution, stride 2, padding 1, no bias, bf16 channels-last: x [B, H, W, Cin], weight [Cout, 3, 3, Cin] ->
 * y [B, (H+1)/2, (W+1)/2, Cout].  Cin % 32 == 0, Cout % 8 == 0.
 *
 * Replaces: the second convolution of the v2 patch embedding (classification/models/vig.py:655).
 */
int vig_conv3x3s2_fwd(const void* x, const void* weight, void* y, int B, int H, int W, int Cin, int Cout, void* stream);

/*
 * fp32 product on the matrix cores, operands in three bf16 pieces (fp32 precision):
 *   out[m, n] = sum_k A(m, k) B(n, k) + bias[n] + add[m, n]     (bias, add: NULL for none)
 * A(m, k) = a[m*lda + k], or a[k*lda + m] with a_across; B(n, k) = b[n*ldb + k], or b[k*ldb + n] with b_across (not a_across
 * alone).  With a_across also a_sums[m] = sum_k A(m, k) unless NULL.  A layer, its input gradient and its weight gradient are
 * (x, w), (dy, w across) and (dy across, x across).  a, b and the workspace start on 16-byte boundaries; where the
 * contraction is contiguous, K is a multiple of 8 and the row distance one of 4.  Operands beyond 1 GiB and other
 * shapes: VIG_ENOTSUP.  The workspace (vig_matmul_f32_workspace bytes) holds partial tiles of long contractions over
 * few tiles; they are added in a fixed order.
 *
 * Replaces: the fp32 linear layers and their gradients of classification/models/vig.py:295-330,486-497 (cuBLAS).
 */
size_t vig_matmul_f32_workspace(long long M, int N, long long K);
int vig_matmul_f32(const float* a, long long lda, int a_across, const float* b, long long ldb, int b_across,
                   const float* bias, const float* add, long long ldadd, float* out, long long ldo, float* a_sums,
                   long long M, int N, long long K, void* workspace, size_t workspace_bytes, void* stream);

/*
 * The closing norm and the mean over tokens in one pass, bf16: out [B, C] = mean over l of the RMS-normalised
 * (x + residual)[b, l, :], the sum and the normalised value rounded to bf16 as vig_rmsnorm_fwd with round_sum stores them, the mean in fp32.
 * C % 8 == 0, C <= 1024.
 *
 * Replaces: classification/models/vig.py:896-905 (norm_f and the average pool).
 */
size_t vig_rmsnorm_pool_workspace(int B, int L, int C);
int vig_rmsnorm_pool_fwd(const void* x, const void* residual, const float* weight, void* out, void* workspace,
                         size_t workspace_bytes, int B, int L, int C, float eps, void* stream);

/*
 * Weight and bias gradients of a linear layer over bf16 rows (what autograd derives for the nn.Linear layers of the block):
 *   dweight [N, K] (fp32) = sum over rows of dy[row, n] * x[row, k];  dbias [N] (fp32) = sum over rows of dy[row, n],
 * fp32 accumulation in a fixed order.  dy rows are dy_row_stride elements apart, x rows x_row_stride (multiples of 8, 16-byte
 * aligned bases: either may be a column block of a wider tensor); N % 8 == 0, K % 8 == 0; dbias NULL: not wanted.
 * `workspace` holds vig_linear_bwd_weight_workspace(rows, N, K) bytes of partial sums.
 */
size_t vig_linear_bwd_weight_workspace(long long rows, int N, int K);
int vig_linear_bwd_weight(const void* dy, long long dy_row_stride, const void* x, long long x_row_stride, float* dweight,
                          float* dbias, void* workspace, size_t workspace_bytes, long long rows, int N, int K, void* stream);

/*
 * The same of up to four layers over the same number of rows, in one launch and one that adds the partial sums, or, where that is quicker (many
 * tiles and rows), in a pair of launches a layer: arrays of `count` entries, each as above; dbias may be NULL, and so may its entries.
 */
size_t vig_linear_bwd_weight_many_workspace(long long rows, const int* N, const int* K, int count);
int vig_linear_bwd_weight_many(const void* const* dy, const long long* dy_row_stride, const void* const* x,
                               const long long* x_row_stride, float* const* dweight, float* const* dbias, void* workspace,
                               size_t workspace_bytes, long long rows, const int* N, const int* K, int count, void* stream);

/*
 * The layer norms of the patch embedding for training: y [rows, C] = layernorm(x + pre_bias) * weight + bias, through SiLU if silu, x [rows, C]
 * and y bf16 or fp32 (fp32 x: fp32 y), all between them fp32; pre_bias [C] or NULL.  C % 8 == 0, C <= 1024, at most VIG_STEM_NORM_ROWS rows.
 * _bwd: dx [rows, C] in x's type (NULL: not wanted) and dparams [3, C]: the gradients of weight, bias and pre_bias; dy in y's type.
 *
 * Replaces: LayerNorm2d and nn.SiLU of V2PatchEmbed (classification/models/vig.py:619-624,651-656), the convolutions' bias adds, and what
 * autograd derives for them.
 */
#define VIG_STEM_NORM_ROWS (0x7fffffffLL - 16384)
int vig_stem_norm_fwd(const void* x, const float* pre_bias, const float* weight, const float* bias, void* y, long long rows, int C, float eps,
                      int silu, int x_dtype, int y_dtype, void* stream);
size_t vig_stem_norm_bwd_workspace(long long rows, int C);
int vig_stem_norm_bwd(const void* x, const float* pre_bias, const float* weight, const float* bias, const void* dy, void* dx, float* dparams,
                      void* workspace, size_t workspace_bytes, long long rows, int C, float eps, int silu, int x_dtype, int y_dtype,
                      void* stream);

/*
 * Several backward kernels leave partial rows in their workspace that a sum over the rows finishes, a launch each.  The _later forms put
 * that sum off (`later` NULL: they do not): they enter it in `later` (zero before the first one), the gradients concerned (dw_db, dw, dweight, dbias) are filled by
 * vig_sum_jobs_run, one launch for all, on the same stream, and until then every workspace and every output has to stay.  Results bit
 * for bit as without.  A full list is refused with VIG_EINVAL (a form enters up to one, one, one and 2 * count of them).
 * vig_sum_jobs_run empties the list.
 */
#define VIG_SUM_JOBS 12
typedef struct {
  const float* part; /* [rows, cols] */
  float* out;        /* [cols] */
  long long cols;
  int rows, fours;   /* fours: few rows, columns taken four at a time */
} vig_sum_job;
typedef struct {
  vig_sum_job job[VIG_SUM_JOBS];
  int count;
} vig_sum_jobs;
int vig_dwconv3x3_bwd_later(const void* x, const void* dy, const void* pre, const float* weight, void* dx, float* dw_db,
                      void* workspace, size_t workspace_bytes, int B, int h, int w, int C, int io_dtype, vig_sum_jobs* later, void* stream);
int vig_locality_blend_bwd_strided_later(const void* o, const void* local, const void* g_lin, const float* w_g, const float* w_l,
                                   const void* dy, void* d_o, void* d_local, void* d_glin, float* dw, void* workspace,
                                   size_t workspace_bytes, int B, int H, int L, int Dv, long long g_row_stride,
                                   long long d_glin_row_stride, float eps, int silu_out, int io_dtype, vig_sum_jobs* later, void* stream);
int vig_rmsnorm_mixed_bwd_later(const void* sum, const float* weight, const void* dy, const void* d_sum, void* ds, void* dx,
                          float* dweight, void* workspace, size_t workspace_bytes, long long rows, int C, float eps,
                          int sum_dtype, int y_dtype, vig_sum_jobs* later, void* stream);
int vig_linear_bwd_weight_many_later(const void* const* dy, const long long* dy_row_stride, const void* const* x,
                               const long long* x_row_stride, float* const* dweight, float* const* dbias, void* workspace,
                               size_t workspace_bytes, long long rows, const int* N, const int* K, int count, vig_sum_jobs* later, void* stream);
int vig_sum_jobs_run(vig_sum_jobs* jobs, void* stream);

#ifdef __cplusplus
}
#endif
#endif /* VIG_GLA_H_ */
