/*
 * fields_amd.h — C ABI of the MI355X (gfx950) Field-block hot path.
 *
 * The Field recurrence of Fields LM, per (batch b, time t, channel c), C = d_model / 2:
 *
 *   inj   = tanh(raw[b,t,c]) + i*tanh(raw[b,t,C+c])
 *   v     = 0.9 * sigmoid(raw[b,t,2C+c])              (independent vacancy)
 *   lam   = tr[c] + i*ti[c]
 *   disp  = v * lam * s[t-1]                          (displaced readout)
 *   s[t]  = (1 - v) * lam * s[t-1] + gamma[c]*v*inj   (causal write), s[-1] = state_in or 0
 *   read[b,t,:] = [Re s | Im s | Re disp | Im disp]   (4C floats)
 *
 * All pointers are device pointers unless stated. Every entry point is stream-ordered on
 * `stream`, performs no allocation and no host synchronisation (so a caller may capture it
 * in a hipGraph), keeps no global mutable state and is reentrant: calls on different
 * streams must use different workspaces. The one exception is fl_scan_forward_static, whose
 * look-back state is a per-GPU array inside the library (see its comment).
 *
 * Complex state vectors are stored planar, [B, 2C] floats: the first C entries of a row
 * are the real parts and the next C the imaginary parts (the layout of read[:, t, :2C]).
 *
 * Return value: FL_OK or one of the FL_ERR_* codes below. FL_ERR_HIP_BASE + e means that
 * HIP reported error e (a hipError_t) on launch.
 */
#ifndef FIELDS_AMD_H_
#define FIELDS_AMD_H_

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* element types of raw / read buffers */
#define FL_DTYPE_F32 0
#define FL_DTYPE_BF16 1

/* algorithm selector for fl_scan_forward_ex (low 8 bits); bits 8.. select a tiling variant of
 * FL_ALGO_LOOKBACK for tuning: 0 = default (LDS-staged 16-byte loads and stores where raw is bf16
 * with 16-byte aligned rows, read is fp32 and C is a multiple of 64; register loads and stores
 * otherwise), 1..5 = other tilings, 6 = LDS-staged where possible, 7 = default tiling with
 * register loads and stores on every input */
#define FL_ALGO_AUTO 0
#define FL_ALGO_CHUNKED3 1 /* chunk summary -> chunk carry -> chunk materialise (three launches) */
#define FL_ALGO_LOOKBACK 2 /* single launch, decoupled look-back across chunks (default) */

#define FL_OK 0
#define FL_ERR_INVALID_ARGUMENT 1 /* shape / stride / pointer check failed (Python: ValueError) */
#define FL_ERR_DTYPE 2            /* unsupported raw or read dtype (Python: TypeError) */
#define FL_ERR_WORKSPACE 3        /* workspace NULL or smaller than fl_scan_workspace_bytes */
#define FL_ERR_CAPTURE 4          /* fl_scan_forward_static: first call on a device under capture */
#define FL_ERR_HIP_BASE 1000      /* FL_ERR_HIP_BASE + hipError_t */

/*
 * Chunked forward scan over a whole sequence batch.
 *
 * Replaces `fused_field_read(raw, transition_r, transition_i, gamma, block_c, chunk_t)`
 * (src/fields_official/reference/field_only_v4_chunked_triton_wiki100.py:1108-1123) and the
 * three Triton launches of `_ChunkedFieldReadFunction.forward` (same file, 913-1018:
 * `_field_chunk_summary_kernel` 443-516, `_field_chunk_carry_kernel` 519-550,
 * `_field_chunk_materialize_kernel` 553-622). The reference always starts from state 0 and
 * takes fp32 raw only; state_in/state_out and bf16 raw are extensions (state_in = NULL and
 * fp32 raw reproduce the reference call).
 *
 *   raw        [B, T, 3C] of raw_dtype; element (b,t,j) at raw + b*raw_stride_b + t*raw_stride_t + j
 *              (strides in elements, channel stride 1, raw_stride_t >= 3C)
 *   tr, ti, gamma  [C] fp32
 *   state_in   [B, 2C] fp32 planar, or NULL for the zero state
 *   state_out  [B, 2C] fp32 planar, or NULL; receives s[T-1]
 *   read       [B, T, 4C] contiguous, read_dtype: FL_DTYPE_F32, or FL_DTYPE_BF16 (values rounded
 *              to nearest even; 7,168 instead of 11,264 bytes per token at C = 512 with bf16 raw)
 *   workspace  device scratch of at least fl_scan_workspace_bytes(B, T, C) bytes, 256-byte
 *              aligned, ZERO-FILLED before its first use and then reused as is: its first 2 KiB
 *              hold launch counters that every call leaves ready for the next one. Calls on one
 *              workspace must be stream-ordered (one workspace per stream). Every launch advances
 *              an epoch kept there; the launch at each 2^30-launch wrap of its tag bits zero-fills
 *              the rest of the workspace itself, so it is never zero-filled again by the caller.
 *   workspace_bytes  the size of that allocation. It must not exceed the allocation: the wrap
 *              launch zero-fills workspace_bytes after the header (every word an earlier call at
 *              any shape may have left), so a larger value writes past the buffer.
 *
 * Workspace header (first 2 KiB; little-endian words at these byte offsets):
 *   128  u32  error word: bit 0 a bounded wait gave up, bit 1 a ticket beyond the launch's tiles
 *             (set by the kernels, never cleared by them)
 *   384  u32  spin limit: polls before a wait gives up (0 = 2^20); written by the caller
 *   392  u64  address of a host-visible (pinned, device-mapped) u32 that the kernels set non-zero
 *             whenever they set the error word, so a caller can see a failure without reading
 *             device memory; 0 = none; written by the caller
 * A wait that gives up makes what depends on it NaN (the tile's outputs and every later tile of
 * its chain, a row's RMSNorm scale, the backward's gradients), so an output computed without a
 * value it needed cannot pass for a valid one. The same header leads the backward's workspace.
 */
int fl_scan_forward(const void* raw, int raw_dtype, int64_t B, int64_t T, int64_t C,
                    int64_t raw_stride_b, int64_t raw_stride_t, const float* tr, const float* ti,
                    const float* gamma, const float* state_in, float* state_out, void* read,
                    int read_dtype, void* workspace, size_t workspace_bytes, void* stream);

/*
 * fl_scan_forward without a workspace argument, for callers that cannot allocate device memory
 * (code under HIP graph capture, tight serving loops, harnesses that forbid hipMalloc). It has no
 * counterpart in the reference. It calls no hipMalloc, hipFree or allocating library routine: the
 * look-back state lives in a file-scope device array of FL_STATIC_SCRATCH_BYTES in this library,
 * one copy per GPU, held until the process ends.
 *
 *   * Shapes: B * ceil(C / 64) * ceil(T / 128) <= FL_STATIC_MAX_TILES (config 2 needs 1,024,
 *     B = 1 with T = 65,536 and C = 512 needs 4,096); larger shapes return FL_ERR_WORKSPACE.
 *   * The first call on each device zero-fills that device's array on `stream`: it must not be
 *     made under stream capture (FL_ERR_CAPTURE). Later calls may be captured.
 *   * Every call on one GPU shares that GPU's array: calls that overlap on one GPU (two streams,
 *     two threads) race and must be serialised by the caller.
 *   * A bounded wait that gives up leaves NaN in the outputs that depend on it (there is no error
 *     word the caller can read).
 * Arguments and results as fl_scan_forward (FL_ALGO_AUTO); results are bit-identical to it.
 */
#define FL_STATIC_MAX_TILES 12288
#define FL_STATIC_SCRATCH_BYTES 31508480 /* 2 KiB header + 12,288 status words + tagged words */
int fl_scan_forward_static(const void* raw, int raw_dtype, int64_t B, int64_t T, int64_t C,
                           int64_t raw_stride_b, int64_t raw_stride_t, const float* tr,
                           const float* ti, const float* gamma, const float* state_in,
                           float* state_out, void* read, int read_dtype, void* stream);

/* As fl_scan_forward with an explicit algorithm (FL_ALGO_*). */
int fl_scan_forward_ex(const void* raw, int raw_dtype, int64_t B, int64_t T, int64_t C,
                       int64_t raw_stride_b, int64_t raw_stride_t, const float* tr,
                       const float* ti, const float* gamma, const float* state_in,
                       float* state_out, void* read, int read_dtype, void* workspace,
                       size_t workspace_bytes, int algo, void* stream);

/*
 * Forward scan with the mixer's read_norm RMSNorm fused into the epilogue: writes
 *
 *   out[b,t,j] = (read[b,t,j] * rsqrt(sum_i read[b,t,i]^2 / (4C) + eps)) * norm_weight[j]
 *
 * for the read that fl_scan_forward computes (in fp32), without writing read itself. Replaces
 * `self.read_norm(fused_field_read(...))` in `IndependentVacancyField.forward`
 * (field_only_v4_chunked_triton_wiki100.py:1176-1193, RMSNorm 300-309); the out_proj GEMM
 * then reads `out` directly. out_dtype FL_DTYPE_BF16 gives the fp32 value rounded to nearest
 * even, which is what the reference's out_proj sees under bf16 autocast.
 *
 * Arguments as fl_scan_forward, plus norm_weight [4C] fp32 and eps (>= 0); the same workspace.
 * Single-launch path only; C <= 4096.
 */
int fl_scan_norm_forward(const void* raw, int raw_dtype, int64_t B, int64_t T, int64_t C,
                         int64_t raw_stride_b, int64_t raw_stride_t, const float* tr,
                         const float* ti, const float* gamma, const float* state_in,
                         float* state_out, const float* norm_weight, float eps, void* out,
                         int out_dtype, void* workspace, size_t workspace_bytes, void* stream);

/*
 * Backward of fl_scan_forward: the gradients of a loss L given dL/dread (and dL/dstate_out).
 *
 * Replaces `_ChunkedFieldReadFunction.backward`
 * (field_only_v4_chunked_triton_wiki100.py:1020-1105; Triton kernels 625-910: chunk summary,
 * chunk carry, chunk materialise, then a torch sum of the parameter partials). Two launches on
 * `stream`: the reverse scan (decoupled look-back over chunks taken in reverse time order), whose
 * tiles write per-tile parameter-gradient partials into the workspace, then a reduction that adds
 * them up in a fixed order (bit-reproducible).
 *
 *   raw, strides, tr, ti, gamma, state_in   as given to the forward call
 *   read            [B, T, 4C] fp32, the forward output (the state planes at every 8th row
 *                   are read: the state before each 8-step group, from which s_{t-1} of the
 *                   group's steps is recomputed; the reference reads it back at every step)
 *   grad_read       [B, T, 4C] fp32 contiguous
 *   grad_state_out  [B, 2C] fp32 planar, or NULL (state_out unused)
 *   grad_raw        [B, T, 3C] contiguous, grad_raw_dtype F32 or BF16 (overwritten)
 *   grad_tr, grad_ti, grad_gamma  [C] fp32 (overwritten)
 *   grad_state_in   [B, 2C] fp32 planar, or NULL
 *   workspace       >= fl_scan_backward_workspace_bytes(B, T, C), 256-byte aligned, zero-filled
 *                   before first use, then reused (one per stream), as for fl_scan_forward;
 *                   workspace_bytes must not exceed the allocation (the same wrap clear)
 * A block that finds the ticket counter out of range (error bit 1) computes nothing, so the
 * parameter gradients of that call are NaN (its reduction sums every tile's partials).
 */
int fl_scan_backward(const void* raw, int raw_dtype, int64_t B, int64_t T, int64_t C,
                     int64_t raw_stride_b, int64_t raw_stride_t, const float* tr, const float* ti,
                     const float* gamma, const float* state_in, const float* read,
                     const float* grad_read, const float* grad_state_out, void* grad_raw,
                     int grad_raw_dtype, float* grad_tr, float* grad_ti, float* grad_gamma,
                     float* grad_state_in, void* workspace, size_t workspace_bytes, void* stream);

/* Workspace size in bytes for fl_scan_backward (host function, no device call). Replaces the
 * ten [B, n_chunks, C] torch.empty buffers of field_only_v4_chunked_triton_wiki100.py:1027-1037. */
size_t fl_scan_backward_workspace_bytes(int64_t B, int64_t T, int64_t C);

/*
 * Workspace size in bytes for fl_scan_forward at this shape (host function, no device call).
 * Replaces the six [B, n_chunks, C] fp32 torch.empty buffers of
 * field_only_v4_chunked_triton_wiki100.py:941-952.
 */
size_t fl_scan_workspace_bytes(int64_t B, int64_t T, int64_t C);

/*
 * Single-token recurrent step for the decode loop: reads state (s[t-1]) and raw_t, writes
 * read_t and overwrites state with s[t], in one pass.
 *
 * The reference has no incremental step; this is the per-t body of
 * `_field_chunk_materialize_kernel` (field_only_v4_chunked_triton_wiki100.py:583-621) applied
 * to one token with the state carried between calls. Equal to row t of fl_scan_forward.
 *
 *   raw_t  [B, 3C] of raw_dtype, row stride raw_stride_b elements (>= 3C), channel stride 1
 *   state  [B, 2C] fp32 planar, updated in place
 *   read_t [B, 4C] contiguous, read_dtype FL_DTYPE_F32
 */
int fl_decode_step(const void* raw_t, int raw_dtype, int64_t B, int64_t C, int64_t raw_stride_b,
                   const float* tr, const float* ti, const float* gamma, float* state,
                   void* read_t, int read_dtype, void* stream);

/*
 * fl_decode_step with the read_norm RMSNorm fused in: state advances as in fl_decode_step and
 * out_t [B, 4C] (out_dtype F32 or BF16, contiguous) receives the normalised read_t, as
 * fl_scan_norm_forward defines it. The decode-loop counterpart of fl_scan_norm_forward
 * (field_only_v4_chunked_triton_wiki100.py:1176-1193 and 300-309 for one token).
 */
int fl_decode_norm_step(const void* raw_t, int raw_dtype, int64_t B, int64_t C,
                        int64_t raw_stride_b, const float* tr, const float* ti,
                        const float* gamma, float* state, const float* norm_weight, float eps,
                        void* out_t, int out_dtype, void* stream);

/*
 * Boundary scan of the softpatch mixer: s[b,t,r] = a[b,t] * s[b,t-1,r] + drive[b,t,r] with
 * s[b,-1,:] = state_in (or 0), written to out [B, T, R]; state_out [B, R] receives s[b,T-1,:].
 *
 * Replaces `hierarchical_scan(a, drive, block=32)` in `BoundaryStateMixer.forward`
 * (src/fields_official/reference/official_source/field_hybrid_attentionfree_qualification_v3.py:458-460
 * and field_hybrid_speed_optimization_v6.py:333-335), where a = 1 - boundary is one value per
 * token broadcast over the rank R. All buffers fp32 and contiguous; state_in / state_out may be
 * NULL. No workspace.
 */
int fl_boundary_scan(const float* a, const float* drive, int64_t B, int64_t T, int64_t R,
                     const float* state_in, float* state_out, float* out, void* stream);

/*
 * The softpatch mixer around that scan (no gradients), bf16 in and out, fp32 maths:
 * fl_softpatch_norm: h = RMSNorm(x) weight over rows of dim (a multiple of 8, at most 4,096) and
 *   score[row] = h . w_score + bias[0];
 * fl_softpatch_scan: with boundary = clamp(sigmoid(score + 1.5 prior), 0.01, 0.99) per token,
 *   s_t = (1 - boundary_t) s_{t-1} + boundary_t z_t from s_{-1} = 0; out [B, T, 2R] = [z | s],
 *   state_out [B, R] = s_{T-1} in fp32. z [B, T, R], score and (fp32) prior [B, T], contiguous;
 *   workspace: fl_softpatch_workspace_bytes, no initial contents needed.
 */
int fl_softpatch_norm(const void* x, int64_t rows, int64_t dim, const void* weight, float eps, const void* w_score,
                      const void* bias, void* h, void* score, void* stream);
size_t fl_softpatch_workspace_bytes(int64_t B, int64_t T, int64_t R);
int fl_softpatch_scan(const void* z, const void* score, const float* prior, int64_t B, int64_t T, int64_t R,
                      float* state_out, void* out, void* workspace, size_t workspace_bytes, void* stream);

/*
 * Field block elementwise tail for inference, one launch per row block:
 *   x_new  = x + out * sigmoid(gate_pre)            (IndependentVacancyField.forward return,
 *                                                    field_only_v4_chunked_triton_wiki100.py:1193-1195)
 *   normed = RMSNorm(x_new) * norm_weight           (FieldBlock.ff_norm, same file 1219-1221, 300-309)
 * out / gate_pre are the out_proj / gate_proj GEMM outputs (g_dtype), x / x_new / normed the
 * residual stream (x_dtype); all [rows, dim] contiguous except gate_pre, whose rows lie
 * gate_stride >= dim elements apart (a column slice of a GEMM output that also holds other
 * columns, e.g. write_proj and gate_proj computed in one GEMM). Every intermediate is rounded where
 * the stock ops round it (bf16 ops compute in fp32 and round their result).
 */
int fl_gate_residual_norm(const void* x, int x_dtype, const void* out, const void* gate_pre,
                          int g_dtype, int64_t rows, int64_t dim, int64_t gate_stride,
                          const float* norm_weight, float eps, void* x_new, void* normed,
                          void* stream);

/* fl_gate_residual_norm with norm_weight of either element type (w_dtype): the bf16 values are
 * widened exactly, as the stock RMSNorm's weight.float() does. */
int fl_gate_residual_norm_w(const void* x, int x_dtype, const void* out, const void* gate_pre,
                            int g_dtype, int64_t rows, int64_t dim, int64_t gate_stride,
                            const void* norm_weight, int w_dtype, float eps, void* x_new,
                            void* normed, void* stream);

/*
 * One token of a whole Field block for up to 128 rows (FieldBlock.forward of one position,
 * field_only_v4_chunked_triton_wiki100.py:1167-1221), bf16 weights and activations, fp32 sums:
 *   [raw | g] = x [write_w | gate_w]^T + bias,  normed = fl_decode_norm_step(raw, state),
 *   x1 = x + (normed out_w^T + out_b) * sigmoid(g),  h = RMSNorm(x1) ff_norm_w,
 *   out = x1 + (silu(h gate^T) * (h up^T)) down_w^T  with up_w = [gate; up] [2 hidden, dim].
 * x, out [rows, dim] contiguous; weights as their layers hold them ([out features, in features]),
 * 16-byte aligned; dim and hidden multiples of 8; biases may be NULL; tr, ti, gamma, read_norm_w
 * fp32, ff_norm_w of ff_norm_dtype; state [rows, dim] fp32 advances in place. Rounded to bf16 where the
 * separate ops round, except that the RMSNorm's row scale is applied to the fp32 sums. The weights are
 * read once per row tile of 16 (32 from rows x dim of 65,536 on): wide blocks with many rows are faster
 * through products that read them once.
 */
size_t fl_block_step_workspace_bytes(int64_t rows, int64_t dim, int64_t hidden);
int fl_block_step(const void* x, int64_t rows, int64_t dim, int64_t hidden, const void* write_w, const void* write_b,
                  const void* gate_w, const void* gate_b, const float* tr, const float* ti, const float* gamma,
                  float* state, const float* read_norm_w, float read_eps, const void* out_w, const void* out_b,
                  const void* ff_norm_w, int ff_norm_dtype, float ff_eps, const void* up_w, const void* down_w,
                  void* out, void* workspace, size_t workspace_bytes, void* stream);

/*
 * Transition parameters of the Field mixer (field_only_v4_chunked_triton_wiki100.py:1169-1173),
 * fp32 [C] each: radius = clamp(sigmoid(radius_logit), 0.5, 0.99995), tr = radius cos(theta),
 * ti = radius sin(theta), gamma = sqrt(max(1 - radius^2, 1e-4)). With n_weight > 0, weight32
 * [n_weight] also receives the bf16 vector weight16 as fp32 (the read_norm weight, which the scan
 * takes in fp32); weight16 / weight32 may be NULL when n_weight is 0.
 */
int fl_field_params(const float* radius_logit, const float* theta, int64_t C, const void* weight16,
                    int64_t n_weight, float* tr, float* ti, float* gamma, float* weight32,
                    void* stream);

/*
 * SwiGLU activation of the Field block FFN (PackedSwiGLU.forward, same file 312-325):
 * out[r, j] = silu(gate_up[r, j]) * gate_up[r, hidden + j], [rows, 2*hidden] -> [rows, hidden].
 */
int fl_swiglu(const void* gate_up, int dtype, int64_t rows, int64_t hidden, void* out,
              void* stream);

/*
 * The Mamba-2 mixer between its projections (no gradients), geometry headdim 64, d_state 128,
 * d_conv 4, one group (src/fields_official/reference/official_source/
 * field_fusion_wiki100_mamba2_v25.py:73-91, 455-468): with inner = 64 heads and a row of the input
 * projection zxbcdt = [z inner | x inner | B 128 | C 128 | dt heads],
 *   [x | B | C] = silu(causal depthwise conv),  dt = softplus(dt + dt_bias),  A = -exp(A_log),
 *   h_t = exp(dt_t A) h_{t-1} + dt_t x_t B_t^T,  y_t = h_t C_t + D x_t                 (per head)
 *   out = RMSNorm(y silu(z)) norm_w       over the inner width, fp32 maths, written as out_dtype.
 * zxbcdt [B, L, *] of dtype, rows stride_t and sequences stride_b elements apart (both even),
 * conv_w [inner + 256, 4] and conv_b of conv_dtype, A_log / dt_bias / D [heads] fp32, norm_w [inner]
 * of norm_dtype, out [B, L, inner] contiguous; ssm_out [B, heads, 64, 128] fp32 receives h_{L-1}
 * (NULL: not wanted). workspace: fl_mamba_workspace_bytes(B, L, heads) bytes, 16-byte aligned, no
 * initial contents needed.
 *
 * fl_mamba_step advances one token: zxbcdt [B, *], conv_state [B, inner + 256, 4] (the last four
 * inputs, newest last) and ssm updated in place; workspace as for L = 1.
 */
size_t fl_mamba_workspace_bytes(int64_t B, int64_t L, int64_t heads);
int fl_mamba_prefill(const void* zxbcdt, int dtype, int64_t B, int64_t L, int64_t heads, int64_t stride_b,
                     int64_t stride_t, const void* conv_w, const void* conv_b, int conv_dtype,
                     const float* A_log, const float* dt_bias, const float* D, const void* norm_w,
                     int norm_dtype, float eps, void* out, int out_dtype, float* ssm_out,
                     void* workspace, size_t workspace_bytes, void* stream);
int fl_mamba_step(const void* zxbcdt, int dtype, int64_t B, int64_t heads, int64_t stride_b,
                  const void* conv_w, const void* conv_b, int conv_dtype, const float* A_log,
                  const float* dt_bias, const float* D, const void* norm_w, int norm_dtype, float eps,
                  float* conv_state, float* ssm, void* out, int out_dtype, void* workspace,
                  size_t workspace_bytes, void* stream);

/*
 * Attention of the refresh blocks over a whole sequence (no gradients), bf16, head dimension 64
 * (src/fields_official/reference/official_source/field_fusion_system_smoke_v21.py:131-253):
 *   out[b,t,h,:] = local + sigmoid(mix_logit) * global,
 * local: RoPE'd causal attention inside t's window of `window` tokens; global: attention to a null
 * slot (score 0, value 0) and the landmarks of the chunks completed before t's.
 * q [B, T, q_heads * 64] with row / sequence strides (multiples of 8), not yet rotated; kv
 * [B, T, 2 * kv_heads * 64] contiguous, keys then values; landmark_kv [B, n_landmarks, 2 * kv_heads * 64]
 * likewise (row j's key sits at position (j + 1) * landmark_chunk - 1); cos / sin [>= T, 32] bf16;
 * q_heads / kv_heads in {1, 2, 4, 8}; window a multiple of 64, landmark_chunk of 32; mix_logit one
 * value of mix_dtype; out [B, T, q_heads * 64]. The workspace
 * (fl_refresh_workspace_bytes, 16-byte aligned) then holds the rotated keys, for fl_refresh_state.
 *
 * fl_refresh_state: from that workspace and the same kv / landmark_kv, the decode state after the
 * sequence, zeros included: kt [B, kv_heads, 64, window] and v [B, kv_heads, window, 64] (the rows after
 * the last whole window in slots 0 ..), lkt [B, kv_heads, 64, slots] and lv [B, kv_heads, slots, 64]
 * (landmark j in slot j + 1; slots > n_landmarks), bf16.
 *
 * fl_latent_mean: mean over every completed chunk of rows, [B, T / chunk, width] bf16 (fp32 sums), and
 * the fp32 sum of the rows after the last one, tail [B, width] (zeros if none). latent [B, T, width]
 * bf16 with strides (multiples of 8), width a multiple of 8.
 *
 * fl_rms_norm: out = x rsqrt(mean x^2 + eps) weight over rows of dim (a multiple of 8, at most 4,096),
 * bf16 with fp32 maths (field_fusion_300m_screen_v20.py:94-104).
 */
size_t fl_refresh_workspace_bytes(int64_t B, int64_t T, int64_t kv_heads, int64_t n_landmarks);
int fl_refresh_attention(const void* q, int64_t q_stride_b, int64_t q_stride_t, const void* kv,
                         const void* landmark_kv, int64_t B, int64_t T, int64_t q_heads, int64_t kv_heads,
                         int64_t window, int64_t n_landmarks, int64_t landmark_chunk, const void* cos,
                         const void* sin, const void* mix_logit, int mix_dtype, void* out, void* workspace,
                         size_t workspace_bytes, void* stream);
int fl_refresh_state(const void* workspace, const void* kv, const void* landmark_kv, int64_t B, int64_t T,
                     int64_t kv_heads, int64_t window, int64_t n_landmarks, int64_t slots, void* kt, void* v,
                     void* lkt, void* lv, void* stream);
int fl_latent_mean(const void* latent, int64_t stride_b, int64_t stride_t, int64_t B, int64_t T, int64_t chunk,
                   int64_t width, void* mean, float* tail, void* stream);
int fl_rms_norm(const void* x, int64_t rows, int64_t dim, const void* weight, int w_dtype, float eps, void* out,
                void* stream);

/*
 * The Field block's elementwise work in training (field_only_v4_chunked_triton_wiki100.py:300-325,
 * 1169-1173, 1193-1195, 1219-1221), fp32 residual stream and maths; rows of dim (a multiple of 8, at
 * most 4,096), every [rows, dim] operand contiguous and 16-byte aligned:
 * fl_train_norm: out = x rstd weight, rstd = (mean x^2 + eps)^-1/2 per row (kept for the backward);
 * fl_train_gate_norm: x_new = x + out * sigmoid(gate) (rounded in g_dtype as the stock ops round), and
 *   its norm;
 * the backwards give the gradients of every input; gw [dim] is summed over the rows in a fixed order
 *   through workspace (fl_train_workspace_bytes(dim));
 * fl_swiglu_backward: gradient of fl_swiglu (hidden a multiple of 8);
 * fl_field_params_backward: gradients of fl_field_params' tr, ti, gamma.
 */
size_t fl_train_workspace_bytes(int64_t dim);
int fl_train_norm(const float* x, int64_t rows, int64_t dim, const float* weight, float eps, void* out, int out_dtype,
                  float* rstd, void* stream);
int fl_train_norm_backward(const void* gy, int gy_dtype, const float* x, int64_t rows, int64_t dim,
                           const float* weight, const float* rstd, float* gx, float* gw, void* workspace,
                           size_t workspace_bytes, void* stream);
int fl_train_gate_norm(const float* x, const void* out, const void* gate, int g_dtype, int64_t rows, int64_t dim,
                       const float* weight, float eps, float* x_new, void* normed, int normed_dtype, float* rstd,
                       void* stream);
int fl_train_gate_norm_backward(const float* g_x_new, const void* g_normed, int normed_dtype, const float* x_new,
                                const void* out, const void* gate, int g_dtype, int64_t rows, int64_t dim,
                                const float* weight, const float* rstd, float* gx, void* g_out, void* g_gate,
                                float* gw, void* workspace, size_t workspace_bytes, void* stream);
int fl_swiglu_backward(const void* gate_up, const void* gy, int dtype, int64_t rows, int64_t hidden, void* g_gate_up,
                       void* stream);
int fl_field_params_backward(const float* radius_logit, const float* theta, int64_t C, const float* gtr,
                             const float* gti, const float* ggamma, float* g_logit, float* g_theta, void* stream);

/*
 * Elementwise work of the refresh blocks in the stock ops' own roundings (same file, 131-253), bf16:
 * fl_refresh_step_in: one token at *pos (a device int64): q [B, q_heads * 64] = rotated queries of
 *   qlat [B, q_heads * 64 + latent]; rotated keys and values of kv [B, 2 * kv_heads * 64] into slot
 *   *pos % window of kt [B, kv_heads, 64, window] and v [B, kv_heads, window, 64]; lat_sum [B, latent]
 *   (fp32) += latent, restarted where *pos % chunk is 0 (chunk a power of two); mean = lat_sum / chunk;
 * fl_refresh_step_out: the rotated key and the value of kv into slot min(*pos / chunk + 1, slots - 1) of
 *   lkt [B, kv_heads, 64, slots] and lv [B, kv_heads, slots, 64];
 *   positions are clamped to the tables cos / sin [rope_len, 32];
 * fl_mask_scores: out [rows, lk] fp32 = scale * scores where column j <= the row's limit, else -inf; limit:
 *   mode 0 row % lq (causal), 1 *pos % period, 2 *pos / period;
 * fl_masked_softmax: out [rows, lk] bf16 = softmax of the scores fl_mask_scores forms, lk <= 1024; mode 3:
 *   limit (row % lq) / period;
 * fl_rope_heads: a prompt's heads of 64 for the products, windows = ceil(T / window), window <= T, zeros past
 *   T: rotated queries of x [B, T, q_heads * 64] (strides in elements, multiples of 8) to q [B, q_heads, T, 64]
 *   and local [B, windows, q_heads, window, 64]; of kv [B, T, 2 * kv_heads * 64] the rotated keys to
 *   kt [B, windows, kv_heads, 64, window] and the values to v [B, windows, kv_heads, window, 64];
 * fl_mix_heads: out [B, T, heads * 64] = local (as above) + sigmoid(mix_logit[0]) * g [B, heads, T, 64], g
 *   null for zeros;
 * fl_gate_add: out = x + sigmoid(gate) * a over n values, n a multiple of 8;
 * fl_mix: out = y + sigmoid(mix_logit[0]) * g over n values;
 * and of the Mamba-2 blocks as they run under bf16 autocast (field_fusion_wiki100_mamba2_v25.py:73-91):
 * fl_conv_silu: out [B, L, channels] fp32 = silu(causal depthwise conv of width 4), x bf16 with strides;
 * fl_decay_product: out [B, heads, n_chunks, s, s] bf16 = cb [B, n_chunks, s, s] exp(acs_i - acs_j) for
 *   j <= i and cb * 0 above, acs [B, heads, n_chunks, s] fp32, s a multiple of 8;
 * fl_ssd_operands: bf16 xdt [B, heads, n_chunks, s, P] = x dt and xw [B, heads, n_chunks, P, s] = x dt w_end,
 *   zeros past L; x [B, L, heads * P], dt [B, >= L, heads] with strides in elements, w_end [B, heads, n_chunks, s];
 * fl_ssd_finish: out [B, L, heads * P] fp32 = ((y + y_off exp(acs)) + D x) silu(z), y, y_off bf16
 *   [B, heads, n_chunks, s, P], x fp32 and z bf16 with strides in elements, multiples of 4; P a multiple of 4;
 * fl_state_update: ssm [B, heads, P, N] = ssm decay [B, heads] + xdt [B, heads, P] bm [B, N] in place
 *   (rows of bm bm_stride apart), and ssm16 its bf16 copy; N a multiple of 4.
 */
int fl_refresh_step_in(const void* qlat, const void* kv, const void* cos, const void* sin, const int64_t* pos,
                       int64_t B, int64_t q_heads, int64_t kv_heads, int64_t latent, int64_t rope_len, int64_t window,
                       int64_t chunk, void* q, void* kt, void* v, float* lat_sum, void* mean, void* stream);
int fl_refresh_step_out(const void* kv, const void* cos, const void* sin, const int64_t* pos, int64_t B,
                        int64_t kv_heads, int64_t rope_len, int64_t chunk, int64_t slots, void* lkt, void* lv,
                        void* stream);
int fl_mask_scores(const void* scores, int64_t rows, int64_t lk, int64_t lq, int mode, const int64_t* pos,
                   int64_t period, float scale, float* out, void* stream);
int fl_masked_softmax(const void* scores, int64_t rows, int64_t lk, int64_t lq, int mode, const int64_t* pos,
                      int64_t period, float scale, void* out, void* stream);
int fl_rope_heads(const void* x, int64_t x_stride_b, int64_t x_stride_t, const void* kv, int64_t kv_stride_b,
                  int64_t kv_stride_t, const void* cos, const void* sin, int64_t B, int64_t T, int64_t q_heads,
                  int64_t kv_heads, int64_t window, void* q, void* local, void* kt, void* v, void* stream);
int fl_mix_heads(const void* local, const void* g, const void* mix_logit, int mix_dtype, int64_t B, int64_t T,
                 int64_t heads, int64_t window, void* out, void* stream);
int fl_gate_add(const void* x, const void* gate, const void* a, int64_t n, void* out, void* stream);
int fl_conv_silu(const void* x, int64_t stride_b, int64_t stride_t, int64_t B, int64_t L, int64_t channels,
                 const void* w, const void* bias, int w_dtype, float* out, void* stream);
int fl_decay_product(const void* cb, const float* acs, int64_t B, int64_t heads, int64_t n_chunks, int64_t s,
                     void* out, void* stream);
int fl_ssd_operands(const float* x, int64_t x_stride_b, int64_t x_stride_t, const float* dt, int64_t dt_stride_b,
                    const float* w_end, int64_t B, int64_t heads, int64_t n_chunks, int64_t s, int64_t P, int64_t L,
                    void* xdt, void* xw, void* stream);
int fl_ssd_finish(const void* y, const void* y_off, const float* acs, const float* x, int64_t x_stride_b,
                  int64_t x_stride_t, const float* D, const void* z, int64_t z_stride_b, int64_t z_stride_t, int64_t B,
                  int64_t heads, int64_t n_chunks, int64_t s, int64_t P, int64_t L, float* out, void* stream);
int fl_state_update(const float* decay, const float* xdt, const float* bm, int64_t bm_stride, int64_t B, int64_t heads,
                    int64_t P, int64_t N, float* ssm, void* ssm16, void* stream);
int fl_mix(const void* y, const void* g, const void* mix_logit, int mix_dtype, int64_t n, void* out, void* stream);

/* Library version string (host function). No counterpart in the reference. */
const char* fl_version(void);

#ifdef __cplusplus
}
#endif

#endif /* FIELDS_AMD_H_ */
