/*
 * glm_moe.h -- C ABI of the MI355X (gfx950) routed-expert MoE library
 * (libglm_moe.so), the drop-in backend of glm-tpu's route-grouped FP8
 * routed-expert path.
 *
 * Every entry point takes plain device pointers and sizes, never allocates,
 * and enqueues its kernels on `stream` (a hipStream_t; NULL = default stream).
 * Nothing synchronises with the host: dynamic validity is written to a device
 * byte, exactly as the reference keeps its health bit on device.
 *
 * Return values: GLM_MOE_OK, or a status whose message glm_moe_last_error()
 * returns (thread-local).  GLM_MOE_ERR_ARGUMENT is the static shape/dtype
 * refusal the reference raises as ValueError at trace time.
 *
 * Tensor layouts (row-major, checkpoint [out, in] orientation):
 *   hidden        bf16 [tokens, H]          (uint16_t bit patterns)
 *   route ids     int32 [tokens, top_k], flat index t * top_k + slot
 *   route weights f32 [tokens, top_k]
 *   gate/up bits  uint8 e4m3fn [E, I, H],  scales f32 [E, I/128, H/128]
 *   down bits     uint8 e4m3fn [E, H, I],  scales f32 [E, H/128, I/128]
 *
 * Each declaration names the reference interface (GianluigiVitale/glm-tpu,
 * file:line) that it replaces.
 */
#ifndef GLM_MOE_H
#define GLM_MOE_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define GLM_MOE_ABI_VERSION 1

enum glm_moe_status {
  GLM_MOE_OK = 0,
  GLM_MOE_ERR_ARGUMENT = 1,  /* static geometry / dtype refusal (ValueError) */
  GLM_MOE_ERR_WORKSPACE = 2, /* workspace smaller than *_workspace_bytes() */
  GLM_MOE_ERR_DEVICE = 3     /* HIP runtime error (launch or device) */
};

enum glm_moe_dtype { GLM_MOE_F32 = 0, GLM_MOE_BF16 = 1 };

/* glm_moe_routed_experts flags */
#define GLM_MOE_ROUTE_SUM_BF16 0x1u   /* the decode body's per-owner bf16 route sum (routed_experts.py:293): JAX
                                         sums bf16 in FP32 and rounds once, so on one device (one owner) it is the
                                         FP32 route sum rounded once -- the same output as without the flag */
#define GLM_MOE_CHECK_WEIGHTS 0x2u    /* weights must be finite and >= 0 (prefill health, routed_experts.py:83) */
#define GLM_MOE_DROP_UNOWNED 0x4u     /* routes with ids outside [0, E) contribute zero (decode ownership, routed_experts.py:250-253) */
#define GLM_MOE_FP8_ACTIVATIONS 0x8u  /* native FP8 MFMA mode (no reference counterpart): activations quantised per
                                         (row, 128-wide K block) to e4m3 with an FP32 scale amax/448, e4m3 x e4m3
                                         block products, FP32 accumulation of product x weight scale x activation
                                         scale.  Prefill shapes only (more than 8 routes per expert on average,
                                         H/128 and I/128 multiples of 4, at most 64); others are refused. */

int glm_moe_abi_version(void);
const char* glm_moe_last_error(void);

/* Replaces glm_tpu/layers/fp8.py:113-126 decode_fp8_table (and the
 * dequantize_fp8_bits_block_weight arithmetic, :37-72):
 * out[n][k] = bf16(f32(e4m3(bits[n][k])) * scale[n / block_n][k / block_k]),
 * scale is [ceil(n / block_n), ceil(k / block_k)]. */
int glm_moe_decode_fp8_table(const uint8_t* bits, const float* scale, int64_t n, int64_t k,
                             int32_t block_n, int32_t block_k, uint16_t* out_bf16, void* stream);

/* Replaces the expert activation of glm_tpu/layers/moe/routed_experts.py:102,280
 * (and layers/mlp.py:48,65), (g * sigmoid(g) * u).astype(bf16) over bf16 g, u:
 * out[i] = bf16(bf16(g[i] * bf16(sigmoid(g[i]))) * u[i]), one bf16 rounding per
 * op -- the device function every gate/up kernel of this library applies in its
 * epilogue.  gate, up and out are n bf16 values. */
int glm_moe_swiglu_bf16(const uint16_t* gate, const uint16_t* up, int64_t n, uint16_t* out, void* stream);

/* Finite-bit gate of FP8 checkpoint payloads: adds to *count (device uint64)
 * the number of e4m3fn NaN encodings (0x7F, 0xFF) among n bytes; a loader
 * refuses any payload with a non-zero count.  Replaces the U8 branch of
 * _validate_finite_chunk (glm_tpu/model_loader/sharded_state/format.py:307-315),
 * run on the GPU over tables already in HBM.  The caller zeroes *count; bits
 * must be 4-byte aligned. */
int glm_moe_count_nonfinite_fp8(const uint8_t* bits, int64_t n, uint64_t* count, void* stream);

/* Replaces glm_tpu/layers/moe/router.py:20-55 route_glm_noaux_tc_logits: FP32
 * sigmoid scores of logits [tokens, experts]; the top_k experts of scores + bias
 * (bias may be NULL: zero), best first, ties to the lowest id; weights = the
 * chosen unbiased scores over their FP32 sum.  ids int32 / weights f32
 * [tokens, top_k].  experts <= 1024, top_k <= min(64, experts). */
int glm_moe_route_noaux_tc(const float* router_logits, int64_t tokens, int32_t num_experts,
                           const float* correction_bias, int32_t top_k, int32_t* route_indices,
                           float* route_weights, void* stream);

/* Per-row health of a layer routed from logits, the reference's router_valid &
 * grouped_valid (glm_tpu/layers/moe/router.py:161-166,
 * glm_tpu/models/glm_moe_dsa/decoder_layer.py:146): row_valid[t] = *layer_valid
 * and the row's logits, the bias (nullable) and the row's route weights
 * [tokens, top_k] are finite.  top_k <= min(64, experts). */
int glm_moe_route_row_health(const float* router_logits, int64_t tokens, int32_t num_experts,
                             const float* correction_bias, const float* route_weights, int32_t top_k,
                             const uint8_t* layer_valid, uint8_t* row_valid, void* stream);

/* Replaces glm_tpu/layers/moe/routed_experts.py:139-164 group_prefill_routes:
 * sorted_flat_ids = argsort(flat ids, stable), inverse_permutation, group_sizes
 * = bincount (invalid ids count as expert 0), *valid = all ids in [0, E) and no
 * duplicate id within a token's row.  num_experts <= 1024. */
int glm_moe_group_routes(const int32_t* route_indices, int64_t tokens, int32_t top_k,
                         int32_t num_experts, int32_t* sorted_flat_ids,
                         int32_t* inverse_permutation, int32_t* group_sizes, uint8_t* valid,
                         void* workspace, size_t workspace_bytes, void* stream);
/* Optional scratch of glm_moe_group_routes: with at least this many bytes of
 * workspace, large route sets are grouped by many workgroups (same result);
 * with NULL / too few bytes, by one. */
size_t glm_moe_group_routes_workspace_bytes(int64_t tokens, int32_t top_k, int32_t num_experts);

/* Replaces glm_tpu/layers/moe/routed_experts.py:167-183 gather_prefill_route_rows /
 * restore_prefill_route_rows and panels.py:98-104 unpack_expert_panel_rows:
 * dst[i] = mask[i] ? src[clamp(index[i] / div, 0, src_rows - 1)] : 0, whole rows of
 * row_bytes (a multiple of 4).  mask may be NULL (keep every row). */
int glm_moe_gather_rows(const void* src, int64_t src_rows, int64_t row_bytes,
                        const int32_t* index, int32_t div, const uint8_t* mask, int64_t rows,
                        void* dst, void* stream);

/* Replaces glm_tpu/kernels/fp8_grouped_matmul/panels.py:26-83 build_expert_panels
 * (32-row panels; capacity = ceil(rows / 32) + local_groups - 1).  group_offset is
 * a device int32 scalar.  num_groups <= 1024. */
int glm_moe_build_expert_panels(const int32_t* group_sizes, int32_t num_groups,
                                const int32_t* group_offset, int32_t rows, int32_t local_groups,
                                int32_t* expert_ids, int32_t* row_starts, int32_t* live_counts,
                                int32_t* active_panels, int32_t* restore_indices,
                                uint8_t* owned_rows, uint8_t* valid, void* stream);

/* Replaces panels.py:86-95 pack_expert_panel_rows: out [capacity, 32, row] with
 * rows past a panel's live count zero. */
int glm_moe_pack_expert_panel_rows(const void* values, int64_t rows, int64_t row_bytes,
                                   const int32_t* row_starts, const int32_t* live_counts,
                                   int32_t capacity, void* out, void* stream);

/* Replaces glm_tpu/kernels/fp8_grouped_matmul/panel_kernel.py:31-153
 * prefill_panel_fp8_matmul: sorted bf16 rows lhs [m, k] against their panel's local
 * expert ([groups, n, k] bits, [groups, n/128, k/128] scales), FP32 accumulation,
 * out [m, n] f32 or bf16 in sorted row order; unowned rows, and every row of an
 * invalid plan, are zero.  The plan is build_expert_panels' output. */
int glm_moe_panel_fp8_matmul(const uint16_t* lhs, int64_t m, int64_t k, const uint8_t* weight_bits,
                             const float* scale, int32_t groups, int64_t n,
                             const int32_t* panel_expert_ids, const int32_t* panel_row_starts,
                             const int32_t* panel_live_counts, const int32_t* active_panels,
                             int32_t capacity, const uint8_t* owned_rows, const uint8_t* valid,
                             int32_t result_dtype, void* out, void* stream);

/* The same with a workspace of glm_moe_panel_fp8_matmul_workspace_bytes bytes,
 * where the call lists runs of an expert's panels as tiles of up to 256 rows,
 * so that its weights are read once per tile instead of once per panel.  The
 * size is 0 (and a workspace is not looked at) for calls that run panel by panel:
 * k above 8192, m x k bf16 of 2 GiB and more, m n k below 2^29; so do pointers
 * not 16-byte aligned and a NULL workspace, as in glm_moe_panel_fp8_matmul. */
size_t glm_moe_panel_fp8_matmul_workspace_bytes(int64_t m, int64_t k, int32_t groups, int64_t n);
int glm_moe_panel_fp8_matmul_ws(const uint16_t* lhs, int64_t m, int64_t k, const uint8_t* weight_bits,
                                const float* scale, int32_t groups, int64_t n,
                                const int32_t* panel_expert_ids, const int32_t* panel_row_starts,
                                const int32_t* panel_live_counts, const int32_t* active_panels,
                                int32_t capacity, const uint8_t* owned_rows, const uint8_t* valid,
                                int32_t result_dtype, void* out, void* workspace, size_t workspace_bytes,
                                void* stream);

/* Replaces glm_tpu/kernels/fp8_grouped_matmul/kernel.py:125-299 fp8_routed_projection:
 * one bf16 row per route slot lhs [slots, k] against the slot's expert
 * (ids clipped to [0, experts)) in 1 or 2 tables; out [slots, tables, n] f32 or bf16;
 * unowned slots are zero.  Needs glm_moe_routed_projection_workspace_bytes(slots),
 * which calls with k above 8192 or lhs or bits not 16-byte aligned use. */
size_t glm_moe_routed_projection_workspace_bytes(int32_t slots);
int glm_moe_routed_projection(const uint16_t* lhs, int32_t slots, int64_t k, int32_t tables,
                              const uint8_t* bits0, const float* scale0, const uint8_t* bits1,
                              const float* scale1, int32_t experts, int64_t n,
                              const int32_t* local_expert_ids, const uint8_t* owned,
                              int32_t result_dtype, void* out, void* workspace,
                              size_t workspace_bytes, void* stream);

/* The routed-expert half of glm_tpu/layers/moe/routed_experts.py:27-128
 * prefill_moe_from_routes (and of :186-304 moe_grouped_routes) on one device:
 * group routes -> gate/up FP8 projections with fused bf16 SwiGLU -> down FP8
 * projection with fused bf16 route weighting -> FP32 route sum in slot order,
 * one bf16 rounding (GLM_MOE_ROUTE_SUM_BF16, the decode body's per-owner bf16
 * sum, gives the same result on one device).
 * out bf16 [tokens, H]; *valid = all ids in [0, E), no duplicate id in a row (and
 * weights finite >= 0 with GLM_MOE_CHECK_WEIGHTS).  As in the reference, an
 * invalid route set is still computed with its safe ids (an out-of-range id
 * counts as expert 0) and only *valid reports it; with GLM_MOE_DROP_UNOWNED an
 * out-of-range route instead contributes zero (the decode body's ownership).
 * Work is launched only for the experts the routes select. */
size_t glm_moe_routed_experts_workspace_bytes(int64_t tokens, int32_t top_k, int32_t num_experts,
                                              int64_t hidden, int64_t intermediate);
int glm_moe_routed_experts(const uint16_t* hidden, int64_t tokens, int64_t hidden_size,
                           const int32_t* route_indices, const float* route_weights,
                           int32_t top_k, int32_t num_experts, int64_t intermediate,
                           const uint8_t* gate_bits, const float* gate_scale,
                           const uint8_t* up_bits, const float* up_scale,
                           const uint8_t* down_bits, const float* down_scale, uint32_t flags,
                           uint16_t* out, uint8_t* valid, void* workspace, size_t workspace_bytes,
                           void* stream);

/* The MoE layer from router logits, for any number of tokens:
 * glm_moe_route_noaux_tc followed by glm_moe_moe_layer (shared non-null) or
 * glm_moe_routed_experts (shared null), bit for bit, in one call.  On decode
 * shapes with num_experts <= 256 the routing runs inside the decode gate/up
 * kernel (each workgroup routes its own token; no launch of its own);
 * otherwise the router kernel runs first, one wave per token over the whole
 * GPU (routing inside the route plan's few workgroups was measured slower).
 * Replaces the composition of the reference's prefill MLP from the logits on
 * -- route_glm_noaux_tc_logits (glm_tpu/layers/moe/router.py:20-55, the
 * selection inside prefill_router, :102-166) feeding prefill_moe_from_routes
 * (routed_experts.py:27-128, whose group_prefill_routes is :139-164),
 * glm_tpu/models/glm_moe_dsa/decoder_layer.py:123-146.  router_logits
 * [tokens, num_experts] f32, correction_bias [num_experts] f32 (nullable:
 * zero); route_indices / route_weights [tokens, top_k] are outputs;
 * top_k <= 64.  Same workspace as glm_moe_routed_experts. */
int glm_moe_moe_layer_from_router_logits(const uint16_t* hidden, int64_t tokens, int64_t hidden_size,
                                         const float* router_logits, const float* correction_bias, int32_t top_k,
                                         int32_t num_experts, int64_t intermediate, const uint8_t* gate_bits,
                                         const float* gate_scale, const uint8_t* up_bits, const float* up_scale,
                                         const uint8_t* down_bits, const float* down_scale, uint32_t flags,
                                         const uint16_t* shared, float routed_scale, int32_t* route_indices,
                                         float* route_weights, uint16_t* out, uint8_t* valid, void* workspace,
                                         size_t workspace_bytes, void* stream);

/* One expert-parallel share of the routed experts: the tables hold the
 * local_experts experts of global ids [expert_offset, expert_offset +
 * local_experts) out of num_experts; route_indices are global ids.  Only the
 * owned routes are planned, tiled and computed (work is launched for the
 * share's selected experts alone); out f32 [tokens, H] is the share's FP32
 * route sum -- rounded to bf16 values with GLM_MOE_ROUTE_SUM_BF16, the decode
 * body's per-owner bf16 sum -- which the caller sums over the expert axis and
 * passes to glm_moe_moe_layer_epilogue.  Replaces the share-local part of
 * prefill_moe_from_routes (glm_tpu/layers/moe/routed_experts.py:82-112, the
 * owned panels of panels.py:26-83 with offset = axis_index("expert") *
 * local_experts) and of moe_grouped_routes (:250-293, the owned-slot mask).
 * *valid is the whole route set's health (ids in [0, num_experts), no
 * duplicate in a row, weights finite and >= 0 with GLM_MOE_CHECK_WEIGHTS), the
 * same on every share.  An invalid id stands for expert 0 (owned by the share
 * at offset 0), or is dropped with GLM_MOE_DROP_UNOWNED.  Workspace:
 * glm_moe_routed_experts_workspace_bytes(tokens, top_k, local_experts, H, I).
 * local_experts <= 1023. */
int glm_moe_routed_experts_share(const uint16_t* hidden, int64_t tokens, int64_t hidden_size,
                                 const int32_t* route_indices, const float* route_weights, int32_t top_k,
                                 int32_t num_experts, int32_t expert_offset, int32_t local_experts,
                                 int64_t intermediate, const uint8_t* gate_bits, const float* gate_scale,
                                 const uint8_t* up_bits, const float* up_scale, const uint8_t* down_bits,
                                 const float* down_scale, uint32_t flags, float* out, uint8_t* valid,
                                 void* workspace, size_t workspace_bytes, void* stream);

/* The layer epilogue after the sum over the expert axis (the psum of
 * glm_tpu/layers/moe/routed_experts.py:113-117 / :294-295, then :125 / :303):
 * out = bf16(bf16(bf16(routed) * bf16(routed_scale)) + shared) with routed the
 * FP32 [tokens, H] sum of the shares' partials and shared the shared expert's
 * bf16 rows; a non-finite output clears *valid (:126), which is otherwise left
 * as the share call set it.  hidden_size a multiple of 8. */
int glm_moe_moe_layer_epilogue(const float* routed, int64_t tokens, int64_t hidden_size, const uint16_t* shared,
                               float routed_scale, uint16_t* out, uint8_t* valid, void* stream);

/* Stage timing for benchmarks: glm_moe_routed_experts_timed is
 * glm_moe_routed_experts whose kernels record HIP events at their own start
 * and end (hipExtLaunchKernelGGL): the kernel of stage i (0 route plan,
 * 1 gate/up, 2 down, 3 combine) records events[2i] and events[2i + 1], and
 * bit i of *timed_stages is set when stage i ran a kernel (the decode path
 * has no separate plan or combine kernel).  Events come from
 * glm_moe_event_create.  No reference counterpart (the reference labels its
 * kernels for the TPU profiler, glm_tpu/kernels/names.py:1-31). */
int glm_moe_event_create(void** event);
int glm_moe_event_destroy(void* event);
int glm_moe_event_elapsed_ms(void* start, void* stop, float* ms);
int glm_moe_routed_experts_timed(const uint16_t* hidden, int64_t tokens, int64_t hidden_size,
                                 const int32_t* route_indices, const float* route_weights,
                                 int32_t top_k, int32_t num_experts, int64_t intermediate,
                                 const uint8_t* gate_bits, const float* gate_scale,
                                 const uint8_t* up_bits, const float* up_scale,
                                 const uint8_t* down_bits, const float* down_scale,
                                 uint32_t flags, uint16_t* out, uint8_t* valid, void* workspace,
                                 size_t workspace_bytes, void* const* events, uint32_t* timed_stages,
                                 void* stream);

/* The whole MoE layer output given the shared expert's rows: the routed
 * experts exactly as glm_moe_routed_experts, then, fused into the kernel that
 * finishes the route sum, out = bf16(bf16(routed * bf16(routed_scale)) + shared).
 * Replaces the layer epilogue of prefill_moe_from_routes and moe_grouped_routes
 * (glm_tpu/layers/moe/routed_experts.py:119-127 and :297-304); the shared
 * expert itself (bf16 resident GEMMs, :119-124 / :269-302) is the caller's,
 * e.g. hipBLASLt, and shared holds its bf16 output [tokens, hidden_size].
 * valid additionally requires every output element to be finite (:126).
 * Same workspace as glm_moe_routed_experts. */
int glm_moe_moe_layer(const uint16_t* hidden, int64_t tokens, int64_t hidden_size,
                      const int32_t* route_indices, const float* route_weights, int32_t top_k,
                      int32_t num_experts, int64_t intermediate, const uint8_t* gate_bits,
                      const float* gate_scale, const uint8_t* up_bits, const float* up_scale,
                      const uint8_t* down_bits, const float* down_scale, uint32_t flags,
                      const uint16_t* shared, float routed_scale, uint16_t* out, uint8_t* valid,
                      void* workspace, size_t workspace_bytes, void* stream);

/* glm_moe_moe_layer of prefill shapes with the shared expert computed inside the
 * same launches from its resident bf16 tables (gate / up [intermediate,
 * hidden_size], down [hidden_size, intermediate]), at the rounding points of
 * glm_moe_moe_layer_resident: its rows are work items beside the experts' in the
 * gate/up and the down launch.  With router_logits (nullable; correction_bias
 * nullable) the layer routes first and route_indices / route_weights are
 * outputs, as glm_moe_moe_layer_from_router_logits.  Shapes for which
 * glm_moe_moe_layer_shared_workspace_bytes is not 0: more than the decode
 * kernels' routes, hidden_size a multiple of 256, both sizes at most 8192,
 * operands below 2 GiB; no FP8 mode.  hidden and the shared tables are 16-byte
 * aligned (else GLM_MOE_ERR_ARGUMENT).  Replaces prefill_moe_from_routes' shared
 * expert and epilogue (glm_tpu/layers/moe/routed_experts.py:119-127) with the
 * routed half (:82-117). */
size_t glm_moe_moe_layer_shared_workspace_bytes(int64_t tokens, int32_t top_k, int32_t num_experts, int64_t hidden,
                                                int64_t intermediate);
int glm_moe_moe_layer_shared(const uint16_t* hidden, int64_t tokens, int64_t hidden_size,
                             const float* router_logits, const float* correction_bias, int32_t* route_indices,
                             float* route_weights, int32_t top_k, int32_t num_experts, int64_t intermediate,
                             const uint8_t* gate_bits, const float* gate_scale, const uint8_t* up_bits,
                             const float* up_scale, const uint8_t* down_bits, const float* down_scale, uint32_t flags,
                             const uint16_t* shared_gate, const uint16_t* shared_up, const uint16_t* shared_down,
                             float routed_scale, uint16_t* out, uint8_t* valid, void* workspace,
                             size_t workspace_bytes, void* stream);

/* 1 when a layer of this geometry runs on the decode kernels (tokens * top_k
 * <= 64 and the hidden / intermediate sizes they stage), the shapes
 * glm_moe_moe_layer_resident takes; else 0.  Host-only query, no reference
 * counterpart (the reference picks its layer body by program, not by shape). */
int glm_moe_uses_decode_kernels(int64_t tokens, int32_t top_k, int64_t hidden_size, int64_t intermediate);

/* Weight rows of a work item of a bf16 layer's prefill projections, 512 (tall
 * stripes) or 256, for a call with the tables of local_experts of num_experts
 * on the current device; 0 where the layer does not run on the prefill
 * kernels.  Host-only query, no reference counterpart. */
int glm_moe_prefill_stripe_rows(int64_t tokens, int32_t top_k, int32_t local_experts, int32_t num_experts,
                                int64_t hidden_size, int64_t intermediate);

/* The whole decode MoE layer in two kernels: glm_moe_moe_layer with the
 * shared expert computed inside the same launches from its resident bf16
 * tables (gate/up [shared_intermediate, hidden_size], down [hidden_size,
 * shared_intermediate]; shared_intermediate must equal intermediate) instead
 * of a caller-computed output -- one pass over HBM for routed and shared
 * weights.  Replaces moe_grouped_routes' shared expert and epilogue
 * (glm_tpu/layers/moe/routed_experts.py:269-304; resident_matmul,
 * glm_tpu/layers/linear.py:26-33): bf16 operands, FP32 sums, bf16 rounding of
 * gate/up, SwiGLU and down.  Decode shapes only (tokens * top_k <= 64); the
 * shared weights are streamed once per token, so it pays for a single row (the
 * decode body).  Same workspace as glm_moe_routed_experts. */
int glm_moe_moe_layer_resident(const uint16_t* hidden, int64_t tokens, int64_t hidden_size,
                               const int32_t* route_indices, const float* route_weights, int32_t top_k,
                               int32_t num_experts, int64_t intermediate, const uint8_t* gate_bits,
                               const float* gate_scale, const uint8_t* up_bits, const float* up_scale,
                               const uint8_t* down_bits, const float* down_scale, uint32_t flags,
                               const uint16_t* shared_gate, const uint16_t* shared_up,
                               const uint16_t* shared_down, int64_t shared_intermediate, float routed_scale,
                               uint16_t* out, uint8_t* valid, void* workspace, size_t workspace_bytes,
                               void* stream);

/* glm_moe_moe_layer_resident without a workspace argument, for callers that
 * cannot allocate (code under HIP graph capture, tight serving loops, harnesses
 * that forbid hipMalloc).  No reference counterpart: the reference's functional
 * JAX code has no caller-visible memory.  Its scratch (the routes' and the
 * shared expert's bf16 SwiGLU rows, at most 512 KiB: tokens * top_k <= 64,
 * intermediate <= 2048) lives in a static device array of the library, one copy
 * per GPU, held until the process ends; nothing in it needs clearing (every
 * element the down kernel reads is written by the gate/up kernel of the same
 * call).  It calls no allocator.  Every call on one GPU shares that GPU's
 * scratch: calls that overlap on one GPU (different streams, or host threads
 * without ordering) race.  Decode shapes only; same arguments and results as
 * glm_moe_moe_layer_resident. */
int glm_moe_moe_layer_resident_noalloc(const uint16_t* hidden, int64_t tokens, int64_t hidden_size,
                                       const int32_t* route_indices, const float* route_weights, int32_t top_k,
                                       int32_t num_experts, int64_t intermediate, const uint8_t* gate_bits,
                                       const float* gate_scale, const uint8_t* up_bits, const float* up_scale,
                                       const uint8_t* down_bits, const float* down_scale, uint32_t flags,
                                       const uint16_t* shared_gate, const uint16_t* shared_up,
                                       const uint16_t* shared_down, int64_t shared_intermediate,
                                       float routed_scale, uint16_t* out, uint8_t* valid, void* stream);

/* The decode MoE MLP from router logits, in the same two launches as
 * glm_moe_moe_layer_resident: the noaux_tc routing of
 * glm_moe_route_noaux_tc (route_glm_noaux_tc_logits,
 * glm_tpu/layers/moe/router.py:20-55) is computed inside the gate/up kernel,
 * each workgroup for its own token, instead of in a launch of its own; then the
 * layer of glm_moe_moe_layer_resident.  Replaces the composition of the
 * reference's decode MLP body, router then moe_grouped_routes
 * (glm_tpu/models/glm_moe_dsa/decoder_layer.py:636-656), from the router
 * logits on.  router_logits [tokens, num_experts] f32, correction_bias
 * [num_experts] f32 (nullable: zero); route_indices / route_weights
 * [tokens, top_k] are outputs (the selected ids and renormalised weights,
 * bit-equal to glm_moe_route_noaux_tc's).  Decode shapes only, at most 256
 * experts.  Same workspace as glm_moe_routed_experts. */
int glm_moe_moe_layer_from_logits(const uint16_t* hidden, int64_t tokens, int64_t hidden_size,
                                  const float* router_logits, const float* correction_bias, int32_t top_k,
                                  int32_t num_experts, int64_t intermediate, const uint8_t* gate_bits,
                                  const float* gate_scale, const uint8_t* up_bits, const float* up_scale,
                                  const uint8_t* down_bits, const float* down_scale, uint32_t flags,
                                  const uint16_t* shared_gate, const uint16_t* shared_up,
                                  const uint16_t* shared_down, int64_t shared_intermediate, float routed_scale,
                                  int32_t* route_indices, float* route_weights, uint16_t* out, uint8_t* valid,
                                  void* workspace, size_t workspace_bytes, void* stream);

/* The bf16 shared expert of a few rows (1 <= tokens <= 8): gate and up
 * [shared_intermediate, hidden_size], SwiGLU, down [hidden_size,
 * shared_intermediate], out [tokens, hidden_size] bf16, in two launches that
 * read every weight byte once for all rows.  Replaces the resident bf16 shared
 * expert of the layer bodies (glm_tpu/layers/moe/routed_experts.py:119-124 and
 * :269-302; resident_matmul, glm_tpu/layers/linear.py:26-33) at their
 * rounding points: bf16 gate and up sums, bf16 SwiGLU (:123, :280), bf16 down
 * sums; FP32 accumulation of exact bf16 products.  Its output is the `shared`
 * input of glm_moe_moe_layer.  Workspace: the SwiGLU rows,
 * glm_moe_shared_expert_rows_workspace_bytes(tokens, shared_intermediate). */
size_t glm_moe_shared_expert_rows_workspace_bytes(int64_t tokens, int64_t shared_intermediate);
int glm_moe_shared_expert_rows(const uint16_t* hidden, int64_t tokens, int64_t hidden_size,
                               const uint16_t* shared_gate, const uint16_t* shared_up, const uint16_t* shared_down,
                               int64_t shared_intermediate, uint16_t* out, void* workspace, size_t workspace_bytes,
                               void* stream);

/* Synthetic FP8 expert tables for tests and benchmarks, the reference's fixture
 * recipe (tools/equivalence/fixture.py:158-172) with 128x128 block scales:
 * w ~ N(0, sigma) (counter-based hash + Box-Muller), scale = amax/448 per block,
 * bits = e4m3fn(clamp(w/scale, +-448)) RNE.  bits [experts, n, k], scales
 * [experts, n/128, k/128].  Deterministic in (seed, geometry). */
int glm_moe_synthesize_fp8_weights(uint64_t seed, int32_t experts, int64_t n, int64_t k,
                                   float sigma, uint8_t* bits, float* scales, void* stream);

#ifdef __cplusplus
}
#endif

#endif /* GLM_MOE_H */
