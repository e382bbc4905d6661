/* tlhip_debug.h -- measurement and diagnostic hooks of libtlhip.so. NOT part of the drop-in boundary (include/tlhip.h is
 * what a maintainer of the reference binds in place of cuda_kernels.h:104-643); none of these has a counterpart in the
 * reference. bench.py, tools/ and the tests use them through tinyllama.cpp_amd/capi.py (DEBUG_SIGNATURES). */
#ifndef TLHIP_DEBUG_H
#define TLHIP_DEBUG_H
#include "tlhip.h"
#ifdef __cplusplus
extern "C" {
#endif

/* From now on every chain launch of the decode step (tl_gemv.hip, chain_kernel) writes 8 realtime stamps (100 MHz) per
 * workgroup into buf_dev, laid out [launch][task][256 workgroups][8] u64 in launch order, until cap_u64 words are used:
 * [0] workgroup entry, [1] first weight loads issued, [2] predecessor task seen complete, [3] x staged, [4] last loads
 * issued, [5] all stores acknowledged and the workgroup met, [6] arrival added. NULL switches the stamps off. Run the step
 * eagerly (TL_NO_GRAPH=1): a captured graph keeps the pointer it was captured with. */
int tl_chain_set_stamps(unsigned long long* buf_dev, size_t cap_u64);

/* Measurement hook (no counterpart in the reference): `iters` back-to-back tl_matvec_q launches cycling through
 * `nw` equally-shaped matrices (use more than the 256 MiB Infinity Cache holds), timed with HIP events on `stream`. */
int tl_bench_matvec(const tl_qweight* const* ws, int nw, const float* x_dev, float* y_dev, int iters, int warmup,
                    float* avg_us_out, void* stream);
/* Measurement hook (experiment, no counterpart in the reference): the tl_bench_matvec chain captured into a two-branch
 * graph in which a second stream pulls matrix i+1 into the Infinity Cache while the GEMV over matrix i runs
 * (prefetch_blocks workgroups of 256 threads; 0 = no prefetch branch, same graph otherwise). */
int tl_bench_matvec_prefetch(const tl_qweight* const* ws, int nw, const float* x_dev, float* y_dev, int reps,
                             int prefetch_blocks, float* avg_us_out);
/* Diagnostic hook (no counterpart in the reference): one tl_matvec_q-shaped launch of an instrumented build of the
 * GEMV kernel; stamps_dev[10 * grid * waves] u64 receives per-wave shader-clock stamps (see tl_gemv.hip). */
int tl_debug_gemv_stamps(const tl_qweight* w, const float* x_dev, float* y_dev, unsigned long long* stamps_dev,
                         int* grid_out, int* waves_out, void* stream);
/* Measurement hook (no counterpart in the reference): runs n_steps greedy decode steps EAGERLY (no graph) on the
 * model's stream with a HIP event after every kernel, and accumulates per-kernel-kind milliseconds and launch
 * counts into kind_ms_out[9] / kind_launches_out[9]: 0 embed, 1 norm+QKV GEMV, 2 RoPE+KV write, 3 attention,
 * 4 O GEMV+residual, 5 norm+gate/up GEMV+SwiGLU, 6 down GEMV+residual, 7 norm+lm_head GEMV, 8 sample+advance. */
int tl_model_profile_decode(tl_model* m, int first_token, int start_pos, int n_steps, float* kind_ms_out,
                            int* kind_launches_out);
/* Measurement hook (no counterpart in the reference): `iters` back-to-back launches of ONE kind of the decode step's
 * GEMV kernels (kinds as above: 1, 4, 5, 6, 7), cycling through the layers so that every launch streams from HBM,
 * timed with HIP events on the engine's stream. Leaves activations / logits in an unspecified state. kind 9: the
 * step's all-reduce of f32[hidden] of a linked tensor-parallel shard (a collective call: every rank makes it). */
int tl_model_bench_kernel(tl_model* m, int kind, int iters, int warmup, float* avg_us_out, double* bytes_per_launch_out);

/* Diagnostic hook (no counterpart in the reference): launches of the expanded-plane GEMM kernel (tl_qweight_expand) so far
 * in this process: lets a test prove which kernel formed a result. */
int tl_debug_gemm_px_launches(long long* count_out);
/* ... and launches that split activations into a chunk product's planes (those that attention writes itself are none) */
int tl_debug_split_launches(long long* count_out);
/* ... and attentions by the two-part f16 kernels (tl_hattn.hip): one a layer of a prompt's chunk that takes them */
int tl_debug_half_attention_launches(long long* count_out);
/* ... and GEMV launches with a norm whose input is not staged from registers as a whole (graph captures count once) */
int tl_debug_gemv_general_norms(long long* count_out);
/* ... and f16 products of Q4_K and Q6_K matrices in one launch, counts_out[9] by the Q4_K tiles' workgroup shape (tl_debug_half_gemm) */
int tl_debug_half_pair_launches(long long* counts_out);
/* ... and one-token products of a layer list that carry the residual norm in front of them (graph captures count once) */
int tl_debug_resid_products(long long* count_out);

/* Test hook (no counterpart in the reference): tl_matmul_q through the f16 form that a model's chunks and multi-sequence steps
 * take (tl_hgemm.hip), any number of tokens, in a workgroup shape (0: 64 rows x 16 tokens, 1: 128 x 32, 2: 256 x 64, 3: in waves of 64
 * rows, 512 x 64 in Q4_K and 256 x 64 in Q8_K, 4: 128 x 64, 5 and 6: 64 and 128 rows x 8 tokens, whose two parts share an instruction, 7:
 * 128 x 16 in waves of 16 rows, 8: 64 x 32 in the same) and a number of K slices, none of them empty. Rows that are not whole super-blocks
 * (Q8_0) run shape 4 where 2 is asked for: the same sums, and no plan chooses 2 for them. */
int tl_debug_half_gemm(const tl_qweight* w, const float* x_dev, float* y_dev, int num_tokens, int shape, int slices, void* stream);

/* Test hook (no counterpart in the reference): tl_dense_matmul's product with one term through the kernel that takes the items from a
 * bf16 plane (tl_dense.hip): rows ldx floats apart, whole steps of 64 columns, the first `exact_items` (at most 32) items with two
 * terms, `waves` 4 (two workgroups a CU) or 8 (one), plane_dev room for [num_tokens + 32][cols] bf16 (NULL: the kernel that converts
 * them itself, in the tile of TL_DENSE_TILE, whose order of sums the first items have in either). */
int tl_debug_dense_plane(const void* w_bf16_dev, int rows, int cols, const float* x_dev, int ldx, float* y_dev, int num_tokens,
                         int exact_items, int waves, void* plane_dev, void* stream);
/* ... and whether a model's product of these sizes takes that kernel, with room for `room` bf16 numbers, on `cus` compute units (a rule
 * on the host: no device) */
int tl_debug_dense_plane_taken(int rows, int cols, int num_tokens, long long room, int cus);

/* Test hook (no counterpart in the reference): tl_swa_attention's product through the two-part f16 kernels that prompt chunks
 * take (tl_hattn.hip); head sizes 64, 96 or 128 over 64 and 128 over 128, a positive scale, 16-byte addresses. */
int tl_debug_half_attention(const float* q_dev, const float* k_cache_dev, const float* v_cache_dev, float* out_dev,
                            int num_tokens, int start_pos, int heads, int kv_heads, int dim, int vdim, int window, float scale,
                            void* stream);

/* Test hook (no counterpart in the reference): the row-tile attention of packed prompts (tl_prefill.hip) over q [T][heads][dim], token i
 * at positions_host[i] of sequence seq_idx_host[i], whose caches [*][kv_heads][dim] lie seq_stride floats apart; dim 64 or 128. */
int tl_debug_packed_attention(const float* q_dev, const float* k_cache_dev, const float* v_cache_dev, float* out_dev, long long seq_stride,
                              const int* positions_host, const int* seq_idx_host, int num_tokens, int heads, int kv_heads, int dim,
                              float scale, void* stream);

/* Test hook (no counterpart in the reference): the attention of multi-sequence steps and of prompts of few tokens (tl_batch.hip) over q
 * [T][heads][dim], token i at positions_dev[i] of sequence seq_idx_dev[i] (both NULL: at start_pos + i of sequence 0), whose caches
 * [max_seq][kv_heads][dim] lie seq_stride floats apart; tokens elsewhere are left out. dim 64 or 128, 1, 2, 3, 4 or 8 heads a kv head. */
int tl_debug_batch_attention(const float* q_dev, const float* k_cache_dev, const float* v_cache_dev, float* out_dev, long long seq_stride,
                             const int* positions_dev, const int* seq_idx_dev, int start_pos, int num_tokens, int heads, int kv_heads,
                             int dim, int max_seq, int num_seq, float scale, void* stream);

/* Parity hook for layer-list models (no counterpart in the reference): cb(ctx, layer, x_dev, num_tokens, width) is called after
 * every layer of every forward pass, the stream synchronised, with the residual stream on the device. NULL switches it off.
 * With the hook set the decode step must run eagerly (TL_NO_GRAPH=1 at finalize): a captured step cannot call back. */
typedef void (*tl_layer_hook_fn)(void* ctx, int layer, const float* x_dev, int num_tokens, int width);
int tl_model_debug_layer_hook(tl_model* m, tl_layer_hook_fn cb, void* ctx);

/* ---- libtlhip_tools.so (csrc/tl_stream.hip; built beside libtlhip.so, not part of it): a measured negative result kept
 * for the record -- a persistent ring-loader engine. */
/* Measurement / parity hook (no counterpart in the reference): y_i = W_i x through the ring-loader engine (tl_stream.hip),
 * the nw equally shaped matrices as nw phases of ONE persistent launch (ys_dev: [nw][rows]); avg_us_out (may be NULL) =
 * microseconds per matrix over `reps` launches. */
int tl_stream_matvec(const tl_qweight* const* ws, int nw, const float* x_dev, float* ys_dev, int reps, float* avg_us_out,
                     void* stream);

#ifdef __cplusplus
}
#endif
#endif
