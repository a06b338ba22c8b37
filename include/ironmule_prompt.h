/*
 * ironmule_prompt.h — C ABI of the 4-bit products for more than 32 activation rows on MI355X
 * (gfx950), in libironmule_qmv.so: prompts and expert batches.
 *
 * The weights are read as they are stored (w, scales, biases of ironmule_qmv.h); the
 * activations are packed first, into the order the matrix instructions read.  Each output is
 * sum_k (s q + b) x with exact products and fp32 sums.
 *
 * Contract (as for ironmule_qmv.h): device pointers allocated by the caller, work queued on
 * `stream`, no allocation or synchronisation per call, int32 return codes with
 * imq_last_error() for the message.
 */
#ifndef IRONMULE_PROMPT_H
#define IRONMULE_PROMPT_H

#include <stddef.h>
#include <stdint.h>

#include "ironmule_qmv.h"
#include "ironmule_step.h"

#ifdef __cplusplus
extern "C" {
#endif

#define IMQ_PROMPT_MAX_PROBLEMS 3
#define IMQ_PROMPT_MAX_EXPERTS 1024
#define IMQ_PROMPT_MAX_ROWS (1 << 20)
#define IMQ_PROMPT_MAX_K (1 << 17)

/* Bytes of packed activations for M rows of K values (0: M or K out of range). */
IMQ_API size_t imq_prompt_packed_bytes(int32_t M, int32_t K);

/* Packs x, M bf16 rows of K values ldx elements apart (16-byte aligned, ldx a multiple of 8),
 * into `packed` (imq_prompt_packed_bytes, 16-byte aligned).  One packing serves every product
 * of the same rows. */
IMQ_API int32_t imq_prompt_pack(const uint16_t* x, int64_t ldx, int32_t M, int32_t K, void* packed, void* stream);

/* Bytes of workspace imq_prompt_product takes for these problems (0: none). */
IMQ_API size_t imq_prompt_product_workspace(const imq_problem* p, int32_t count, int32_t M);

/* y_i = x W_i^T for the packed rows x and 1 to 3 weights of the same K (x and ldx of the
 * problems are not read); y bf16 or fp32, rows ldy apart.  The workspace needs no
 * preparation; calls that share one must not overlap.
 * Replaces the prompt path of ironmule/cuda_native.py:177-179 (dequantise, then a matrix
 * product). */
IMQ_API int32_t imq_prompt_product(const imq_problem* p, int32_t count, const void* packed, int32_t M,
                                   int32_t group_size, int32_t bits, int32_t y_dtype, void* workspace,
                                   size_t workspace_bytes, void* stream);

/* The plan of a product of M rows by 1 to 3 weights of N[i] x K on `cus` compute units, with at most
 * max_splits K-ranges (8 in imq_prompt_product; in a layer 1 for q/k/v and gate/up, 8 for o and
 * down): rows of a workgroup's tile (32, 64 or 128) and K-ranges.  Needs no device. */
IMQ_API int32_t imq_prompt_plan(const int32_t* N, int32_t count, int32_t M, int32_t K, int32_t max_splits, int32_t cus,
                                int32_t* tile_rows, int32_t* splits);

/* imq_prompt_pack and imq_prompt_product of one weight in one call; the workspace (16-byte
 * aligned) holds the packed rows and the product's. */
IMQ_API size_t imq_prompt_matmul_workspace(int32_t M, int32_t N, int32_t K);
IMQ_API int32_t imq_prompt_matmul(const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
                                  const uint16_t* x, int64_t ldx, void* y, int64_t ldy, int32_t M, int32_t N,
                                  int32_t K, int32_t group_size, int32_t bits, int32_t y_dtype, void* workspace,
                                  size_t workspace_bytes, void* stream);

/* Bytes of workspace imq_prompt_experts takes (0: a size out of range). */
IMQ_API size_t imq_prompt_experts_workspace(int32_t experts, int32_t pairs, int32_t K);

/* Rows of a tile in imq_prompt_experts (32 or 64) on `cus` compute units.  Needs no device. */
IMQ_API int32_t imq_prompt_experts_plan(int32_t experts, int32_t pairs, int32_t N, int32_t cus, int32_t* tile_rows);

/* y[p] = x[p / rows_per_x] W[idx[p]]^T for `pairs` (token, expert) pairs over stacked expert
 * weights (E, N, K/8), scales and biases (E, N, K/64): the pairs are sorted by expert on the
 * device, each expert's rows taken together.  An index below zero counts from the last expert;
 * a pair whose index is outside the stack gets zeros.  The workspace (16-byte aligned) needs no
 * preparation.
 * Replaces mx.gather_qmm beyond the gather kernel's pairs (ironmule/cuda_native.py:199-218). */
IMQ_API int32_t imq_prompt_experts(const uint32_t* w, const uint16_t* scales, const uint16_t* biases,
                                   int32_t experts, const uint16_t* x, int64_t ldx, int32_t rows_per_x,
                                   const int32_t* idx, int32_t pairs, void* y, int64_t ldy, int32_t N, int32_t K,
                                   int32_t group_size, int32_t bits, int32_t y_dtype, void* workspace,
                                   size_t workspace_bytes, void* stream);

/* A whole prompt of one request through decoder layers (head size 128), one call per layer:
 *   x = rms_norm(h) ; q,k,v = x W^T ; q,k = rope(rms_norm_head(q, k)) at positions 0 .. tokens-1 ;
 *   KV[slot][0 .. tokens-1] = k, v ; o = causal attention ; h += bf16(o Wo^T) ; x = rms_norm(h) ;
 *   h += bf16(bf16(silu(bf16(x Wg^T)) * bf16(x Wu^T)) Wd^T)
 * with fp32 residual stream h (tokens, hidden) and bf16 activations between the steps.  The last
 * addition of a layer is left in the workspace for the next call (`first` of the first layer is 1,
 * of the others 0) or for imq_prompt_finish, which
 * adds it to the last `rows` rows; the calls of one prompt share one workspace
 * (256-byte aligned, no preparation) and no other call may use it meanwhile.
 * Replaces a prompt's pass through the layers (ironmule/cuda_native.py:171-179;
 * ironmule/dense_plan.py:337-363). */
typedef struct {
  int32_t tokens, hidden, heads, kv_heads, intermediate, capacity, num_slots, slot;
  float eps;
  double theta; /* the rotary base: angles are computed in double */
} imq_prompt_shape;

IMQ_API size_t imq_prompt_layer_workspace(const imq_prompt_shape* shape);
IMQ_API int32_t imq_prompt_layer(const imq_step_layer* layer, const imq_prompt_shape* shape, float* h, int32_t first,
                                 void* workspace, size_t workspace_bytes, void* stream);
IMQ_API int32_t imq_prompt_finish(const imq_prompt_shape* shape, float* h, int32_t rows, void* workspace,
                                  size_t workspace_bytes, void* stream);

#ifdef __cplusplus
}
#endif

#endif /* IRONMULE_PROMPT_H */
