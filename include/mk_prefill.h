/*
 * C ABI of the prompt forward (libmk_prefill.so): the dense Llama forward over a whole prompt that fills the KV cache
 * before decoding starts (the reference runs it as a PyTorch module, megakernels/llama.py:232-296,328-348,384-403).
 *
 * Every function launches on `stream` (a hipStream_t, NULL = default stream) without synchronising and returns 0 or a
 * negative error with a message in mk_prefill_last_error(); a null pointer or a shape outside the kernels is such an error,
 * and nothing is launched then.  All tensors are contiguous device memory; bf16 tensors are
 * passed as uint16_t bit patterns.  A "row" is one position of one sequence: rows = batch * seq.
 */
#ifndef MK_PREFILL_H
#define MK_PREFILL_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* What the kernels need to know of the architecture and of this call. */
typedef struct mk_prefill_shape {
    int32_t batch, seq;
    int32_t num_attention_heads, num_kv_heads, head_dim;   /* four query heads per KV head, head_dim 64 or 128 */
    int32_t hidden_size, intermediate_size, vocab_size;
    int32_t kv_max_len, rope_positions;
    int32_t interleaved;                                   /* rotary pairs adjacent (1) or half a head apart (0) */
    float rms_norm_eps;
} mk_prefill_shape;

/* Positions a sequence's keys and values are padded to in the workspace (mk_prefill_rope, mk_prefill_attention). */
int mk_prefill_padded_seq(int seq);

/* h[row] = embed[ids[row]]; x[row] = rms_norm(h[row]) * norm_weight.  An id outside the vocabulary or a position outside
 * the rope tables or the cache (negative ones count from the end) aborts the kernel, as an index out of range does in
 * PyTorch. */
int mk_prefill_embed(const mk_prefill_shape *shape, const int64_t *ids, const int64_t *positions, const uint16_t *embed,
                     const uint16_t *norm_weight, uint16_t *h, uint16_t *x, void *stream);

/* h += y; x = rms_norm(h) * norm_weight */
int mk_prefill_add_norm(const mk_prefill_shape *shape, const uint16_t *y, const uint16_t *norm_weight, uint16_t *h,
                        uint16_t *x, void *stream);

/* Rotates the query and key heads of qkv [rows, (H + 2 KVH) D], appends keys and values to the layer's cache
 * [cache_batch, kv_max_len, KVH, D] and leaves q [rows, H D], keys [batch, KVH, padded, D] and transposed values
 * [batch, KVH, D, padded] for mk_prefill_attention. */
int mk_prefill_rope(const mk_prefill_shape *shape, const uint16_t *qkv, const int64_t *positions, const float *rope_cos,
                    const float *rope_sin, uint16_t *k_cache, uint16_t *v_cache, uint16_t *q, uint16_t *keys,
                    uint16_t *values_t, void *stream);

/* Causal attention of every sequence over its own keys: out [rows, H D]. */
int mk_prefill_attention(const mk_prefill_shape *shape, const uint16_t *q, const uint16_t *keys, const uint16_t *values_t,
                         uint16_t *out, void *stream);

/* out = silu(gate) * up, all [rows, intermediate_size] */
int mk_prefill_silu_mul(const mk_prefill_shape *shape, const uint16_t *gate, const uint16_t *up, uint16_t *out,
                        void *stream);

/* ids[row] = index of the first maximum of logits[row, 0..vocab_size), a NaN counting as the largest value */
int mk_prefill_argmax(const mk_prefill_shape *shape, const uint16_t *logits, int64_t *ids, void *stream);

/* The weights and the cache of a model; matrices are [out, in], stacked over the layers. */
typedef struct mk_prefill_model {
    const uint16_t *embed, *attn_norm, *qkv, *o, *mlp_norm, *gate, *up, *down, *final_norm, *head;
    const float *rope_cos, *rope_sin;
    uint16_t *k_cache, *v_cache;                           /* [layers, cache_batch, kv_max_len, KVH, D] */
    int32_t num_layers, cache_batch;
} mk_prefill_model;

/* The whole forward where batch * seq is not too large: matrix products included, all in kernels of this library.
 * h [rows, hidden_size] becomes the hidden states, out_ids [rows] the greedy ids.  The workspace's size is
 * mk_prefill_workspace_bytes.  0: not such a call - more than 4096 rows of a model up to 2048 wide; of a wider one fewer than 513 or
 * more than 1024 (3072 to 4096 wide: 2048, above 6144: fewer than 641); a hidden or intermediate size that is no multiple of 64.
 * (Of a model with an intermediate size above 2^20, a cache of 2^31 rows or more than 1024 KV heads: more than
 * 2^21 / hidden_size of more than 64 rows, or a hidden size above 2048.)  Negative: an error. */
int64_t mk_prefill_workspace_bytes(const mk_prefill_shape *shape);
int mk_prefill_forward(const mk_prefill_shape *shape, const mk_prefill_model *model, const int64_t *ids,
                            const int64_t *positions, uint16_t *h, uint16_t *workspace, int64_t *out_ids, void *stream);

/* How mk_prefill_forward of more than 64 rows tiles a product (0 qkv, 1 O, 2 gate and up, 3 down, 4 LM head): plan = index of
 * the kernel's shape, rows and columns of a tile, parts of K.  Host arithmetic only; what tests need to know that they reach
 * every kernel. */
int mk_prefill_tile_plan(const mk_prefill_shape *shape, int product, int32_t plan[4]);

/* Those calls of the above that run in wide tiles, alone: mk_prefill_forward, and its workspace and plans, of longer prompts and
 * wider models.  Workspace 0, or an error: not such a call - fewer than 257 rows, a hidden size below 256, or one in the brackets above. */
int64_t mk_prefill_wide_workspace_bytes(const mk_prefill_shape *shape);
int mk_prefill_wide_forward(const mk_prefill_shape *shape, const mk_prefill_model *model, const int64_t *ids,
                            const int64_t *positions, uint16_t *h, uint16_t *workspace, int64_t *out_ids, void *stream);
int mk_prefill_wide_plan(const mk_prefill_shape *shape, int product, int32_t plan[4]);

const char *mk_prefill_last_error(void);

#ifdef __cplusplus
}
#endif
#endif
