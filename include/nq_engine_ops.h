/* C ABI of libawq_hip.so, part 2 -- the kernels of a Qwen3 decode step that sit between the AWQ
 * linears (include/awq_hip.h): residual add + RMSNorm, per-head q/k RMSNorm + rotary + KV-cache
 * write, attention of one new token per sequence over a paged KV cache, SiLU(gate) * up.
 *
 * Conventions are those of awq_hip.h: device pointers, dense row-major tensors, `dtype` is AWQ_F16
 * or AWQ_BF16 for every 16-bit tensor of a call, `stream` is a hipStream_t as void*, the return
 * value is an awq_status and awq_hip_last_error() holds the message of a failure.
 *
 * The reference runs these steps as torch modules inside its model (no kernels, no KV cache);
 * citations name the module code whose arithmetic each entry point reproduces.
 */
#ifndef NQ_ENGINE_OPS_H_
#define NQ_ENGINE_OPS_H_

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* residual [rows, hidden] += delta (skipped when delta is NULL; the sum is rounded to dtype as
 * `x + sublayer(x)` is), then y = dtype(residual_f32 * rsqrt(mean(residual_f32^2) + eps)) * weight.
 * hidden % 8 == 0, hidden <= 8192.
 * RMSNorm.rms_norm, nanoquantization/layers/norm.py:18-32; the residual adds of
 * Qwen3QuantizedBlock.forward, nanoquantization/models/qwen3_quantized.py:194-215. */
int nq_add_rmsnorm(void* residual, const void* delta, const void* weight, void* y, int64_t rows,
                   int64_t hidden, float eps, int dtype, void* stream);

/* ssq [ceil(hidden / 128)][rows] (fp32): ssq[t][r] = sum of squares of x[r, 128 t .. 128 t + 127], in the summation
 * order of nq_add_rmsnorm.  The RMSNorm statistics that awq_gemv_rmsnorm (include/awq_hip.h) reads, for a residual
 * stream that no awq_gemv_add_residual has produced (the embedding output of a decode step).  hidden % 8 == 0,
 * hidden <= 8192.  The mean of squares of RMSNorm.rms_norm, nanoquantization/layers/norm.py:18-32. */
int nq_row_ssq(const void* x, float* ssq, int64_t rows, int64_t hidden, int dtype, void* stream);
/* The same with the embedding lookup in front: x_out[r] = table[ids[r]] (ids clamped to [0, table_rows)), ssq of x_out.
 * Qwen3QuantizedModel.forward's embed_tokens, nanoquantization/models/qwen3_quantized.py:259-273. */
int nq_embed_row_ssq(const int64_t* ids, const void* table, void* x_out, float* ssq, int64_t rows, int64_t hidden,
                     int64_t table_rows, int dtype, void* stream);

/* qkv [rows, (num_heads + 2*num_kv_heads) * head_dim] is the output of the q|k|v projections
 * side by side.  Every q and k head is RMS-normalised (q_weight / k_weight, [head_dim]) and rotated
 * (half-split rotary, angle table cos_sin f32 [max_positions, head_dim] = cos | sin) at
 * positions[row]; q goes to q_out [rows, num_heads, head_dim], k and the untouched v go to
 * k_cache / v_cache [num_slots / block_size, num_kv_heads, block_size, head_dim] (a head's tokens of one
 * block are contiguous) at slot slots[row] = block * block_size + offset (a row whose slot is outside
 * [0, num_slots) writes no k/v).  If k_out is not NULL the normalised, rotated k heads are also written
 * densely to k_out [rows, num_kv_heads, head_dim] (what a causal prefill attention over the same rows
 * reads).  head_dim even, <= 256.
 * Qwen3QuantizedAttention.forward, nanoquantization/models/qwen3_quantized.py:79-93;
 * RoPE.apply_rope / forward, nanoquantization/layers/rope.py:24-45. */
int nq_qk_norm_rope_store(const void* qkv, const void* q_weight, const void* k_weight,
                          const float* cos_sin, const int64_t* positions, const int64_t* slots,
                          void* q_out, void* k_out, void* k_cache, void* v_cache, int64_t rows, int64_t num_heads,
                          int64_t num_kv_heads, int64_t head_dim, int64_t max_positions,
                          int64_t num_slots, int64_t block_size, float eps, int dtype, void* stream);

/* Bytes of device workspace nq_paged_attention_decode needs (0 is possible); no initialisation
 * needed.  max_context = block_size * max_blocks_per_seq. */
size_t nq_paged_attention_workspace_bytes(int64_t batch, int64_t num_heads, int64_t num_kv_heads,
                                          int64_t head_dim, int64_t max_context);

/* out[b, h, :] = softmax(scale * q[b, h, :] . K_b^T) V_b over the first context_lens[b] tokens of
 * sequence b (the new token's k/v already written).  Token t of sequence b is token t % block_size
 * of block block_table[b, t / block_size] in k_cache / v_cache
 * [num_blocks, num_kv_heads, block_size, head_dim]; query head h reads kv head
 * h / (num_heads / num_kv_heads).  q, out: [batch, num_heads, head_dim].  head_dim 64 or 128,
 * num_heads / num_kv_heads in {1, 2, 4, 8} -- with head_dim 128 and block_size % 16 == 0 any ratio up to 16 (Qwen3-14B
 * has 5); block indices are clamped to the cache.
 * F.scaled_dot_product_attention(..., enable_gqa) of Qwen3QuantizedAttention.forward,
 * nanoquantization/models/qwen3_quantized.py:94-99, restricted to the last query position. */
int nq_paged_attention_decode(const void* q, const void* k_cache, const void* v_cache,
                              const int32_t* block_table, const int32_t* context_lens, void* out,
                              int64_t batch, int64_t num_heads, int64_t num_kv_heads,
                              int64_t head_dim, int64_t block_size, int64_t max_blocks_per_seq,
                              int64_t num_blocks, float scale, int dtype, void* workspace,
                              size_t workspace_bytes, void* stream);

/* out[r, i] = dtype(SiLU(gate_up[r, i])) * gate_up[r, inter + i]; gate_up [rows, 2*inter] is the
 * output of the gate|up projections side by side, out [rows, inter].  inter % 8 == 0.
 * Qwen3QuantizedMLP.forward, nanoquantization/models/qwen3_quantized.py:147-152. */
int nq_silu_mul(const void* gate_up, void* out, int64_t rows, int64_t inter, int dtype, void* stream);

/* The same for gate|up interleaved in words of 8 columns (word 2t = gate outputs 8t..8t+7, word 2t+1 = the up
 * columns of the same outputs): the output layout of a plain product with the interleaved buffers of
 * awq_gemv_swiglu (include/awq_hip.h). */
int nq_silu_mul_interleaved(const void* gate_up, void* out, int64_t rows, int64_t inter, int dtype, void* stream);

/* The same for gate and up [rows, inter] as two tensors, the outputs of the projections one by one. */
int nq_silu_mul_pair(const void* gate, const void* up, void* out, int64_t rows, int64_t inter, int dtype,
                     void* stream);

/* q [batch * tokens, num_heads * head_dim], k and v [.., num_kv_heads * head_dim]: outputs of the separate projections.
 * q and k heads are normalised and rotated as by nq_qk_norm_rope_store, at positions[sequence][token] (per_sequence) or
 * positions[token]; a negative position counts from the end of the table,
 * and one outside the table gives NaN (the module refuses such positions before the call).  q_out keeps q's layout, k_out and v_out are
 * [batch, num_kv_heads, tokens, head_dim].  head_dim 64, 128 or 256. */
int nq_qkv_norm_rope(const void* q, const void* k, const void* v, const void* q_weight, const void* k_weight,
                     const float* cos_sin, const int64_t* positions, int per_sequence, void* q_out, void* k_out,
                     void* v_out, int64_t batch, int64_t tokens, int64_t num_heads, int64_t num_kv_heads,
                     int64_t head_dim, int64_t max_positions, float q_eps, float k_eps, int dtype, void* stream);

/* out[r] = argmax_i logits[r, i] as int64, the lowest index among equal maxima (NaNs are never selected);
 * logits [rows, vocab] dense.  Greedy sampling for the engine's decode loop; the reference has no generation
 * loop, the logits are those of Qwen3QuantizedForCausalLM.forward
 * (nanoquantization/models/qwen3_quantized.py:312-314). */
int nq_argmax_rows(const void* logits, int64_t* out, int64_t rows, int64_t vocab, int dtype, void* stream);

/* Bookkeeping of a decode step over the paged cache (the reference has no generation loop; one launch each instead of
 * a dozen elementwise ones).  `active` is one byte per row (torch.bool).
 * nq_decode_prepare: slots[r] = active[r] ? block_table[r][positions[r] / block_size] * block_size +
 *   positions[r] % block_size : -1 (the slot convention of nq_qk_norm_rope_store), context_lens[r] = positions[r] + 1.
 * nq_decode_advance: out_log[step[0]][r] = next_tokens[r] (skipped when step[0] is outside [0, out_rows)),
 *   ids[r] = next_tokens[r], positions[r] += active[r], step[0] += 1. */
int nq_decode_prepare(const int64_t* positions, const uint8_t* active, const int32_t* block_table, int64_t* slots,
                      int32_t* context_lens, int64_t rows, int64_t max_blocks, int64_t block_size, void* stream);
int nq_decode_advance(const int64_t* next_tokens, const uint8_t* active, int64_t* out_log, int64_t* ids,
                      int64_t* positions, int64_t* step, int64_t rows, int64_t out_rows, void* stream);

/* nq_paged_attention_decode with `out` in the input layout of nq_block_step: [ceil(batch / 16) * 16 rows], pieces of 16 rows x 32
 * columns in the order of the matrix instruction's operand (rows past the batch are not written).  head_dim 128, one or two query
 * heads per kv head.  Reference code as above. */
int nq_paged_attention_decode_tiled(const void* q, const void* k_cache, const void* v_cache,
                                    const int32_t* block_table, const int32_t* context_lens, void* out,
                                    int64_t batch, int64_t num_heads, int64_t num_kv_heads,
                                    int64_t head_dim, int64_t block_size, int64_t max_blocks_per_seq,
                                    int64_t num_blocks, float scale, int dtype, void* workspace,
                                    size_t workspace_bytes, void* stream);

/* A packed weight (qweight [K, N / 8], qscales [K / group_size, N], qzeros, as in awq_hip.h) laid out for nq_block_step:
 * per 16 columns and 128 rows one piece of 1 KiB in the order of the matrix instruction's operand, then per column of every
 * piece its scale and zero point.  N % 16 == 0, K % 128 == 0, group_size % 128 == 0. */
size_t nq_tiled_weight_bytes(int64_t N, int64_t K);
int nq_tile_weight(const int32_t* qweight, const void* qscales, const int32_t* qzeros, void* out, int64_t N, int64_t K,
                   int64_t group_size, int dtype, void* stream);

/* The linears between two attentions of a decode step, in one launch (bf16):
 *   res_mid = res_in + o_proj(attn);  act = SiLU(gate) * up of RMSNorm(res_mid) * norm_mid;  res_out = res_mid + down_proj(act);
 *   and, with qkv, the next layer's q|k|v of RMSNorm(res_out) * norm_next with q/k norm, rotary and cache write, as
 *   awq_gemv_rmsnorm_qkv_rope_store (awq_hip.h) does it.
 * Without qkv (the last layer) that part is left out; norm_next and what follows it may be NULL then.
 * The weights are nq_tile_weight's: o [hidden, heads * 128], gate_up [2 * inter, hidden] with gate and up interleaved by words,
 * down [hidden, inter], qkv [(heads + 2 * kv_heads) * 128, hidden] as [N, K].  res_in, res_out: [rows, hidden]; attn (of heads * 128 columns),
 * act (inter), tiled_mid and tiled_out (res_mid and res_out, hidden) have nq_paged_attention_decode_tiled's layout; squares_mid and squares_out are
 * fp32 [ceil(rows / 16)][hidden / 128][16 rows][16 sums of eight columns' squares].  The result's bits are those of the launches one by one with K cut as awq_gemv_add_residual and
 * awq_gemv_rmsnorm cut it at these sizes (hidden 2048: at 5 to 16 rows).  Rows past `rows` of attn must be numbers.
 * `done`: nq_block_step_flag_words() words that are zero when the launch begins, of its own while it runs; `clear`: as many words of another launch
 * that is over, which this one sets to zero (the launches of a step clear each other's in a ring).  Every buffer is of its own,
 * 16-byte aligned, and attn, res_out, act, q_out, the tiled residuals, the squares, done and clear begin on a line of 128 bytes.
 * next: up to four regions that the launch after this one reads (NULL: none); workgroups that are idle in the last phase bring them near.
 * The launch's workgroups hand rows to each other and wait for each other; one that has looked `spin` times in vain does what is missing
 * itself, so that the launch ends whatever part of it runs at a time.  The sums are in a fixed order: results repeat exactly.
 * rows 1..64, sizes that nq_block_step_supported names (with the head ratios of nq_paged_attention_decode_tiled, which writes attn).
 * Qwen3QuantizedBlock.forward, nanoquantization/models/qwen3_quantized.py:194-215 (and :79-93, :147-152), restricted to one token. */
typedef struct nq_block_step_args {
    const void *o, *gate_up, *down, *qkv;
    const void *attn, *res_in, *norm_mid, *norm_next;
    void *res_out, *tiled_mid, *tiled_out, *act;
    float *squares_mid, *squares_out;
    uint32_t *done, *clear;
    const void *q_weight, *k_weight;
    const float* cos_sin;
    const int64_t *positions, *slots;
    void *q_out, *k_cache, *v_cache;
    int64_t rows, hidden, inter, heads, kv_heads, max_positions, num_slots, block_size, spin;
    const void* next[4];
    size_t next_bytes[4];
    float eps, head_eps;
} nq_block_step_args;
size_t nq_block_step_supported(int64_t rows, int64_t hidden, int64_t inter, int64_t heads, int64_t kv_heads);
size_t nq_block_step_flag_words(void);
int nq_block_step(const nq_block_step_args* args, void* stream);

#ifdef __cplusplus
}
#endif
#endif /* NQ_ENGINE_OPS_H_ */
