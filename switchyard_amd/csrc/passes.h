/* Entry points that the library offers its own Python host code (switchyard_amd/decoder.py) beside
 * the two public headers: pieces of whole passes of the decoder. Conventions as in
 * include/switchyard_moe.h: device pointers, sizes, a hipStream_t; SY_OK or an SY_ERR_* code with a
 * message in sy_last_error(); nothing is allocated and nothing waits. */
#pragma once

#include "../../include/switchyard_moe.h"

extern "C" {

/* T queries per sequence against the KV cache (a prompt, or further tokens behind what the cache
 * holds); replaces the scores / mask / softmax / value product of _attention()
 * (switchyard/model.py:78-84) for T >= 1.
 * q f16 [B*T, heads*D]: query t of sequence b sits at cache position first + t; kcache, vcache
 * f16 [B, kv_heads, capacity, D] hold the positions 0 .. first + T - 1; real uint8 [B, capacity]
 * marks real tokens. A query sees the real positions up to its own; one that would see none (left
 * padding) takes its own value -> out f16 [B*T, heads*D] (fp32 inside, probabilities rounded to
 * f16 for the value product). Query head h reads kv head h / (heads / kv_heads).
 * Limits: D is 64 or 128, first + T <= capacity, sy_prefill_attention_takes(). B == 0 is a no-op. */
SY_API int sy_prefill_attention(const void* q, const void* kcache, const void* vcache, const uint8_t* real, int first,
                                int B, int T, int heads, int kv_heads, int D, int capacity, void* out, void* stream);

/* Whether sy_prefill_attention takes this many positions (the tiles' masks are held in LDS: 786 432 positions
 * of 128, 1 048 576 of 64) of a cache of this capacity (a head's part under 2 GiB). */
SY_API int sy_prefill_attention_takes(int positions, int capacity, int D);

/* sy_decode_attention_qkv (include/switchyard_decode.h) with the keys of a (sequence, head) pair dealt to
 * four workgroups where the pairs are few and both buffers are given: parts f32 [B*heads, 16, D + 2] is
 * scratch of this call; tickets uint32 [B*heads] is zero before the launch and after it, and no two
 * launches that can run at the same time may share it. `out` has the bits of
 * sy_decode_attention_qkv's. */
SY_API int sy_decode_attention_qkv_split(const void* qkv, const void* q_norm, const void* k_norm, float eps, float clip,
                                         const void* cos_table, const void* sin_table, int max_positions,
                                         const int64_t* positions, const int64_t* slot, uint8_t* real, int B, int heads,
                                         int kv_heads, int D, int capacity, void* kcache, void* vcache, void* out,
                                         void* parts, void* tickets, void* stream);

/* For the rows of a batch of B prompts of T positions that starts a cache (tokens int64 [B*T], real uint8
 * [B*T]): twin int32 [B*T] names for each row one whose values are the same in every layer of a decoder with
 * causal attention over real positions. Rows of left padding (in front of their sequence's first real
 * token) that hold the token of the batch's first such row are twins of that row, which is its own
 * twin like every other row. */
SY_API int sy_padding_twins(const int64_t* tokens, const uint8_t* real, int B, int T, int32_t* twin, void* stream);

/* sy_moe_layer's result for h, added to the residual x, and the RMS norm of the sum: x_out [N, H] =
 * x + moe_layer(h) (may be x), h_out [N, H]. Expert outputs are computed once per twin: twin int32 [N] or
 * null; twin[t] is a row with the same values as t and is its own twin. Limits: H a multiple of 512,
 * at most 128 experts and top-8; the projections run on the MFMA tiles whatever L->mfma_tiles says. */
SY_API int sy_moe_add_rmsnorm(const SyMoeLayer* L, const void* h, const int32_t* twin, const void* x, const void* weight,
                              float eps, void* x_out, void* h_out, void* stream);

/* x f16 [rows, K] @ weight f16 [Nout, K]^T -> out f16 [rows, Nout] as one weight stream per 16 rows: the bits
 * of sy_grouped_gemv with one expert that owns every row. K a multiple of 8 up to 4096. */
SY_API int sy_dense_rows(const void* x, const void* weight, int rows, int Nout, int K, void* out, void* stream);

/* x f16 [rows, K] @ weight f16 [Nout, K]^T -> out f16 [rows, Nout] on small MFMA tiles, for a few dozen rows: K a
 * multiple of 128, each operand under 2 GiB, no more tiles than compute units (sy_dense_tiles_takes). 16-byte
 * aligned rows. */
SY_API int sy_dense_tiles(const void* x, const void* weight, int rows, int Nout, int K, void* out, void* stream);
SY_API int sy_dense_tiles_takes(int rows, int Nout, int K);

/* x f16 [rows, K] @ weight f16 [Nout, K]^T -> out f16 [rows, Nout] on the 256-row MFMA tile, K summed in order. count: int32
 * on the device or null; only rows 0 .. min(rows, *count) - 1 are read and written. K a multiple of 64 from 256 on;
 * each operand under 2 GiB (sy_dense_gemm_takes). */
SY_API int sy_dense_gemm_takes(int rows, int Nout, int K);
SY_API int sy_dense_gemm(const void* x, const void* weight, int rows, const int32_t* count, int Nout, int K, void* out,
                         void* stream);

/* Whether decode attention's (sequence, head) pairs are few enough for sy_decode_attention_qkv_split to
 * deal their keys to several workgroups. */
SY_API int sy_decode_attention_shares(int B, int heads);

/* What a prompt's pass says about its batch, in two launches (one without `pack`): T new tokens of B sequences at cache
 * positions first .. first + T - 1, real uint8 [B*T] (null: all) -> cache_real [B, capacity] at those positions,
 * positions int64 [B*T] (index among a sequence's real tokens, behind seen int64 [B]; not below 0), next int64 [B] =
 * seen + real tokens. pack int32 [2 B T + 3 B + 1] or null: place [B*T], map [B*T], last [B], count [1] and scratch.
 * Rows of left padding with the token of the batch's first such row (sy_padding_twins says which) exist once:
 * place[r] is position r's row among those that exist, in order, or ~row of the one that stands for it; map[i] is the
 * position of row i, last[b] the row of (b, T - 1), *count the number of rows. */
SY_API int sy_prompt_span(const int64_t* tokens, const uint8_t* real, int B, int T, int first, int capacity, const int64_t* seen,
                          uint8_t* cache_real, int64_t* positions, int64_t* next, int32_t* pack, void* stream);

/* A prompt's pass layer by layer, around projections that the caller makes: sy_prompt_embed (x = embedding rows, h =
 * their norm), then per layer sy_prompt_attention (qkv f16 [N, (heads + 2 kv_heads) D] -> out [N, heads D]; q is
 * scratch of that size) and sy_prompt_moe (o [N, H]: x += o, h = its norm, x += the MoE layer of h, xn = the next
 * norm). N = B * T rows; where count, map and place (sy_prompt_span) are given only the first *count rows exist, and
 * the others are neither read nor written. Up to SY_PROMPT_FEW_ROWS rows all of them exist, and the experts run on the
 * weight stream up to gemv_max_rows. Limits: sy_prefill_attention's, and sy_moe_add_rmsnorm's or, for few rows, those of a
 * decode step. */
#define SY_PROMPT_FEW_ROWS 64
typedef struct SyPrompt {
  int B, T, first, capacity, H, heads, kv_heads, D, k, norm, max_positions, gemv_max_rows;
  float eps, clip;
  const void *cos, *sin;
  const int64_t* positions;
  const uint8_t* real;
  const int32_t *place, *map, *count;
  void* scratch; /* sy_moe_layer_scratch_bytes of the largest layer */
  size_t scratch_bytes;
} SyPrompt;
typedef struct SyPromptLayer {
  int E, I;
  const void *q_norm, *k_norm, *mlp_norm, *router, *gate_up, *down, *next_norm;
  void *kcache, *vcache; /* [B, kv_heads, capacity, D] */
} SyPromptLayer;
SY_API int sy_prompt_embed(const SyPrompt* p, const int64_t* tokens, const void* embed, int vocab, const void* weight, void* x, void* h,
                           void* stream);
SY_API int sy_prompt_attention(const SyPrompt* p, const SyPromptLayer* L, const void* qkv, void* q, void* out, void* stream);
SY_API int sy_prompt_moe(const SyPrompt* p, const SyPromptLayer* L, const void* o, void* x, void* h, void* xn, void* stream);

/* One decode step of a model of `layers` layers for B <= SY_STEP_MAX_ROWS sequences: tok int64 [B] -> out f16
 * [B, vocab] (logits), the new keys and values written at *slot and real[:, *slot] set; the counters
 * stay where they are. All weights f16, nn.Linear layout. The experts run on the weight stream up to
 * gemv_max_rows sequences and on the MFMA tiles above. Scratch is the caller's
 * (sy_decode_step_scratch_bytes; 0 for a shape that is not taken), 256-byte aligned, and overwritten.
 * Limits: those of the launches (at most 128 experts, top-8, H and heads * D at most 4096). */
#define SY_STEP_MAX_ROWS 16
typedef struct SyDecodeLayer {
  const void *wqkv, *q_norm, *k_norm, *wo, *mlp_norm, *router, *gate_up, *down, *next_norm; /* next_norm: of the next layer, or the final one */
  void *kcache, *vcache; /* [B, kv_heads, capacity, D] */
} SyDecodeLayer;
typedef struct SyDecodeStep {
  int B, layers, H, heads, kv_heads, D, capacity, E, I, k, norm, vocab, embed_rows, max_positions, gemv_max_rows;
  float eps, clip;
  const void *embed, *first_norm, *lm_head, *cos, *sin;
  const int64_t *tok, *positions, *slot;
  uint8_t* real;
  void *out, *scratch;
  size_t scratch_bytes;
} SyDecodeStep;
SY_API size_t sy_decode_step_scratch_bytes(const SyDecodeStep* s);
SY_API int sy_decode_step(const SyDecodeStep* step, const SyDecodeLayer* layers, void* stream);

}  // extern "C"
