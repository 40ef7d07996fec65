// A prompt's pass (Decoder.prefill_fused, switchyard_amd/decoder.py): what its launches need to know about the batch,
// and the launches of a layer's two halves, enqueued from one host call each.
//
// The rows of a batch of left-padded prompts. A row in front of its sequence's first real token holds the same numbers
// in every layer as any other such row with the same token (decode.hip, padding_twins_kernel, says why), so a pass
// needs one of them only. prompt_span and prompt_pack number the rows that exist, in their order in the batch:
//   place[r]  of position r = b T + t: its row, or ~row where the position is padding whose row another position holds
//   map[i]    the position of row i
//   count     how many rows there are
// and every launch of the pass works on `count` rows, which only the device knows: its grid is for all B T, and the
// workgroups without rows leave at once. 8 prompts of 256 to 512 tokens: about 3200 rows for 4096, and a layer's combine + norm
// 32.0 -> 29.1 us, add + norm 13.2 -> 11.2; 3 of 1000 to 2000: 44.1 -> 40.6, 18.3 -> 15.7. The projections follow the count only where
// the caller knows that there is enough padding (PACKED_GEMM_MAX_REAL in decoder.py).
//
// The host: mask, positions and counters were fourteen launches of PyTorch's (65 us) in front of the first layer, now two,
// and a layer five calls beside its projections, now two: 128 tokens in 2489 us, now 2369.
#include "common.h"
#include "passes.h"
#include "../../include/switchyard_decode.h"

namespace {

constexpr int SPAN_THREADS = 256, SPAN_WAVES = SPAN_THREADS / WAVE;

// Inclusive count of `flag` over the workgroup's threads in order; `total` is the count over all of them.
__device__ __forceinline__ int block_count(bool flag, int* lds, int& total) {
  const uint64_t m = __ballot(flag);
  const int wave = threadIdx.x >> 6;
  __syncthreads();   // the counts before have been read
  if ((threadIdx.x & 63) == 0) lds[wave] = __popcll(m);
  __syncthreads();
  int before = 0;
  total = 0;
#pragma unroll
  for (int w = 0; w < SPAN_WAVES; ++w) {
    before += w < wave ? lds[w] : 0;
    total += lds[w];
  }
  return before + __popcll(m & lanemask_lt()) + (flag ? 1 : 0);
}

// One workgroup per sequence: its part of the cache's mask, its tokens' rotary positions (the index among the
// sequence's real tokens, behind the `seen` it already holds), the position after them, and, for prompt_pack, the
// first real token, and how many of its rows exist: not those of padding whose token is that of the batch's
// first row of padding, except that row itself.
__global__ void __launch_bounds__(SPAN_THREADS)
prompt_span_kernel(const int64_t* __restrict__ tokens, const uint8_t* __restrict__ real, int B, int T, int first, int capacity,
                   const int64_t* __restrict__ seen, uint8_t* __restrict__ cache_real, int64_t* __restrict__ positions,
                   int64_t* __restrict__ next, int* __restrict__ first_real, int* __restrict__ rows) {
  __shared__ int lds[SPAN_WAVES], s_pad, s_first, s_gone;
  const int b = blockIdx.x, tid = threadIdx.x;
  if (tid == 0) {
    s_pad = B;     // the first sequence that starts with padding
    s_first = T;   // this sequence's first real token
    s_gone = 0;    // rows of this sequence that do not exist
  }
  int run = 0;
  const long before = (long)seen[b];
  for (int t0 = 0; t0 < T; t0 += SPAN_THREADS) {
    const int t = t0 + tid;
    const bool is = t < T && (!real || real[(size_t)b * T + t] != 0);
    int total;
    const int order = run + block_count(is, lds, total);
    run += total;
    if (t < T) {
      const long at = before + order - 1;
      positions[(size_t)b * T + t] = at < 0 ? 0 : at;
      cache_real[(size_t)b * capacity + first + t] = is;
      if (is) atomicMin(&s_first, t);
    }
  }
  if (tid == 0) next[b] = before + run;
  if (!rows) return;
  for (int r = tid; r < B; r += SPAN_THREADS)
    if (!real[(size_t)r * T]) {
      atomicMin(&s_pad, r);
      break;
    }
  __syncthreads();
  const int lead = s_first;
  if (s_pad < B) {
    const int64_t pad = tokens[(size_t)s_pad * T];
    for (int t = tid; t < lead; t += SPAN_THREADS)
      if (tokens[(size_t)b * T + t] == pad && !(b == s_pad && t == 0)) atomicAdd(&s_gone, 1);
  }
  __syncthreads();
  if (tid == 0) {
    first_real[b] = lead;
    rows[b] = T - s_gone;
  }
}

__global__ void __launch_bounds__(SPAN_THREADS)
prompt_pack_kernel(const int64_t* __restrict__ tokens, const uint8_t* __restrict__ real, int B, int T,
                   const int* __restrict__ first_real, const int* __restrict__ rows, int* __restrict__ place,
                   int* __restrict__ map, int* __restrict__ last, int* __restrict__ count) {
  __shared__ int lds[SPAN_WAVES], s_pad, s_base, s_pad_base;
  const int b = blockIdx.x, tid = threadIdx.x;
  if (tid == 0) {
    s_pad = B;
    s_base = 0;       // rows of the sequences before this one
    s_pad_base = 0;   // and of those before the one with the batch's first padding
  }
  __syncthreads();
  for (int r = tid; r < B; r += SPAN_THREADS)
    if (!real[(size_t)r * T]) {
      atomicMin(&s_pad, r);
      break;
    }
  __syncthreads();
  const int pad_b = s_pad;
  for (int r = tid; r < B; r += SPAN_THREADS) {
    if (r < b) atomicAdd(&s_base, rows[r]);
    if (r < pad_b) atomicAdd(&s_pad_base, rows[r]);
  }
  __syncthreads();
  const int base = s_base, pad_row = s_pad_base, lead = first_real[b];
  const int64_t pad = pad_b < B ? tokens[(size_t)pad_b * T] : 0;
  int run = 0;
  for (int t0 = 0; t0 < T; t0 += SPAN_THREADS) {
    const int t = t0 + tid, r = b * T + t;
    const bool gone = t < lead && pad_b < B && tokens[r] == pad && !(b == pad_b && t == 0);
    const bool is = t < T && !gone;
    int total;
    const int row = base + run + block_count(is, lds, total) - 1;
    run += total;
    if (t < T) place[r] = is ? row : ~pad_row;
    if (is) map[row] = r;
    if (t == T - 1) last[b] = is ? row : pad_row;
  }
  if (b == B - 1 && tid == 0) *count = base + run;
}

}  // namespace

extern "C" SY_API int sy_prompt_span(const int64_t* tokens, const uint8_t* real, int B, int T, int first, int capacity,
                                     const int64_t* seen, uint8_t* cache_real, int64_t* positions, int64_t* next, int32_t* pack,
                                     void* stream) {
  SY_REQUIRE(B >= 0 && T >= 1 && (long)B * T < (1l << 30), "prompt_span: B = %d, T = %d", B, T);
  SY_REQUIRE(first >= 0 && (long)first + T <= capacity, "prompt_span: positions %d .. %ld of %d", first, (long)first + T - 1, capacity);
  if (B == 0) return SY_OK;
  SY_REQUIRE(seen && cache_real && positions && next, "prompt_span: null pointer");
  SY_REQUIRE(!pack || (tokens && real), "prompt_span: rows are packed by their tokens and mask");
  const size_t N = (size_t)B * T;
  int32_t *place = pack, *map = pack ? pack + N : nullptr, *last = pack ? map + N : nullptr, *count = pack ? last + B : nullptr;
  int32_t *first_real = pack ? count + 1 : nullptr, *rows = pack ? first_real + B : nullptr;
  prompt_span_kernel<<<B, SPAN_THREADS, 0, (hipStream_t)stream>>>(tokens, real, B, T, first, capacity, seen, cache_real, positions, next,
                                                                  first_real, rows);
  int rc = sy_check_launch("prompt_span");
  if (rc || !pack) return rc;
  prompt_pack_kernel<<<B, SPAN_THREADS, 0, (hipStream_t)stream>>>(tokens, real, B, T, first_real, rows, place, map, last, count);
  return sy_check_launch("prompt_pack");
}

extern "C" SY_API int sy_prompt_embed(const SyPrompt* p, const int64_t* tokens, const void* embed, int vocab, const void* weight, void* x,
                                      void* h, void* stream) {
  SY_REQUIRE(p, "prompt_embed: null pointer");
  const int N = p->B * p->T;
  return p->count ? sy_embed_rmsnorm_packed(tokens, p->map, p->count, embed, vocab, weight, p->eps, N, p->H, x, h, stream)
                  : sy_embed_rmsnorm(tokens, embed, vocab, weight, p->eps, N, p->H, x, h, stream);
}

// The first half of a layer behind its projection: q/k norm, rotary embedding and cache write, then attention.
extern "C" SY_API int sy_prompt_attention(const SyPrompt* p, const SyPromptLayer* L, const void* qkv, void* q, void* out, void* stream) {
  SY_REQUIRE(p && L, "prompt_attention: null pointer");
  int rc = sy_qk_norm_rope_prompt(qkv, L->q_norm, L->k_norm, p->eps, p->clip, p->cos, p->sin, p->max_positions, p->positions, p->first,
                                  p->place, p->B, p->T, p->heads, p->kv_heads, p->D, p->capacity, q, L->kcache, L->vcache, stream);
  if (rc) return rc;
  return sy_prefill_attention_rows(q, L->kcache, L->vcache, p->real, p->first, p->B, p->T, p->heads, p->kv_heads, p->D, p->capacity,
                                   p->place, out, stream);
}

// The second half behind the output projection o: add and norm, the MoE layer, add and the next norm.
extern "C" SY_API int sy_prompt_moe(const SyPrompt* p, const SyPromptLayer* L, const void* o, void* x, void* h, void* xn, void* stream) {
  SY_REQUIRE(p && L, "prompt_moe: null pointer");
  const int N = p->B * p->T;
  SyMoeLayer moe = {N, L->E, p->k, p->norm, p->H, L->I, 1, 0, L->router, L->gate_up, L->down, p->scratch, p->scratch_bytes};
  if (N <= SY_PROMPT_FEW_ROWS) {
    // a short prompt is as many rows as a step of many sequences, and goes through its launches: norm, router, route and sort
    // are one where they were four (one prompt of 32 tokens, beside the projections: 22.7 -> 11 us a layer)
    SY_REQUIRE(!p->count, "prompt_moe: %d rows are not packed", N);
    moe.mfma_tiles = N > p->gemv_max_rows;
    return sy_few_rows_moe_layer(&moe, (void*)x, o, L->mlp_norm, p->eps, L->next_norm, h, xn, stream);
  }
  const int rc = sy_add_rmsnorm_counted(x, o, L->mlp_norm, p->eps, N, p->count, p->H, x, h, stream);
  if (rc) return rc;
  return sy_moe_add_rmsnorm_rows(&moe, h, nullptr, p->count, x, L->next_norm, p->eps, x, xn, stream);
}
