// One decode step of the whole model from one host call: the launches that Decoder.step_fused makes
// layer by layer (switchyard_amd/decoder.py), enqueued here back to back. There is no kernel in this
// file.
//
// Why: a step of one sequence is 114 launches of 3 to 16 us, and from Python each costs the host about
// 13 us (the checks, the allocation of its outputs, the marshalling): 1467 us to enqueue a step, now
// 527, and one sequence's step behind 700 positions takes 1134 us where it took 1299.
//
// What the launches are, per layer: q/k/v projection (a weight stream), attention with the q/k norm, the
// rotary embedding and the cache write in its prologue, output projection, residual add + norm + router
// logits + route + sort, gate/up, down, and combine + residual add + the next norm. Up to 64 choices
// (8 tokens of top-8) the gate/up stream sorts for itself, and routes too where it can, as in sy_moe_layer.
#include "common.h"
#include "../../include/switchyard_decode.h"
#include "passes.h"

namespace {

struct StepScratch {
  size_t x, xn, qkv, a, o, h, logits, idx, w, counts, offsets, token, wsorted, pos_of, act, y, parts, tickets, end;
};

StepScratch step_scratch(const SyDecodeStep& s) {
  StepScratch r;
  size_t at = 0;
  auto take = [&](size_t bytes) {
    const size_t here = at;
    at += (bytes + 255) / 256 * 256;
    return here;
  };
  const size_t B = s.B, M = B * s.k, qd = (size_t)s.heads * s.D, kvd = (size_t)s.kv_heads * s.D;
  r.x = take(B * s.H * 2);
  r.xn = take(B * s.H * 2);
  r.qkv = take(B * (qd + 2 * kvd) * 2);
  r.a = take(B * qd * 2);
  r.o = take(B * s.H * 2);
  r.h = take(B * s.H * 2);
  r.logits = take(B * s.E * 2);
  r.idx = take(M * 4);
  r.w = take(M * 2);
  r.counts = take((size_t)s.E * 4);
  r.offsets = take((size_t)(s.E + 1) * 4);
  r.token = take(M * 4);
  r.wsorted = take(M * 2);
  r.pos_of = take(M * 4);
  r.act = take(M * s.I * 2);
  r.y = take(M * s.H * 2);
  const bool shares = sy_decode_attention_shares(s.B, s.heads);
  r.parts = take(shares ? B * s.heads * 16 * (s.D + 2) * 4 : 0);
  r.tickets = take(shares ? B * s.heads * 4 : 0);
  r.end = at;
  return r;
}

int check_shape(const SyDecodeStep& s) {
  SY_REQUIRE(s.B >= 1 && s.B <= SY_STEP_MAX_ROWS, "decode_step: 1 <= B <= %d (got %d)", SY_STEP_MAX_ROWS, s.B);
  SY_REQUIRE(s.layers >= 0 && s.heads >= 1 && s.kv_heads >= 1 && s.D >= 1 && s.H >= 8 && s.I >= 8 && s.vocab >= 1,
             "decode_step: layers = %d, heads = %d, kv_heads = %d, D = %d, H = %d, I = %d, vocab = %d", s.layers, s.heads,
             s.kv_heads, s.D, s.H, s.I, s.vocab);
  SY_REQUIRE(s.E >= 1 && s.E <= 128 && s.k >= 1 && s.k <= 8 && s.k <= s.E, "decode_step: at most 128 experts and top-8 (got E = %d, k = %d)",
             s.E, s.k);
  return SY_OK;
}

}  // namespace

extern "C" SY_API size_t sy_decode_step_scratch_bytes(const SyDecodeStep* s) {
  return s && check_shape(*s) == SY_OK ? step_scratch(*s).end : 0;
}

extern "C" SY_API int sy_decode_step(const SyDecodeStep* step, const SyDecodeLayer* layers, void* stream) {
  SY_REQUIRE(step && layers, "decode_step: null pointer");
  const SyDecodeStep& s = *step;
  if (int rc = check_shape(s)) return rc;
  SY_REQUIRE(s.tok && s.embed && s.first_norm && s.lm_head && s.out && s.scratch, "decode_step: null pointer");
  const StepScratch at = step_scratch(s);
  SY_REQUIRE(s.scratch_bytes >= at.end && ((uintptr_t)s.scratch & 255) == 0,
             "decode_step: scratch of %zu bytes, 256-byte aligned, needed (%zu given)", at.end, s.scratch_bytes);
  char* b = (char*)s.scratch;
  void *x = b + at.x, *xn = b + at.xn, *qkv = b + at.qkv, *a = b + at.a, *o = b + at.o, *h = b + at.h, *logits = b + at.logits;
  void *w = b + at.w, *wsorted = b + at.wsorted, *act = b + at.act, *y = b + at.y;
  int32_t *idx = (int32_t*)(b + at.idx), *counts = (int32_t*)(b + at.counts), *offsets = (int32_t*)(b + at.offsets);
  int32_t *token = (int32_t*)(b + at.token), *pos_of = (int32_t*)(b + at.pos_of);
  const bool shares = sy_decode_attention_shares(s.B, s.heads);
  void *parts = shares ? b + at.parts : nullptr, *tickets = shares ? b + at.tickets : nullptr;
  const int B = s.B, H = s.H, I = s.I, E = s.E, k = s.k, qd = s.heads * s.D, kvd = s.kv_heads * s.D;
  const bool stream_experts = B <= s.gemv_max_rows;

  int rc = sy_embed_rmsnorm_step(s.tok, s.embed, s.embed_rows, s.first_norm, s.eps, B, H, x, xn, (unsigned*)tickets,
                                 shares ? B * s.heads : 0, stream);
  for (int i = 0; i < s.layers && !rc; ++i) {
    const SyDecodeLayer& L = layers[i];
    // one projection after another; the first that fails ends the step
    rc = sy_dense_rows(xn, L.wqkv, B, qd + 2 * kvd, H, qkv, stream);
    if (!rc)
      rc = sy_decode_attention_qkv_split(qkv, L.q_norm, L.k_norm, s.eps, s.clip, s.cos, s.sin, s.max_positions, s.positions,
                                         s.slot, s.real, B, s.heads, s.kv_heads, s.D, s.capacity, L.kcache, L.vcache, a, parts,
                                         tickets, stream);
    if (!rc) rc = sy_dense_rows(a, L.wo, B, H, qd, o, stream);
    if (rc) break;
    const SyFewRows few = {h, logits, w, wsorted, act, y, idx, counts, offsets, token, pos_of};
    rc = sy_few_rows_moe(x, o, L.mlp_norm, s.eps, L.router, B, H, I, E, k, s.norm, L.gate_up, L.down, L.next_norm, stream_experts, few, xn,
                         stream);
  }
  if (!rc) rc = sy_dense_rows(xn, s.lm_head, B, s.vocab, H, s.out, stream);
  return rc;
}
