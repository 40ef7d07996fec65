"""The work whose speed this repository is judged by: single mixture-of-experts layers from one token
to thousands, and the passes of the decoder around them (one decode step of a batch, one prompt).

Everything has the OLMoE-1B-7B shape (`decoder.OLMOE_1B_7B`: 16 layers, hidden 2048, 64 experts of
width 1024, top-8, 16 heads of 128, vocabulary 50304) in fp16, random-initialised, as bench.py and
the tests have it.

  layer    `kernels.moe_layer`: the model hook's body, called from somebody's own decoder
  step     `Decoder.step_fused`: every sequence of a batch advances by one token
  prefill  `Decoder.prefill_fused` into a new `KVCache`: a batch of left-padded prompts
"""

import math

import torch

from switchyard_amd import decoder, kernels

SHAPE = decoder.OLMOE_1B_7B
H, I, E, K = SHAPE.hidden, SHAPE.intermediate, SHAPE.experts, SHAPE.top_k
QKV = (SHAPE.heads + 2 * SHAPE.kv_heads) * SHAPE.head_dim
NEW_TOKENS = 32        # room a prompt's cache has for the tokens that will be generated
MOST_TOKENS = 6144     # of one prefill pass


def listed():
    return [
        # one token of one sequence: the shortest path through the layer, all latency
        dict(name="layer_1", kind="layer", tokens=1, skew=0.0, norm=False),
        # the decode batch that the layer's headline figure is quoted on
        dict(name="layer_8", kind="layer", tokens=8, skew=0.0, norm=False),
        # a batch of sequences that is no round number, with normalised router weights
        dict(name="layer_37", kind="layer", tokens=37, skew=0.0, norm=True),
        # a chunk of one prompt whose tokens favour some experts (a trained router's load is uneven)
        dict(name="layer_333_skewed", kind="layer", tokens=333, skew=1.0, norm=False),
        # a prompt of a thousand tokens, or a chunk of that size: bound by the weights still
        dict(name="layer_1024", kind="layer", tokens=1024, skew=0.0, norm=False),
        # a batch of prompts: bound by the matrix cores
        dict(name="layer_4096", kind="layer", tokens=4096, skew=0.0, norm=False),
        # one user's next token behind a conversation of some length
        dict(name="step_1", kind="step", batch=1, past=700),
        # a small serving batch behind prompts of up to 512 tokens
        dict(name="step_8", kind="step", batch=8, past=512),
        # a full serving batch, half-way through its generation
        dict(name="step_64", kind="step", batch=64, past=576),
        # one user's prompt (time to the first token)
        dict(name="prefill_1x437", kind="prefill", batch=1, length=437),
        # a serving batch's prompts
        dict(name="prefill_8x512", kind="prefill", batch=8, length=512),
        # a few long documents of different lengths
        dict(name="prefill_3x2000", kind="prefill", batch=3, length=2000),
    ]


def _between(rng, low, high):
    """A whole number whose logarithm is uniform."""
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high + 1))))))


def draw(rng):
    kind = rng.choice(["layer", "layer", "step", "prefill"])
    if kind == "layer":
        return dict(kind=kind, tokens=_between(rng, 1, 4096), skew=rng.choice([0.0, 0.0, 1.0]), norm=rng.random() < 0.3)
    if kind == "step":
        return dict(kind=kind, batch=_between(rng, 1, 64), past=_between(rng, 16, 1000))
    length = _between(rng, 16, 2000)
    return dict(kind=kind, batch=_between(rng, 1, min(16, MOST_TOKENS // length)), length=length)


def _lengths(batch, longest, gen):
    """How many real tokens each row of a left-padded batch has: one row fills it, the others at least half."""
    n = torch.randint(longest // 2, longest + 1, (batch,), generator=gen, device="cuda")
    n[0] = longest
    return n


def _real(lengths, width):
    return torch.arange(width, device="cuda")[None, :] >= (width - lengths)[:, None]


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*dims, std=1.0):
        return (torch.randn(*dims, generator=gen, device="cuda", dtype=torch.float32) * std).half()

    if case["kind"] == "layer":
        # the recipe of the benchmark and of the tests: unit rows, weights of 0.02. A skewed router
        # adds to each expert's logits a bias that falls with the expert's rank (Zipf, exponent 1.1),
        # carried by one constant feature of the rows, as a trained router's uneven load is.
        h = normal(case["tokens"], H)
        router = normal(E, H, std=0.02)
        if case["skew"]:
            rank = torch.randperm(E, generator=gen, device="cuda") + 1
            h[:, 0] = 1.0
            router[:, 0] = (-1.1 * case["skew"] * torch.log(rank.float())).half()
        return dict(kind="layer", h=h, router=router, gate_up=normal(E, 2 * I, H, std=0.02),
                    down=normal(E, H, I, std=0.02), norm=case["norm"])

    model = decoder.Decoder(SHAPE, decoder.random_weights(SHAPE, seed=seed))
    batch = case["batch"]
    if case["kind"] == "prefill":
        length = case["length"]
        tokens = torch.randint(SHAPE.vocab, (batch, length), generator=gen, device="cuda")
        real = _real(_lengths(batch, length, gen), length)
        return dict(kind="prefill", model=model, tokens=tokens * real, real=real, capacity=length + NEW_TOKENS)

    # the cache as the prompt left it: normalised keys, values of the projection's size
    past = case["past"]
    cache = decoder.KVCache(SHAPE, batch, past + NEW_TOKENS, torch.float16, "cuda")
    lengths = _lengths(batch, past, gen)
    for layer in range(SHAPE.layers):
        cache.k[layer, :, :, :past] = normal(batch, SHAPE.kv_heads, past, SHAPE.head_dim)
        cache.v[layer, :, :, :past] = normal(batch, SHAPE.kv_heads, past, SHAPE.head_dim, std=0.9)
    cache.real[:, :past] = _real(lengths, past)
    cache.next_position.copy_(lengths)
    cache.filled = past
    tok = torch.randint(SHAPE.vocab, (batch, 1), generator=gen, device="cuda")
    return dict(kind="step", model=model, tok=tok, cache=cache, slot=torch.tensor([past], device="cuda"))


@torch.no_grad()
def run(state):
    if state["kind"] == "layer":
        return kernels.moe_layer(state["h"], state["router"], state["gate_up"], state["down"], K, state["norm"])
    model = state["model"]
    if state["kind"] == "prefill":
        # a new conversation: its cache is part of the pass, as in Decoder.generate
        tokens = state["tokens"]
        cache = decoder.KVCache(SHAPE, tokens.shape[0], state["capacity"], torch.float16, tokens.device)
        logits = model.prefill_fused(tokens, cache, state["real"])
        return dict(logits=logits, keys=cache.k, values=cache.v)
    # the counters stay where they are (Decoder.generate moves them with the arg-max, afterwards),
    # so the same step can be taken again
    cache = state["cache"]
    logits = model.step_fused(state["tok"], cache, state["slot"], advance=False)
    return dict(logits=logits, keys=cache.k, values=cache.v, real=cache.real)


def _experts_used(tokens):
    return E * (1.0 - (1.0 - K / E) ** tokens)


def _layer_work(tokens):
    weights = 2 * (_experts_used(tokens) * 3 * H * I + E * H)
    return weights, tokens * (K * 6 * H * I + 2 * E * H)


def work(case):
    if case["kind"] == "layer":
        weights, flops = _layer_work(case["tokens"])
        return dict(bytes=weights + 2 * 2 * case["tokens"] * H, flops=flops)
    batch = case["batch"]
    attention_weights = 2 * (QKV * H + SHAPE.heads * SHAPE.head_dim * H)
    key_bytes = 2 * 2 * SHAPE.kv_heads * SHAPE.head_dim      # of one position of one layer
    longest = case["past" if case["kind"] == "step" else "length"]
    real = longest * (1 + 0.75 * (batch - 1))                # real tokens: the other rows' mean length is 0.75
    if case["kind"] == "step":
        tokens, pairs = batch, real + batch                  # pairs of a query and a key that it sees
        cache_bytes = (real + batch) * key_bytes             # read, and the new position written
    else:
        tokens, pairs = real, longest ** 2 / 2 * (1 + 7 / 12 * (batch - 1))
        cache_bytes = real * key_bytes                       # written
    weights, flops = _layer_work(tokens)
    return dict(bytes=SHAPE.layers * (weights + attention_weights + cache_bytes) + 2 * SHAPE.vocab * H
                + 2 * 2 * tokens * H + 2 * batch * SHAPE.vocab,
                flops=SHAPE.layers * (flops + 2 * tokens * H * (QKV + SHAPE.heads * SHAPE.head_dim)
                                      + 4 * pairs * SHAPE.heads * SHAPE.head_dim) + 2 * batch * SHAPE.vocab * H)


def tolerance(case):
    """About four times what correct implementations at this precision were seen to differ by."""
    if case["kind"] == "layer":
        # against the layer in fp32 from the same fp16 logits: rel 6.0e-4 to 6.5e-4 from 1 to 4096 tokens
        # (the two projection kernels against each other: 1e-4)
        return {"rel": 0.003, "max": 0.05}
    if case["kind"] == "step":
        # against the step in PyTorch operators: logits rel 0.0044 (1 sequence) and 0.013 (8), max 0.15. Where
        # two experts are nearly tied, a rounding decides which one a token takes, and 16 layers
        # carry it on; the caches differ in one position only (rel 1e-4)
        return {"rel": 0.03, "max": 0.6}
    # against the prompt in PyTorch operators: keys and values rel 0.0017 (437 tokens) and 0.0024 (3 x
    # 1000), max 0.17 and 0.87 at a token that takes another expert for the same reason
    return {"rel": 0.01, "max": 0.99}
