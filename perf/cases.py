"""Performance cases of the indexer: the work a serving or prefill program has it do, at the sizes it has it done.

``listed()`` names the cases, ``draw(rng)`` draws one more from the same ranges, ``prepare`` makes on the GPU what the
program holds before the call, ``run`` is one pass through the public entry points, and ``work``, ``tolerance`` and
``exact`` say what the pass cannot do without, how far another correct implementation may be off, and what the outputs
are in 64 bits.

Kinds:
  decode       one batched decode step: dense scores of every cached key and the exact top-k of each sequence
  single       one fp32 query against one fp32 context, and its ranked (stable) top-k
  prefill      a causal prefill of one layer: scores and per-query top-k in one call
  chunk        a chunk of queries against a long cached context, then the per-query top-k
  encode_step  the indexer's encoders for one new token per sequence, keys appended to the cache
  encode       the indexer's encoders for a prefill chunk
  temporal     a pruned decode step seeded by the previous step's top-k
  progressive  the 8-head screen and promotion of one sequence, then the top-k of what it accepted
"""

from __future__ import annotations

import math

import torch

from dsa_amd import decode, metrics, progressive_kernel, sidecar, temporal

HEADS = 64
DIM = 128
ROPE_DIM = 64
THETA = 10_000.0
CACHE_ROWS = 1024  # cached keys per sequence of an encode step
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32, "fp8": torch.bfloat16}
KEY_BYTES = {"bf16": 256.0, "f16": 256.0, "f32": 512.0, "fp8": 128.0 + 4.0 / 128.0}
# Sequences x keys of the largest decode step, query x key pairs of the largest prefill, and token x hidden products of
# the largest encoder call: no drawn case is larger.
MOST_KEYS = 524288
MOST_PAIRS = 512 * 32768
MOST_ENCODE = 4096 * 2048


def listed() -> list[dict]:
    return [
        # Interactive decoding of a short conversation: one sequence, where launches and latency count.
        {"name": "decode_one_4k", "kind": "decode", "dtype": "bf16", "batch": 1, "length": 4096, "k": 256},
        # A half-full server whose context is no round number.
        {"name": "decode_ragged_f16", "kind": "decode", "dtype": "f16", "batch": 5, "length": 20011, "k": 2048},
        # The headline decode step: 16 sequences of 32K keys.
        {"name": "decode_batch_32k", "kind": "decode", "dtype": "bf16", "batch": 16, "length": 32768, "k": 2048},
        # Long-context decoding on a quantised key cache.
        {"name": "decode_long_fp8", "kind": "decode", "dtype": "fp8", "batch": 4, "length": 131072, "k": 2048},
        # The full-precision single-sequence path that analyses and checks run.
        {"name": "single_f32_4k", "kind": "single", "dtype": "f32", "length": 4096, "k": 256},
        # One layer of a causal prefill, every query's top-512.
        {"name": "prefill_causal_4k", "kind": "prefill", "dtype": "bf16", "batch": 1, "queries": 4096, "length": 4096,
         "k": 512},
        # Chunked prefill: the next 512 tokens of a prompt whose context has reached 32K.
        {"name": "chunk_512_of_32k", "kind": "chunk", "dtype": "bf16", "queries": 512, "length": 32768, "k": 2048},
        # The encoders of a decode step: 16 sequences, one token each.
        {"name": "encode_step_16", "kind": "encode_step", "tokens": 16, "hidden": 2048},
        # The encoders of a prefill chunk.
        {"name": "encode_prefill_4k", "kind": "encode", "tokens": 4096, "hidden": 2048},
        # The pruned decode step at its dynamic threshold, context just past 16K.
        {"name": "temporal_dynamic_16k", "kind": "temporal", "dtype": "bf16", "batch": 4, "length": 16639, "k": 2048,
         "block": 64, "method": "dynamic", "order": "previous_hot", "wave": 9, "margin": 1.0},
        # The pruned decode step with a fixed threshold on the long quantised cache.
        {"name": "temporal_static_fp8", "kind": "temporal", "dtype": "fp8", "batch": 4, "length": 131072, "k": 2048,
         "block": 64, "method": "static", "order": "address", "wave": 0, "margin": 0.0},
        # The 8-head screen with promotion at 32K keys, as the method comparison runs it.
        {"name": "progressive_32k", "kind": "progressive", "dtype": "bf16", "length": 32768, "k": 2048, "block": 64,
         "direct": 0.594},
    ]


def _spread(rng, low: int, high: int) -> int:
    """A size between low and high, even over its logarithm; most are odd or ragged."""

    value = int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))
    if rng.random() < 0.3:
        value = value // 64 * 64
    return max(low, min(high, value))


def draw(rng) -> dict:
    kind = rng.choice(["decode"] * 4 + ["single", "prefill", "chunk", "encode_step", "encode", "temporal", "temporal",
                                        "progressive"])
    if kind == "decode":
        batch = _spread(rng, 1, 16)
        length = _spread(rng, 1024, min(131072, MOST_KEYS // batch))
        return {"kind": kind, "dtype": rng.choice(["bf16", "f16", "fp8"]), "batch": batch, "length": length,
                "k": min(length // 2, _spread(rng, 128, 2048))}
    if kind == "single":
        length = _spread(rng, 1024, 32768)
        return {"kind": kind, "dtype": "f32", "length": length, "k": min(length // 4, _spread(rng, 64, 2048))}
    if kind == "prefill":
        length = _spread(rng, 256, 4096)
        batch = rng.randint(1, max(1, min(4, MOST_PAIRS // (length * length))))
        return {"kind": kind, "dtype": rng.choice(["bf16", "f16"]), "batch": batch,
                "queries": rng.randint(length // 4, length), "length": length, "k": _spread(rng, 64, 2048)}
    if kind == "chunk":
        length = _spread(rng, 6144, 32768)
        queries = _spread(rng, 16, min(1024, MOST_PAIRS // length))
        return {"kind": kind, "dtype": rng.choice(["bf16", "fp8"]), "queries": queries, "length": length,
                "k": _spread(rng, 256, 2048)}
    if kind == "encode_step":
        return {"kind": kind, "tokens": rng.randint(1, 16), "hidden": rng.choice([1024, 2048, 4096])}
    if kind == "encode":
        hidden = rng.choice([1024, 2048, 4096])
        return {"kind": kind, "tokens": _spread(rng, 17, min(4096, MOST_ENCODE // hidden)), "hidden": hidden}
    if kind == "temporal":
        batch = _spread(rng, 1, 8)
        block = rng.choice([16, 32, 64, 128])
        length = _spread(rng, 4096, min(131072, MOST_KEYS // batch, 2048 * block))
        method = rng.choice(["static", "dynamic", "dynamic"])
        blocks = -(-length // block)
        return {"kind": kind, "dtype": rng.choice(["bf16", "fp8"]), "batch": batch, "length": length,
                "k": _spread(rng, 256, 2048), "block": block, "method": method,
                "order": "address" if method == "static" else rng.choice(["address", "previous_hot", "upper_hot"]),
                "wave": 0 if method == "static" else max(1, -(-blocks // 32)), "margin": rng.choice([0.0, 0.25, 0.5, 1.0])}
    length = _spread(rng, 4096, 65536)
    return {"kind": kind, "dtype": rng.choice(["bf16", "f16"]), "length": length, "k": _spread(rng, 256, 2048),
            "block": rng.choice([16, 32, 64, 128]), "direct": rng.choice([0.5, 0.594, 0.703, 0.9])}


# ---------------------------------------------------------------------------------------------------------------------
# Inputs


def _queries(gen, shape, dtype) -> torch.Tensor:
    return (torch.randn(*shape, HEADS, DIM, generator=gen, device="cuda") / math.sqrt(DIM)).to(dtype)


def _weights(gen, shape) -> torch.Tensor:
    return torch.randn(*shape, HEADS, generator=gen, device="cuda") / 8.0


def _keys(gen, batch: int, length: int, dtype: str):
    """Cached keys: unit normal with one in a hundred four times as long (sinks and hot tokens); fp8 keys are drawn
    around ten topics and quantised with one scale per 128 keys."""

    if dtype != "fp8":
        keys = torch.randn(batch, length, DIM, generator=gen, device="cuda")
        hot = torch.rand(batch, length, generator=gen, device="cuda") < 0.01
        keys[hot] *= 4.0
        return keys.to(DTYPES[dtype]), None
    centroids = torch.randn(batch, 10, DIM, generator=gen, device="cuda")
    topic = torch.randint(0, 10, (batch, length), generator=gen, device="cuda")
    raw = torch.gather(centroids, 1, topic[..., None].expand(-1, -1, DIM))
    raw += torch.randn(batch, length, DIM, generator=gen, device="cuda")
    raw /= math.sqrt(2.0)
    groups = -(-length // 128)
    padded = torch.nn.functional.pad(raw, (0, 0, 0, groups * 128 - length)).reshape(batch, groups, 128 * DIM)
    scales = padded.abs().amax(dim=2) / 448.0
    codes = (padded / scales[..., None]).reshape(batch, groups * 128, DIM)[:, :length].to(torch.float8_e4m3fn)
    return codes.contiguous(), scales.contiguous()


def _wide_keys(keys: torch.Tensor, scales, dtype) -> torch.Tensor:
    """The keys' values ``[B, L, 128]`` in a wider type (fp8 codes times their scales)."""

    wide = keys.to(dtype)
    if scales is not None:
        wide = wide * scales.to(dtype).repeat_interleave(128, dim=1)[:, : keys.shape[1], None]
    return wide


def _plain_scores(queries: torch.Tensor, weights: torch.Tensor, keys: torch.Tensor, heads=None) -> torch.Tensor:
    """``sum_h w_h relu(q_h . k)`` of queries ``[n, 64, 128]`` against keys ``[L, 128]``, in the keys' type."""

    q, w = queries.to(keys.dtype), weights.to(keys.dtype)
    if heads is not None:
        q, w = q[:, heads], w[:, heads]
    out = torch.empty(q.shape[0], keys.shape[0], dtype=keys.dtype, device=keys.device)
    step = max(1, (1 << 27) // (q.shape[1] * keys.shape[0]))
    columns = keys.t().contiguous()
    for i in range(0, q.shape[0], step):
        part = q[i : i + step]
        dots = (part.reshape(-1, DIM) @ columns).clamp_(min=0).reshape(part.shape[0], part.shape[1], -1)
        out[i : i + step] = dots.mul_(w[i : i + step, :, None]).sum(dim=1)
    return out


def _block_max(scores: torch.Tensor, block: int) -> torch.Tensor:
    blocks = -(-scores.shape[1] // block)
    pad = blocks * block - scores.shape[1]
    return torch.nn.functional.pad(scores, (0, pad), value=-math.inf).reshape(scores.shape[0], blocks, block).amax(dim=2)


def prepare(case: dict, seed: int) -> dict:
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    kind = case["kind"]
    state = {"case": case}
    if kind in ("encode_step", "encode"):
        hidden, tokens = case["hidden"], case["tokens"]
        module = sidecar.LightningIndexerSidecar(hidden_size=hidden).to("cuda", torch.bfloat16).eval()
        module.weights_proj.to(torch.float32)  # the head weights stay fp32, as the module declares them
        with torch.no_grad():
            for p in (module.wq.weight, module.wk.weight, module.weights_proj.weight):
                p.copy_(torch.randn(p.shape, generator=gen, device="cuda") * hidden**-0.5)
            module.k_norm.weight.copy_(1 + 0.1 * torch.randn(DIM, generator=gen, device="cuda"))
            module.k_norm.bias.copy_(0.1 * torch.randn(DIM, generator=gen, device="cuda"))
        state["module"] = module
        state["hidden"] = torch.randn(tokens, hidden, generator=gen, device="cuda").to(torch.bfloat16)
        if kind == "encode_step":
            state["positions"] = torch.randint(0, CACHE_ROWS, (tokens,), generator=gen, device="cuda")
            state["cache"] = torch.zeros(tokens * CACHE_ROWS, DIM, device="cuda", dtype=torch.bfloat16)
            state["rows"] = torch.arange(tokens, device="cuda") * CACHE_ROWS + state["positions"]
        else:
            start = int(torch.randint(0, 16384, (1,), generator=gen, device="cuda"))
            state["positions"] = torch.arange(start, start + tokens, device="cuda")
        return state
    dtype, length = case["dtype"], case["length"]
    batch = case.get("batch", 1)
    if kind == "prefill" or kind == "chunk":
        state["q"] = _queries(gen, (batch, case["queries"]), DTYPES[dtype])
        state["w"] = _weights(gen, (batch, case["queries"]))
    else:
        state["q"] = _queries(gen, (batch,), DTYPES[dtype])
        state["w"] = _weights(gen, (batch,))
    state["keys"], state["scales"] = _keys(gen, batch, length, dtype)
    if kind == "single":
        state["q"], state["w"], state["keys"] = state["q"][0], state["w"][0], state["keys"][0]
    elif kind == "temporal":
        # The previous step: one key fewer, a query the current one has drifted from, its dense scores and top-k.
        k, block = case["k"], case["block"]
        q_prev = state["q"]
        drift = torch.randn(q_prev.shape, generator=gen, device="cuda") / math.sqrt(DIM)
        state["q"] = (0.95 * q_prev.float() + math.sqrt(1 - 0.95**2) * drift).to(q_prev.dtype)
        wide = _wide_keys(state["keys"], state["scales"], torch.float32)
        now = torch.cat([_plain_scores(state["q"][b : b + 1], state["w"][b : b + 1], wide[b]) for b in range(batch)])
        prev = torch.cat([_plain_scores(q_prev[b : b + 1], state["w"][b : b + 1], wide[b, : length - 1])
                          for b in range(batch)])
        state["prev_max"] = _block_max(prev, block)
        state["prev_topk"] = torch.topk(prev, k, dim=1).indices.sort(dim=1).values.contiguous()
        sigma = (now[:, : length - 1] - prev).std(dim=1, unbiased=False)
        state["gamma"] = (case["margin"] * sigma).contiguous()
    elif kind == "progressive":
        state["q"], state["w"], state["keys"] = state["q"][0], state["w"][0], state["keys"][0]
        blocks = -(-length // case["block"])
        selected = torch.argsort(state["w"].abs(), descending=True, stable=True)[:8].to(torch.int32)
        mask = torch.ones(HEADS, dtype=torch.bool, device="cuda")
        mask[selected.long()] = False
        state["selected"] = selected.contiguous()
        state["remaining"] = torch.arange(HEADS, dtype=torch.int32, device="cuda")[mask].contiguous()
        direct = torch.zeros(blocks, dtype=torch.bool, device="cuda")
        direct[torch.randperm(blocks, generator=gen, device="cuda")[: round(case["direct"] * blocks)]] = True
        state["direct"] = direct
        # The threshold that promotes a tenth of the screened blocks, halfway between two blocks' maxima.
        screen = _plain_scores(state["q"][None], state["w"][None], state["keys"].float(), selected.long())
        cold = _block_max(screen, case["block"])[0][~direct]
        ranked = cold.sort(descending=True).values
        promoted = max(1, min(ranked.numel() - 1, round(0.1 * ranked.numel())))
        state["threshold"] = ((ranked[promoted - 1] + ranked[promoted]) / 2).reshape(1)
    return state


# ---------------------------------------------------------------------------------------------------------------------
# One pass


def run(state: dict):
    case = state["case"]
    kind = case["kind"]
    if kind == "decode":
        indices, scores = decode.indexer_topk(state["q"], state["w"], state["keys"], case["k"], key_scales=state["scales"],
                                              return_scores=True)
        return {"scores": scores, "topk": indices}
    if kind == "single":
        scores = progressive_kernel.full_scores_hip(state["q"], state["w"], state["keys"])
        return {"scores": scores, "topk": metrics.topk(scores, case["k"])}
    if kind == "prefill":
        scores, indices = sidecar.score_encoded_topk(state["q"], state["w"], state["keys"], case["k"], causal=True)
        return {"scores": scores, "topk": indices}
    if kind == "chunk":
        scores = sidecar.score_encoded(state["q"], state["w"], state["keys"], causal=True, key_scales=state["scales"])
        return {"scores": scores, "topk": metrics.topk(scores[0], case["k"], sorted=False)}
    if kind == "encode_step":
        keys = state["module"].encode_keys(state["hidden"], state["positions"], out=state["cache"], out_rows=state["rows"])
        queries, weights = state["module"].encode_queries(state["hidden"], state["positions"])
        return {"keys": keys, "queries": queries, "weights": weights}
    if kind == "encode":
        keys = state["module"].encode_keys(state["hidden"], state["positions"])
        queries, weights = state["module"].encode_queries(state["hidden"], state["positions"])
        return {"keys": keys, "queries": queries, "weights": weights}
    if kind == "temporal":
        step = temporal.temporal_step(
            state["q"], state["w"], state["keys"], state["prev_max"], case["length"] - 1, state["prev_topk"],
            state["gamma"], block_size=case["block"], method=case["method"], scan_order=case["order"],
            wave=max(1, case["wave"]), key_scales=state["scales"])
        return {"scores": step.scores, "kept": step.evaluated_blocks, "topk": step.topk, "scored": step.qk_scored}
    result = progressive_kernel.progressive_scores_hip(
        state["q"], state["w"], state["keys"], state["selected"], state["direct"], state["threshold"],
        block_size=case["block"], remaining_heads=state["remaining"])
    return {"scores": result.scores, "accepted": result.accepted_blocks, "block_max": result.block_max,
            "topk": metrics.topk(result.scores, case["k"], sorted=False)}


# ---------------------------------------------------------------------------------------------------------------------
# What a pass costs and how exact it is


def work(case: dict) -> dict:
    kind = case["kind"]
    per_pair = HEADS * (2.0 * DIM + 2.0)  # one dot product, ReLU-weighted sum per head
    if kind in ("encode_step", "encode"):
        tokens, hidden = case["tokens"], case["hidden"]
        features = HEADS * DIM + DIM + HEADS
        weights = 2.0 * hidden * (HEADS * DIM + DIM) + 4.0 * hidden * HEADS
        outputs = tokens * (2.0 * (HEADS * DIM + DIM) + 4.0 * HEADS)
        return {"bytes": tokens * (2.0 * hidden + 8.0) + weights + outputs, "flops": 2.0 * tokens * hidden * features}
    length, k, batch = case["length"], case["k"], case.get("batch", 1)
    query = HEADS * (DIM * (4.0 if case["dtype"] == "f32" else 2.0) + 4.0)
    keys = KEY_BYTES[case["dtype"]] * length
    if kind in ("prefill", "chunk"):
        queries = case["queries"]
        visible = queries * (length - queries) + queries * (queries + 1) / 2.0
        return {"bytes": batch * (keys + queries * (query + 4.0 * length + 8.0 * k)), "flops": batch * visible * per_pair}
    if kind == "progressive":
        accepted = case["direct"] + 0.1 * (1.0 - case["direct"])
        share = accepted + (1.0 - accepted) * 8.0 / HEADS
        return {"bytes": query + keys + 4.0 * length + 8.0 * k, "flops": length * per_pair * share}
    extra = 8.0 * k + 9.0 * -(-length // case["block"]) if kind == "temporal" else 0.0
    return {"bytes": batch * (query + keys + 4.0 * length + 8.0 * k + extra), "flops": batch * length * per_pair}


def tolerance(case: dict) -> dict:
    # Measured against exact(): bf16 encoder rows 2.5e-3 to 3e-3 (rounded after the projection and in the rotation), fp32
    # scores 0.7e-7 to 1.5e-7.  Near-ties at the cut may swap a key in a few rows of many.
    if case["kind"] in ("encode_step", "encode"):
        return {"rel": 1e-2}
    return {"rel": 6e-7, "max": 2e-5, "differ": 0.005}


def _exact_temporal(state: dict, scores: torch.Tensor) -> torch.Tensor:
    """The pruned step's scores (-inf where not evaluated) from 64-bit scores ``[B, L]``: seeds first, then every block
    of the scan whose bound reaches the threshold, refreshed after each wave of blocks by the dynamic method."""

    case = state["case"]
    block, k, length = case["block"], case["k"], case["length"]
    out = torch.full_like(scores, -math.inf)
    for b in range(scores.shape[0]):
        row = scores[b]
        seen = torch.zeros(length, dtype=torch.bool, device=row.device)
        seen[state["prev_topk"][b]] = True
        bound = state["prev_max"][b].double() + state["gamma"][b].double()
        bound = torch.nn.functional.pad(bound, (0, -(-length // block) - bound.numel()), value=math.inf)
        bound[(length - 1) // block] = math.inf
        hot = torch.zeros(bound.numel(), dtype=torch.bool, device=row.device)
        hot[state["prev_topk"][b] // block] = True
        order = torch.arange(bound.numel(), device=row.device)
        if case["order"] != "address":
            order = torch.argsort(bound, descending=True, stable=True)
            if case["order"] == "previous_hot":
                order = order[torch.argsort((~hot[order]).to(torch.int8), stable=True)]
        threshold = row[seen].min()
        wave = case["wave"] if case["method"] == "dynamic" else order.numel()
        block_of = torch.arange(length, device=row.device) // block
        for i in range(0, order.numel(), wave):
            group = order[i : i + wave]
            kept = torch.zeros(bound.numel(), dtype=torch.bool, device=row.device)
            kept[group[~(bound[group] < threshold)]] = True
            seen |= kept[block_of]
            if case["method"] == "dynamic":
                threshold = torch.topk(row[seen], k).values[-1]
        out[b] = torch.where(seen, row, out[b])
    return out


def _exact_encode(state: dict) -> dict:
    module, hidden = state["module"], state["hidden"].double()
    angle = state["positions"].double()[:, None] * THETA ** (-torch.arange(ROPE_DIM // 2, device="cuda").double() / (ROPE_DIM // 2))
    cos, sin = angle.cos(), angle.sin()

    def rope(x):
        c, s = (cos, sin) if x.ndim == 2 else (cos[:, None], sin[:, None])
        a, b, rest = x[..., : ROPE_DIM // 2], x[..., ROPE_DIM // 2 : ROPE_DIM], x[..., ROPE_DIM:]
        return torch.cat((a * c - b * s, b * c + a * s, rest), dim=-1)

    keys = torch.nn.functional.layer_norm(hidden @ module.wk.weight.double().t(), (DIM,), module.k_norm.weight.double(),
                                          module.k_norm.bias.double(), module.k_norm.eps)
    keys = rope(keys)
    if state["case"]["kind"] == "encode_step":
        cache = torch.zeros(state["cache"].shape, dtype=torch.float64, device="cuda")
        cache[state["rows"]] = keys
        keys = cache
    queries = rope((hidden @ module.wq.weight.double().t()).reshape(-1, HEADS, DIM))
    weights = (hidden @ module.weights_proj.weight.double().t()) * (HEADS * DIM) ** -0.5
    return {"keys": keys, "queries": queries, "weights": weights}


@torch.no_grad()
def exact(case: dict, seed: int):
    state = prepare(case, seed)
    kind = case["kind"]
    if kind in ("encode_step", "encode"):
        return _exact_encode(state)
    if kind in ("single", "progressive"):
        wide = state["keys"].double()
        scores = _plain_scores(state["q"][None], state["w"][None], wide)[0]
        if kind == "single":
            return {"scores": scores, "topk": None}
        screen = _plain_scores(state["q"][None], state["w"][None], wide, state["selected"].long())
        maxima = _block_max(screen, case["block"])[0]
        maxima[state["direct"]] = -math.inf
        accepted = state["direct"] | (maxima >= state["threshold"].double())
        kept = accepted.repeat_interleave(case["block"])[: case["length"]]
        return {"scores": scores.masked_fill(~kept, -math.inf), "accepted": None, "block_max": maxima, "topk": None}
    wide = _wide_keys(state["keys"], state["scales"], torch.float64)
    if kind in ("prefill", "chunk"):
        scores = torch.stack([_plain_scores(q, w, k) for q, w, k in zip(state["q"], state["w"], wide)])
        limit = torch.arange(case["queries"], device="cuda")[:, None] + (case["length"] - case["queries"])
        hidden = torch.arange(case["length"], device="cuda")[None] > limit
        return {"scores": scores.masked_fill_(hidden, -math.inf), "topk": None}
    scores = torch.cat([_plain_scores(q[None], w[None], k) for q, w, k in zip(state["q"], state["w"], wide)])
    if kind == "temporal":
        return {"scores": _exact_temporal(state, scores), "kept": None, "topk": None, "scored": None}
    return {"scores": scores, "topk": None}
