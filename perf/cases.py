"""Performance cases of the sparse-prefill attention path.

Each case is one call, or one short fixed sequence of calls, that a program using
this package makes: a prefill attention layer through ``AttentionBackend.forward``
(every method of the backend, both head dims, several head layouts, batches, even
and ragged lengths), one decode step through the same entry, and the stage
functions of ``kernels`` / ``upstream`` called one by one as the selector studies
do. Inputs are bf16 and resident on the GPU, in the layouts transformers hands to
the attention function: the query a transposed view of ``[B, S, Hq, D]``, key and
value contiguous ``[B, Hkv, S, D]`` as a KV cache stores them.

Two kinds of values: ``"noise"`` is i.i.d. N(0, 1) with RoPE, on which routing keeps
every block (the headline workload); ``"topics"`` adds to Q and K a direction per
text segment (segments of 128 to 1024 tokens, 16 topics, query heads from flat to
peaked), on which alpha = 0.08 keeps about 20 % of the blocks at 32K tokens, the
density the reference publishes for real prompts.
"""

from __future__ import annotations

import math

import torch

from exp3_amd import attention, kernels, synthetic
from exp3_amd.upstream import flashprefill_native_forward as upstream

BLOCK = 128
SINK, WINDOW, LAST = 2, 4, 2        # the backend's defaults
TOPICS, SEGMENT = 16, 512
V1_ROUTED = ("fp_v1", "mean_native", "fp_v1_rescue", "fp_v1_rescue_v2")
SELECTORS = ("mean_balanced", "cgf_mean", "dispersion_mean")
MEAN = ("mean_native",) + SELECTORS
# (query heads, KV heads, head dim): Qwen2.5-7B, Llama-like 4:1, Qwen2.5-1.5B, no GQA,
# and the Qwen3.5 full-attention layers
LAYOUTS = ((28, 4, 128), (32, 8, 128), (12, 2, 128), (8, 8, 128), (16, 4, 256))


def _case(kind, seq, method="", alpha=0.08, values="topics", batch=1, layout=LAYOUTS[0], **more):
    return dict(kind=kind, method=method, alpha=alpha, seq=seq, batch=batch, q_heads=layout[0],
                kv_heads=layout[1], head_dim=layout[2], values=values, **more)


def listed():
    return [
        # a short chat turn: launches and latency
        _case("layer", 1089, "mean_native", name="layer_mean_native_1089"),
        # a one-page document with the moment selector (the reference's CPU-runnable length)
        _case("layer", 4096, "cgf_mean", name="layer_cgf_4096"),
        # a small serving batch of ragged prompts, Llama-like heads
        _case("layer", 2113, "mean_balanced", batch=4, layout=LAYOUTS[1],
              name="layer_balanced_b4_2113"),
        # the headline: a 32K layer on unstructured inputs, every block attended
        _case("layer", 32640, "mean_native", values="noise", name="layer_mean_native_32640"),
        # the same layer on a routed prompt, as in a long-document prefill
        _case("layer", 32640, "mean_native", name="layer_mean_native_32640_routed"),
        # the rescue variant at an odd mid length
        _case("layer", 20011, "fp_v1_rescue_v2", name="layer_rescue_v2_20011"),
        # the longest context, the dearest selector
        _case("layer", 131072, "dispersion_mean", alpha=0.04, name="layer_dispersion_131072"),
        # a head-dim-256 layer
        _case("layer", 12001, "fp_v1", layout=LAYOUTS[4], name="layer_fp_v1_d256_12001"),
        # dense prefill through this library's kernel, the baseline the sparse methods run against
        _case("dense", 8192, "dense", name="layer_dense_8192"),
        # one decode step behind a 32K prompt
        _case("decode", 32641, "mean_native", name="decode_32641"),
        # the V1 stages called one by one, with the mean tail and the merge (parity studies)
        _case("stages", 9000, "mean_native", name="stages_v1_9000"),
        # descriptors, scores and selection alone (selector studies)
        _case("selection", 32640, "cgf_mean", name="selection_cgf_32640"),
    ]


def _length(rng, low, high):
    seq = int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))
    return seq if rng.random() < 0.6 else max(low, seq // BLOCK * BLOCK)


def draw(rng):
    kind = rng.choice(("layer", "layer", "layer", "layer", "dense", "decode", "decode", "stages",
                       "selection"))
    layout = rng.choice(LAYOUTS)
    alpha = rng.choice((0.04, 0.08, 0.16))
    values = rng.choice(("topics", "topics", "noise"))
    batch = rng.choice((1, 1, 1, 2, 3, 4))
    if kind == "layer":
        method = rng.choice(V1_ROUTED + SELECTORS)
        return _case(kind, _length(rng, 130, 40000 // batch), method, alpha, values, batch, layout)
    if kind == "dense":
        return _case(kind, _length(rng, 130, 24000 // batch), "dense", alpha, values, batch, layout)
    if kind == "decode":
        batch = rng.choice((1, 1, 2, 4, 8))
        return _case(kind, _length(rng, 130, 131072 // batch), "mean_native", alpha, values, batch,
                     layout)
    if kind == "stages":
        return _case(kind, _length(rng, 130, 16000 // batch), "mean_native", alpha, values, batch,
                     layout)
    return _case(kind, _length(rng, 130, 32640 // batch), rng.choice(SELECTORS), alpha, values,
                 batch, layout)


# ------------------------------------------------------------------- inputs

def _inputs(case, seed):
    """q [B, Sq, Hq, D], k / v [B, S, Hkv, D] bf16 on the GPU; Sq = 1 for a decode step
    (the last position's query)."""
    device = torch.device("cuda")
    gen = torch.Generator(device).manual_seed(seed)
    batch, seq, heads = case["batch"], case["seq"], case["q_heads"]
    kv, dim = case["kv_heads"], case["head_dim"]
    rows = 1 if case["kind"] == "decode" else seq
    inv_freq = synthetic.rope_inv_freq(dim).to(device)
    positions = torch.arange(seq, device=device)
    topic = None
    if case["values"] == "topics":
        spans = torch.randint(SEGMENT // 4, 2 * SEGMENT, (8 * seq // SEGMENT + 8,), generator=gen,
                              device=device)
        segment = torch.searchsorted(spans.cumsum(0), positions, right=True)
        topic = torch.randint(0, TOPICS, (spans.numel(),), generator=gen, device=device)[segment]

    def draw_heads(count, where):
        x = torch.randn(batch, where.numel(), count, dim, generator=gen, device=device)
        return synthetic.apply_rope(x, where, inv_freq)

    k = draw_heads(kv, positions)
    directions = torch.randn(kv, TOPICS, dim, generator=gen, device=device)
    directions = torch.nn.functional.normalize(directions, dim=-1)
    if topic is not None:
        k += 0.75 * math.sqrt(dim) * directions[:, topic].transpose(0, 1)
    k = k.to(torch.bfloat16)
    v = torch.randn(batch, seq, kv, dim, generator=gen, device=device).to(torch.bfloat16)
    amplitude = torch.linspace(3.0, 10.0, heads, device=device) * math.sqrt(dim / 128)
    q = torch.empty(batch, rows, heads, dim, dtype=torch.bfloat16, device=device)
    group = heads // kv
    for g in range(kv):                 # by KV group: bounded fp32 temporaries
        part = slice(g * group, (g + 1) * group)
        x = draw_heads(group, positions[seq - rows:])
        if topic is not None:
            x += amplitude[part, None] * directions[g, topic[seq - rows:]][:, None]
        q[:, :, part] = x.to(torch.bfloat16)
    return q, k, v


class _Layer:
    layer_idx = 0


def prepare(case, seed):
    q, k, v = _inputs(case, seed)
    state = dict(kind=case["kind"], method=case["method"], alpha=case["alpha"],
                 scale=case["head_dim"] ** -0.5)
    if case["kind"] in ("stages", "selection"):
        return dict(state, q=q, k=k, v=v)
    backend = attention.AttentionBackend(alpha=case["alpha"], register=False,
                                         dense_impl="hip" if case["kind"] == "dense" else "sdpa")
    backend.configure(case["method"], case["alpha"])
    return dict(state, backend=backend, layer=_Layer(), query=q.transpose(1, 2),
                key=k.transpose(1, 2).contiguous(), value=v.transpose(1, 2).contiguous())


def run(state):
    scale = state["scale"]
    if state["kind"] == "stages":
        q, k, v = state["q"], state["k"], state["v"]
        descriptors = kernels.block_descriptors(k, v)
        mean_k = upstream.block_mean_k(k)
        scores = upstream.v1_scores(q, mean_k, scale)
        indices, counts = upstream.deal_output_score(scores, SINK, WINDOW, state["alpha"], LAST, 0)
        selected = kernels.mask_from_indices(indices, counts)
        exact_out, exact_lse = upstream.exact_attention(q, k, v, indices, counts, scale)
        mean_out, mean_lse = kernels.mean_tail(q, descriptors, selected, scale)
        out, lse = kernels.merge_exact_mean(exact_out, exact_lse, mean_out, mean_lse)
        return {"mean_k": mean_k, "scores": scores, "indices": indices, "counts": counts,
                "selected": selected, "exact_out": exact_out, "exact_lse": exact_lse,
                "mean_out": mean_out, "mean_lse": mean_lse, "out": out, "lse": lse}
    if state["kind"] == "selection":
        q, k, v = state["q"], state["k"], state["v"]
        d = kernels.block_descriptors(k, v)
        scores = kernels.selector_scores(q, d, scale, state["method"])
        selected = kernels.protected_selection(scores, state["alpha"], SINK, WINDOW, LAST)
        indices, counts = kernels.indices_from_mask(selected)
        return {"mean_k": d.mean_k, "mean_v": d.mean_v, "var_k": d.var_k, "sigma_v": d.sigma_v,
                "scores": scores, "selected": selected, "indices": indices, "counts": counts}
    return state["backend"].forward(state["layer"], state["query"], state["key"], state["value"],
                                    attention_mask=None, scaling=scale)[0]


# --------------------------------------------------------------------- work

def _blocks(seq):
    return (seq + BLOCK - 1) // BLOCK


def _density(case):
    """Share of the causal blocks that are attended: all for noise and dense, else the
    protected blocks plus a fifth of the rest (measured on the topic inputs at alpha 0.08)."""
    if case["kind"] == "dense" or case["values"] == "noise":
        return 1.0
    blocks = _blocks(case["seq"])
    kept = sum(t + 1 if t >= blocks - LAST else min(t + 1, SINK + WINDOW) for t in range(blocks))
    kept /= blocks * (blocks + 1) / 2
    return kept + 0.2 * (1 - kept)


def work(case):
    batch, seq, heads = case["batch"], case["seq"], case["q_heads"]
    kv, dim = case["kv_heads"], case["head_dim"]
    blocks = _blocks(seq)
    query, cache = 2 * batch * seq * heads * dim, 2 * 2 * batch * seq * kv * dim
    if case["kind"] == "decode":
        return {"bytes": cache + 2 * 2 * batch * heads * dim, "flops": 4 * batch * heads * seq * dim}
    pairs = batch * heads * seq * (seq + 1) / 2
    proxy = pairs / BLOCK                               # (row, visible block) pairs
    exact = 4 * dim * pairs * _density(case)
    tail = 4 * dim * proxy * (1 - _density(case))
    score = 2 * dim * proxy * (2 if case["method"] in ("cgf_mean", "dispersion_mean") else 1)
    entries = batch * blocks * blocks * heads           # scores f32, lists int64, mask bool
    moments = 4 * batch * blocks * kv * dim
    if case["kind"] == "dense":
        return {"bytes": 2 * query + cache, "flops": exact}
    if case["kind"] == "layer":
        return {"bytes": 2 * query + cache, "flops": exact + score
                + (0 if case["method"] in ("fp_v1", "fp_v1_rescue") else tail)}
    if case["kind"] == "selection":
        return {"bytes": query + cache + 3 * moments + entries * (4 + 1 + 8), "flops": score}
    # stages: exact and merged outputs bf16, mean output f32
    return {"bytes": query * (1 + 1 + 2 + 1) + cache + moments / 2 + entries * (4 + 8 + 1),
            "flops": exact + score + tail}


def tolerance(case):
    """About four times the present error against 64 bits (listed and drawn cases)."""
    if case["kind"] == "selection":     # fp32 scores: rel 1.5e-6, max 9e-6; no mask entry differed
        return {"rel": 6e-6, "max": 4e-5, "differ": 1e-3}
    if case["kind"] == "decode":        # bf16 outputs: rel 2.3e-3, max 7e-3
        return {"rel": 1e-2, "max": 3e-2}
    if case["kind"] == "stages":        # bf16 outputs: rel 2.7e-3, max 0.052; fp32 scores and LSE 1e-7
        return {"rel": 1e-2, "max": 0.2, "differ": 1e-3}
    return {"rel": 1e-2, "max": 0.3}    # bf16 outputs: rel 2.3e-3, max 0.074


# ---------------------------------------------------- the same in 64 bits

def _by_group(x, heads):
    """[S, Hkv, D] -> [Hq, S, D] in 64 bits."""
    return x.double().transpose(0, 1).repeat_interleave(heads // x.shape[1], 0).contiguous()


def _moments(x):
    """[S, H, D] -> per-block mean and variance [NB, H, D] in 64 bits."""
    seq, heads, dim = x.shape
    blocks = _blocks(seq)
    padded = torch.zeros(blocks * BLOCK, heads, dim, dtype=torch.float64, device=x.device)
    padded[:seq] = x
    padded = padded.view(blocks, BLOCK, heads, dim)
    count = torch.full((blocks, 1, 1), BLOCK, dtype=torch.float64, device=x.device)
    count[-1] = seq - (blocks - 1) * BLOCK
    mean = padded.sum(1) / count
    return mean, ((padded * padded).sum(1) / count - mean * mean).clamp_min(0)


def _protected(t, blocks, device):
    j = torch.arange(t + 1, device=device)
    return (j < SINK) | (t - j < WINDOW) | (t >= blocks - LAST)


def _v1_scores(q, mean_k, t, scale):
    """Tile t's V1 scores [Hq, t + 1]: q [Hq, rows, D], mean_k [Hq, NB, D]."""
    x = torch.matmul(q, mean_k[:, :t + 1].transpose(1, 2).contiguous()) * scale
    rows = torch.arange(q.shape[1], device=q.device) + t * BLOCK
    ends = (torch.arange(t + 1, device=q.device) + 1) * BLOCK - 1
    x = x.masked_fill(rows[:, None] < ends, -math.inf)
    top = x.amax((1, 2), keepdim=True)
    weight = torch.exp(x - torch.where(top.isfinite(), top, 0.0)).sum(1)
    return weight / (weight.sum(1, keepdim=True) + 1e-9)


def _selector_scores(q, mean_k, var_k, sigma_v, t, scale, method):
    """Tile t's selector scores over its history [Hq, t + 1] (0 at j = t)."""
    scores = torch.zeros(q.shape[0], t + 1, dtype=torch.float64, device=q.device)
    if t == 0:
        return scores
    logits = torch.matmul(q, mean_k[:, :t].transpose(1, 2).contiguous()) * scale
    spread = None
    if method != "mean_balanced":
        spread = torch.matmul(q * q, var_k[:, :t].transpose(1, 2).contiguous()) * scale ** 2
        logits = logits + 0.5 * spread
    share = torch.softmax(logits, -1)
    if method == "dispersion_mean":
        share = share * spread.sqrt() * sigma_v[:, None, :t]
    scores[:, :t] = share.mean(1)
    return scores


def _route(case, q, moments, t, scale):
    """(scores [Hq, t + 1], selected [Hq, t + 1]) of tile t."""
    mean_k16, mean_k, var_k, sigma_v = moments
    blocks = _blocks(case["seq"])
    if case["method"] in SELECTORS:
        scores = _selector_scores(q, mean_k, var_k, sigma_v, t, scale, case["method"])
        keep = (scores > 0) & (scores >= case["alpha"] * scores.amax(1, keepdim=True))
    else:
        scores = _v1_scores(q, mean_k16, t, scale)
        keep = scores >= case["alpha"] * scores.amax(1, keepdim=True)
    return scores, keep | _protected(t, blocks, q.device)


def _softmax_value(logits, values):
    """(softmax(logits) @ values, logsumexp); 0 and -inf where every logit is -inf."""
    lse = torch.logsumexp(logits, -1)
    weight = torch.exp(logits - torch.where(lse.isfinite(), lse, 0.0)[..., None])
    return torch.matmul(weight, values), lse


def _tail(case, q, k, v, mean_k, mean_v, unselected, t, scale):
    """Logits [Hq, rows, n] and values [Hq, n, D] of tile t's tail entries (fp_v1: none)."""
    heads, _, dim = q.shape
    if case["method"] not in MEAN + ("fp_v1_rescue", "fp_v1_rescue_v2") or t == 0:
        return q.new_empty(heads, q.shape[1], 0), v.new_empty(heads, 0, dim)
    hidden = torch.where(unselected[:, :t], 0.0, -math.inf).double()[:, None]
    if case["method"] in MEAN:
        logits = torch.matmul(q, mean_k[:, :t].transpose(1, 2).contiguous()) * scale
        return logits + math.log(BLOCK) + hidden, mean_v[:, :t]
    history = k[:, :t * BLOCK].view(heads, t, BLOCK, dim)
    best = torch.matmul(history.reshape(heads, t * BLOCK, dim), q.mean(1)[:, :, None])
    token = best.view(heads, t, BLOCK).argmax(2) + torch.arange(t, device=q.device) * BLOCK
    pick = token[:, :, None].expand(-1, -1, dim)
    keys, values = k.gather(1, pick), v.gather(1, pick)
    logits = torch.matmul(q, keys.transpose(1, 2).contiguous()) * scale + hidden
    if case["method"] == "fp_v1_rescue":
        return logits, values
    rest_k = (mean_k[:, :t] * BLOCK - keys) / (BLOCK - 1)
    rest_v = (mean_v[:, :t] * BLOCK - values) / (BLOCK - 1)
    rest = torch.matmul(q, rest_k.transpose(1, 2).contiguous()) * scale
    return (torch.cat((logits, rest + math.log(BLOCK - 1) + hidden), 2),
            torch.cat((values, rest_v), 1))


def exact(case, seed):
    if case["seq"] * case["seq"] * case["batch"] > 2e9:
        return None                     # the 131072-token layer: minutes in 64 bits
    q, k, v = _inputs(case, seed)
    batch, seq, heads = case["batch"], case["seq"], case["q_heads"]
    scale, blocks, device = case["head_dim"] ** -0.5, _blocks(case["seq"]), q.device
    f64 = dict(dtype=torch.float64, device=device)
    if case["kind"] == "decode":
        out = torch.empty(batch, 1, heads, case["head_dim"], **f64)
        for b in range(batch):
            keys, values = _by_group(k[b], heads), _by_group(v[b], heads)
            logits = torch.matmul(keys, q[b, 0].double()[:, :, None]).transpose(1, 2) * scale
            out[b, 0] = _softmax_value(logits, values)[0][:, 0]
        return out
    routed = case["kind"] in ("stages", "selection")
    scores = torch.zeros(batch, blocks, blocks, heads, **f64) if routed else None
    out, exact_out, mean_out = (torch.zeros(q.shape, **f64) for _ in range(3))
    lse, exact_lse, mean_lse = (torch.full(q.shape[:3], -math.inf, **f64) for _ in range(3))
    stats = []
    for b in range(batch):
        keys, values = _by_group(k[b], heads), _by_group(v[b], heads)
        mean_k, var_k = _moments(k[b])
        mean_v, var_v = _moments(v[b])
        sigma_v = var_v.sum(-1).sqrt()
        stats.append((mean_k, mean_v, var_k, sigma_v))
        expand = heads // case["kv_heads"]
        wide = [x.repeat_interleave(expand, 1).transpose(0, 1).contiguous()
                for x in (mean_k.to(torch.bfloat16).double(), mean_k, var_k, sigma_v)]
        wide_v = mean_v.repeat_interleave(expand, 1).transpose(0, 1).contiguous()
        for t in range(blocks):
            first, last = t * BLOCK, min(seq, (t + 1) * BLOCK)
            query = q[b, first:last].double().transpose(0, 1).contiguous()
            chosen = torch.ones(heads, t + 1, dtype=torch.bool, device=device)
            if case["kind"] != "dense":
                tile_scores, chosen = _route(case, query, wide, t, scale)
            if routed:
                scores[b, t, :t + 1] = tile_scores.T
            if case["kind"] == "selection":
                continue
            logits = torch.matmul(query, keys[:, :last].transpose(1, 2).contiguous()) * scale
            mask = chosen.repeat_interleave(BLOCK, 1)[:, None, :last]
            causal = (torch.arange(last, device=device)
                      <= torch.arange(first, last, device=device)[:, None])
            logits = logits.masked_fill(~(mask & causal), -math.inf)
            extra, extra_v = _tail(case, query, keys, values, wide[1], wide_v, ~chosen, t, scale)
            if case["kind"] == "stages":
                for o, l, x, y in ((exact_out, exact_lse, logits, values[:, :last]),
                                   (mean_out, mean_lse, extra, extra_v)):
                    if x.shape[2]:
                        part, total = _softmax_value(x, y)
                        o[b, first:last] = part.transpose(0, 1)
                        l[b, first:last] = total.T
            result, total = _softmax_value(torch.cat((logits, extra), 2),
                                           torch.cat((values[:, :last], extra_v), 1))
            out[b, first:last] = result.transpose(0, 1)
            lse[b, first:last] = total.T
    if not routed:
        return out
    mean_k, mean_v, var_k, sigma_v = (torch.stack(x) for x in zip(*stats))
    lists = {"indices": None, "counts": None, "selected": None}
    if case["kind"] == "selection":
        return {"mean_k": mean_k, "mean_v": mean_v, "var_k": var_k, "sigma_v": sigma_v,
                "scores": scores, **lists}
    return {"mean_k": mean_k, "scores": scores, **lists, "exact_out": exact_out,
            "exact_lse": exact_lse, "mean_out": mean_out, "mean_lse": mean_lse, "out": out,
            "lse": lse}
