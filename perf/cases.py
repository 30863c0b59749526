"""The calls whose speed this framework is judged by, as a user's program makes them.

A request's life through the public entry points: the prompt's block summary
(``build_summary`` over a KV cache, or ``store_and_build_summary`` when the
summary is made while the cache is written), the prompt anchors' mask
(``select_blocks_union``), then decode steps (``sparse_attention``), called
eagerly or captured once as a HIP graph over the layers and replayed for each
token, and the dense layers' decode (``dense_decode``).  Head counts, head
dims, block sizes, eps and anchors are those of the benchmark and the model
configurations; K/V follow ``refinekv.testing``'s recipe, drawn on the GPU.
"""

import math
import os
import sys

import torch

_PACKAGE = os.path.abspath("refinekv-release_amd")  # (the working folder is the repository's root)
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

from refinekv import (RefineKVConfig, build_summary, select_blocks_union,  # noqa: E402
                      sparse_attention)
from refinekv._hip import dense_decode  # noqa: E402
from refinekv.summary import store_and_build_summary  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
CAPACITY = 128  # cache rows kept for generated tokens
INFLATE = 1 + 2 ** -8


def _decode(name, tokens, **over):
    case = dict(kind="decode", name=name, heads=8, group=4, dim=128, block=32, tokens=tokens,
                suffix=40, eps=0.01, reduction="any", spikes=0.02, anchors=0, layers=8,
                graph=True)
    case.update(over)
    return case


def _summary(name, tokens, **over):
    case = dict(kind="summary", name=name, heads=8, dim=128, block=32, tokens=tokens,
                dtype="bf16", store=False)
    case.update(over)
    return case


def _anchors(name, tokens, anchors, **over):
    case = dict(kind="anchors", name=name, heads=8, group=4, dim=128, block=32, tokens=tokens,
                eps=0.01, reduction="any", spikes=0.02, anchors=anchors)
    case.update(over)
    return case


def listed():
    return [
        # one request's prompt on an ordinary cache, a prompt of whole blocks
        _summary("summary_32k", 32768),
        # a short chat prompt: launches and the call itself count
        _summary("summary_short_ragged", 2003),
        # prompts are seldom whole blocks: a long document's prompt, its
        # summary built while the visible cache takes the keys and values
        # (values still in the projection's layout)
        _summary("summary_store_128k_ragged", 131001, store=True),
        # the 16-bit float type that is not bf16, 16-token blocks, a ragged
        # prompt in a cache with free rows behind it
        _summary("summary_fp16_b16_ragged", 48500, dtype="fp16", block=16),
        # the anchors' mask at the end of prefill: the two model
        # configurations that use anchors
        _anchors("anchors_32k", 32768, 32),
        _anchors("anchors_g7_64k", 65536, 64, heads=4, group=7, block=64, eps=0.005,
                 reduction="max"),
        # one layer's step called eagerly on a short ragged prompt
        _decode("decode_eager_short", 2003, layers=1, graph=False, spikes=0.05),
        # graph-replayed decode steps: the configurations' shapes from an
        # ordinary prompt to the headline's 131072 tokens
        _decode("decode_32k", 32768),
        _decode("decode_g7_64k", 65536, heads=4, group=7, block=64, eps=0.005, reduction="max",
                spikes=0.05, anchors=4),
        _decode("decode_128k", 131072),
        # the longest context of the op sweep at its finest blocks
        _decode("decode_512k_b16", 524288, block=16, spikes=0.05, layers=2),
        # a dense layer's decode over a long cache
        dict(kind="dense", name="dense_64k", heads=8, group=4, dim=128, tokens=65573, layers=4),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _unnamed(case):
    return {key: value for key, value in case.items() if key != "name"}


def draw(rng):
    kind = rng.choice(("decode", "decode", "decode", "summary", "summary", "anchors", "dense"))
    if kind == "summary":
        dim = rng.choice((64, 128, 128, 128, 96, 256))
        dtype = rng.choice(("bf16", "bf16", "bf16", "fp16", "fp32"))
        most = min(100000, 25600000 // (dim * DTYPES[dtype].itemsize))
        return _unnamed(_summary("", _log_int(rng, 500, most), dim=dim, dtype=dtype,
                                 heads=rng.choice((2, 4, 8)), block=rng.choice((16, 32, 64)),
                                 store=rng.random() < 0.4))
    heads, group, dim = rng.choice(((8, 4, 128), (8, 4, 128), (4, 7, 128), (8, 4, 64),
                                    (2, 6, 128), (4, 2, 96), (8, 1, 128)))
    if kind == "dense":
        return dict(kind="dense", heads=heads, group=group, dim=dim,
                    tokens=_log_int(rng, 1000, 131072), layers=2)
    block = rng.choice((16, 32, 32, 64))
    eps = rng.choice((0.005, 0.01, 0.1))
    reduction = rng.choice(("any", "any", "max", "mean"))
    spikes = rng.choice((0.01, 0.02, 0.05, 0.2))
    if kind == "anchors":  # (short prompts with few spikes would expand whole)
        spikes = max(spikes, 0.05)
        return _unnamed(_anchors("", _log_int(rng, 2000, 65536), rng.choice((1, 7, 16, 32, 64)),
                                 heads=heads, group=group, dim=dim, block=block, eps=eps,
                                 reduction=reduction, spikes=spikes))
    tokens = _log_int(rng, 1000, 300000)
    if rng.random() < 0.4:
        tokens = -(-tokens // block) * block
    if rng.random() < 0.15:  # a head dim and group of wide heads
        heads, group, dim, tokens = 2, 8, 256, min(tokens, 100000)
    return _unnamed(_decode("", tokens, heads=heads, group=group, dim=dim, block=block, eps=eps,
                            reduction=reduction, spikes=spikes, suffix=rng.randint(1, 120),
                            anchors=rng.choice((0, 0, 8)), layers=2, graph=rng.random() < 0.7))


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator("cuda").manual_seed(seed * 1000003 + 17)


def _normal(gen, shape, dtype=torch.float32):
    return torch.randn(shape, generator=gen, device="cuda", dtype=dtype)


def _cache(gen, case, mean_query=None):
    """A layer's (1, H, tokens + CAPACITY, D) keys and values: the recipe's
    block offsets and, with queries, query-aligned spikes in the prompt, as
    strong a logit in a group of any size as the recipe's in one of four."""
    heads, tokens, dim, block = case["heads"], case["tokens"], case["dim"], case["block"]
    blocks = -(-tokens // block)
    rows = blocks * block + CAPACITY
    keys = _normal(gen, (heads, rows, dim))
    prompt = keys[:, :blocks * block].unflatten(1, (blocks, block))
    prompt += 0.5 * _normal(gen, (heads, blocks, 1, dim))
    if mean_query is not None:
        count = round(case["spikes"] * heads * blocks)
        pick = torch.randperm(heads * blocks, generator=gen, device="cuda")[:count]
        spike = torch.zeros(heads * blocks, device="cuda")
        spike[pick] = float(case["group"])
        prompt += spike.view(heads, blocks, 1, 1) * mean_query[:, None, None]
    dtype = DTYPES[case.get("dtype", "bf16")]
    keys = keys[:, :tokens + CAPACITY].to(dtype).unsqueeze(0)
    values = _normal(gen, (heads, tokens + CAPACITY, dim)).to(dtype).unsqueeze(0)
    return keys.contiguous(), values


def _config(case):
    return RefineKVConfig(backend="hip", block_size=case["block"], eps=case.get("eps", 0.01),
                          gqa_reduction=case.get("reduction", "any"),
                          anchor_tokens=case.get("anchors", 0))


def _queries(gen, case, count):
    """A query (H, G, 1, D) and `count` anchor queries (H, G, count, D)."""
    query = _normal(gen, (case["heads"], case["group"], 1, case["dim"]))
    anchors = query + 0.5 * _normal(gen, (case["heads"], case["group"], count, case["dim"]))
    return query.bfloat16(), anchors.bfloat16()


def _layer_inputs(case, gen):
    query, anchors = _queries(gen, case, case["anchors"])
    keys, values = _cache(gen, case, query.float()[:, :, 0].mean(1))
    return query, anchors, keys, values


def prepare(case, seed):
    gen = _gen(seed)
    kind, tokens = case["kind"], case["tokens"]
    state = {"case": case}
    if kind == "summary":
        keys, values = _cache(gen, case)
        state["config"] = _config(case)
        if case["store"]:
            # what attention hands to the cache: rotated keys, and values as a
            # view of the (1, tokens, H, D) projection
            keys = keys[:, :, :tokens].contiguous()
            values = values[:, :, :tokens].transpose(1, 2).contiguous().transpose(1, 2)
            shape = (1, case["heads"], tokens + CAPACITY, case["dim"])
            state["cache"] = [torch.empty(shape, dtype=keys.dtype, device="cuda")
                              for _ in range(2)]
        state["keys"], state["values"] = keys, values
    elif kind == "anchors":
        _, anchors, keys, values = _layer_inputs(case, gen)
        config = _config(case)
        state.update(config=config, queries=anchors, workspace={},
                     summary=build_summary(keys[0, :, :tokens], values[0, :, :tokens], config))
    elif kind == "decode":
        config = _config(case)
        layers = []
        length = torch.tensor(case["suffix"], dtype=torch.int32, device="cuda")
        for _ in range(case["layers"]):
            query, anchors, keys, values = _layer_inputs(case, gen)
            keys, values = keys[0], values[0]
            summary = build_summary(keys[:, :tokens], values[:, :tokens], config)
            workspace, mask = {}, None
            if case["anchors"]:
                mask = select_blocks_union(anchors, summary, config, workspace=workspace)
            end = tokens + (CAPACITY if case["graph"] else case["suffix"])
            layers.append(dict(query=query, summary=summary, key_suffix=keys[:, tokens:end],
                               value_suffix=values[:, tokens:end], anchor_mask=mask,
                               workspace=workspace,
                               suffix_length=length if case["graph"] else None))
        state.update(config=config, layers=layers)
        if case["graph"]:
            # as RefineKV(cuda_graph=True) does: a warm step on a side stream,
            # then one captured step, replayed for each token
            side = torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                _decode_step(state)
            torch.cuda.current_stream().wait_stream(side)
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                state["outputs"] = _decode_step(state)
            state["graph"] = graph
    else:
        layers = []
        for _ in range(case["layers"]):
            query = _normal(gen, (case["heads"], case["group"], case["dim"])).bfloat16()
            shape = (1, case["heads"], tokens + CAPACITY, case["dim"])
            layers.append((query, _normal(gen, shape).bfloat16(), _normal(gen, shape).bfloat16(),
                           {}))
        state["layers"] = layers
    return state


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------

def _decode_step(state):
    results = []
    for layer in state["layers"]:
        result = sparse_attention(layer["query"], layer["summary"], layer["key_suffix"],
                                  layer["value_suffix"], state["config"],
                                  anchor_mask=layer["anchor_mask"], workspace=layer["workspace"],
                                  suffix_length=layer["suffix_length"], return_selected=True)
        results.append((result.output, result.selected))
    return results


def _summary_outputs(summary):
    return dict(keys=summary.keys, values=summary.values, counts=summary.counts,
                key_mean=summary.key_mean, value_mean=summary.value_mean,
                ellipsoid=summary.ellipsoid, value_norm=summary.value_norm,
                max_value_norm=summary.max_value_norm)


def run(state):
    case = state["case"]
    kind, tokens = case["kind"], case["tokens"]
    if kind == "summary":
        if not case["store"]:
            return _summary_outputs(build_summary(state["keys"][0, :, :tokens],
                                                  state["values"][0, :, :tokens],
                                                  state["config"]))
        keys, values = (cache[0, :, :tokens] for cache in state["cache"])
        summary = store_and_build_summary(state["keys"][0], state["values"][0], keys, values,
                                          state["config"])
        return dict(_summary_outputs(summary), cache_keys=keys, cache_values=values)
    if kind == "anchors":
        return select_blocks_union(state["queries"], state["summary"], state["config"],
                                   workspace=state["workspace"])
    if kind == "decode":
        if case["graph"]:
            state["graph"].replay()
            return state["outputs"]
        return _decode_step(state)
    return [dense_decode(query, keys[0], values[0], length=tokens, workspace=workspace)
            for query, keys, values, workspace in state["layers"]]


def work(case):
    heads, dim, tokens = case["heads"], case["dim"], case["tokens"]
    if case["kind"] == "dense":
        one = heads * tokens * dim
        return {"bytes": case["layers"] * one * 4,
                "flops": case["layers"] * one * 4 * case["group"]}
    block = case["block"]
    blocks = -(-tokens // block)
    if case["kind"] == "summary":
        size = DTYPES[case["dtype"]].itemsize
        rows = heads * tokens * dim * 2 * size
        # read once; written to the cache where it is stored, and to the
        # zero-padded pages that the summary holds where blocks are not whole
        moved = rows * (1 + case["store"]) + (heads * blocks * block * dim * 2 * size
                                              if tokens % block else 0)
        return {"bytes": moved + heads * blocks * (3 * dim * 2 + 4),
                "flops": heads * tokens * dim * 10}
    scored = heads * blocks * dim
    if case["kind"] == "anchors":
        return {"bytes": scored * 4 + heads * blocks * 5 + heads * case["group"] * dim * 2
                * case["anchors"],
                "flops": scored * 4 * case["group"] * case["anchors"]}
    # the expanded share is the spikes' at the least
    expanded = int(case["spikes"] * blocks) * block * heads * dim
    representatives = scored - int(case["spikes"] * blocks) * heads * dim
    suffix = heads * case["suffix"] * dim
    return {"bytes": case["layers"] * (scored * 4 + representatives * 2
                                       + (expanded + suffix) * 4 + heads * blocks * 5),
            "flops": case["layers"] * 4 * case["group"] * (scored + expanded + suffix
                                                           + representatives)}


def tolerance(case):
    if case["kind"] == "summary":
        # fp32 sums rounded to bf16: against 64-bit sums one ellipsoid value in
        # a hundred thousand rounds the other way (2.3e-5 of the whole, 0.008
        # at the largest), the fp32 norms differ by 4e-8
        return {"rel": 1e-4, "max": 0.032}
    if case["kind"] == "anchors":
        # a mask bit may differ where a risk equals eps to fp32 rounding
        return {"rel": 0.0, "differ": 2e-5}
    # bf16 outputs of fp32 softmax sums: the two decode paths, which sum in
    # different orders, differ by 2.2e-4 of the whole and 0.0073 at the largest
    return {"rel": 9e-4, "max": 0.03, "differ": 2e-5}


# ---------------------------------------------------------------------------
# The same in 64 bits
# ---------------------------------------------------------------------------

def _pad(x, block):
    heads, tokens, dim = x.shape
    blocks = -(-tokens // block)
    out = x.new_zeros(heads, blocks * block, dim)
    out[:, :tokens] = x
    return out.view(heads, blocks, block, dim)


def _round(x):
    return x.to(torch.bfloat16).double()


def _summary64(keys, values, block):
    """The summary of (H, L, D) keys and values, a head at a time; means and
    widths are rounded to bf16 where the ellipsoid's definition takes the
    stored ones, and returned unrounded beside."""
    tokens = keys.shape[1]
    blocks = -(-tokens // block)
    last = tokens - (blocks - 1) * block
    counts = torch.full((blocks,), block, dtype=torch.int64, device=keys.device)
    counts[-1] = last
    live = torch.arange(block, device=keys.device)[None] < counts[:, None]
    fields = {name: [] for name in ("key_mean", "value_mean", "ellipsoid", "value_norm")}
    for h in range(keys.shape[0]):
        k = _pad(keys[h:h + 1], block)[0].double()
        v = _pad(values[h:h + 1], block)[0].double()
        mean = k.sum(1) / counts[:, None]
        fields["key_mean"].append(mean)
        fields["value_mean"].append(v.sum(1) / counts[:, None])
        mean = _round(mean)
        high = k.masked_fill(~live[..., None], -math.inf).amax(1)
        low = k.masked_fill(~live[..., None], math.inf).amin(1)
        width2 = _round(torch.maximum(high - mean, mean - low).clamp_min(1e-6).square())
        radius2 = ((k - mean[:, None]).square() / width2[:, None]).sum(-1)
        radius2 = radius2.masked_fill(~live, 0.0).amax(1)
        fields["ellipsoid"].append(radius2[:, None] * width2 * INFLATE)
        fields["value_norm"].append(v.square().sum(-1).sqrt().masked_fill(~live, 0.0).amax(1))
    out = {name: torch.stack(x) for name, x in fields.items()}
    out["max_value_norm"] = out["value_norm"].amax(-1)
    out["counts"] = counts
    return out


def _select64(query, summary, case):
    """z (H, G, N) and the mask (H, N) of one query (H, G, D)."""
    q = query.double()
    q2 = _round(q.square())
    scale = case["dim"] ** -0.5
    z = torch.einsum("hgd,hnd->hgn", q, _round(summary["key_mean"])) * scale
    z = z + summary["counts"].double().log()
    spread = torch.einsum("hgd,hnd->hgn", q2, _round(summary["ellipsoid"]))
    delta = spread.clamp_min(0).sqrt() * scale * INFLATE
    log_cosh = delta + torch.log1p(torch.exp(-2 * delta)) - math.log(2)
    log_z = torch.logsumexp(z, -1, keepdim=True)
    log_c = torch.logsumexp(z + log_cosh, -1, keepdim=True)
    # cosh(delta) - 1 = 2 sinh(delta / 2)^2
    half = delta / 2
    log_sinh = half + torch.log(-torch.expm1(-delta)) - math.log(2)
    mass = 2 * summary["max_value_norm"][:, None, None] * torch.exp(
        z - log_c + math.log(2) + 2 * log_sinh)
    risk = mass + 2 * summary["value_norm"][:, None] * torch.exp(z - log_z) * torch.tanh(half)
    if case["reduction"] == "mean":
        return z, risk.mean(1) > case["eps"]
    return z, (risk > case["eps"]).any(1)


def _union64(queries, summary, case):
    mask = None
    for a in range(queries.shape[2]):
        one = _select64(queries[:, :, a], summary, case)[1]
        mask = one if mask is None else mask | one
    return mask


def _attend64(case, query, anchors, keys, values):
    tokens, block = case["tokens"], case["block"]
    summary = _summary64(keys[:, :tokens], values[:, :tokens], block)
    z, mask = _select64(query[:, :, 0], summary, case)
    if case["anchors"]:
        mask = mask | _union64(anchors, summary, case)
    scale = case["dim"] ** -0.5
    of_block = torch.arange(tokens, device=keys.device) // block
    outputs = []
    for h in range(case["heads"]):
        take = torch.cat([mask[h][of_block],
                          torch.ones(case["suffix"], dtype=torch.bool, device=keys.device)])
        end = tokens + case["suffix"]
        k, v = keys[h, :end][take].double(), values[h, :end][take].double()
        logits = torch.cat([z[h][:, ~mask[h]], query[h, :, 0].double() @ k.T * scale], -1)
        v = torch.cat([_round(summary["value_mean"][h][~mask[h]]), v])
        outputs.append(logits.softmax(-1) @ v)
    return torch.stack(outputs).unsqueeze(2), mask


def exact(case, seed):
    gen = _gen(seed)
    kind, tokens = case["kind"], case["tokens"]
    if kind == "summary":
        keys, values = (x[0, :, :tokens] for x in _cache(gen, case))
        out = _summary64(keys, values, case["block"])
        out["keys"], out["values"] = _pad(keys, case["block"]), _pad(values, case["block"])
        if case["store"]:
            out["cache_keys"], out["cache_values"] = keys, values
        return out
    if kind == "anchors":
        _, anchors, keys, values = _layer_inputs(case, gen)
        summary = _summary64(keys[0, :, :tokens], values[0, :, :tokens], case["block"])
        return _union64(anchors, summary, case)
    if kind == "decode":
        results = []
        for _ in range(case["layers"]):
            query, anchors, keys, values = _layer_inputs(case, gen)
            results.append(_attend64(case, query, anchors, keys[0], values[0]))
        return results
    results = []
    for _ in range(case["layers"]):
        query = _normal(gen, (case["heads"], case["group"], case["dim"])).bfloat16()
        shape = (1, case["heads"], tokens + CAPACITY, case["dim"])
        keys, values = _normal(gen, shape).bfloat16()[0], _normal(gen, shape).bfloat16()[0]
        out = []
        for h in range(case["heads"]):
            k, v = keys[h, :tokens].double(), values[h, :tokens].double()
            out.append((query[h].double() @ k.T * case["dim"] ** -0.5).softmax(-1) @ v)
        results.append(torch.stack(out))
    return results
