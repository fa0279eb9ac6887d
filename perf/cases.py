"""The work a serving program has this package do, as timed cases.

A case is one pass through the public entry points: a decode step replayed from
a captured HIP graph, an eager fused NF4 + LoRA linear (decode or prefill), the
row operators, the one-launch LoRA update of a base output, or a weight
dequantisation. Weights are ``N(0, 0.02)`` quantised to NF4 with block 64
(optionally with double-quantised block scales), activations ``N(0, 1)``,
adapters ``N(0, 0.02)`` with scale 2 and 10 % of the tokens without one.
"""

from __future__ import annotations

import math

import torch

NULL_SHARE = 0.1
RAGGED_RANKS = (4, 8, 16, 32, 64)
HIDDEN = 4096


# --------------------------------------------------------------------------
# Cases
# --------------------------------------------------------------------------


def _linear(m, n, k, *, slices=1, adapters=32, rank=16, routes="uniform", quant="fp32", exact=False, swiglu=False, bias=False):
    return dict(kind="linear", m=m, n=n, k=k, slices=slices, adapters=adapters, rank=rank, routes=routes, quant=quant,
                exact=exact, swiglu=swiglu, bias=bias)


def _step(m, inter, kv, *, adapters, rank, quant):
    return dict(kind="step", m=m, inter=inter, kv=kv, adapters=adapters, rank=rank, quant=quant)


def listed():
    return [
        # The smallest call: one token through one square projection with one adapter.
        dict(_linear(1, 4096, 4096, adapters=1), name="linear_1"),
        # Decode steps as a server runs them: the four projections of one block (fused QKV, output,
        # gate/up with SwiGLU, down), captured once per batch size and replayed. One user, a few, a full batch.
        dict(_step(1, 12288, 512, adapters=16, rank=8, quant="dq"), name="step_1"),
        dict(_step(7, 12288, 512, adapters=16, rank=8, quant="dq"), name="step_7"),
        dict(_step(64, 12288, 512, adapters=32, rank=16, quant="fp32"), name="step_64"),
        # A crowded batch over compressed adapters of mixed kept ranks (4..64, written as rank 0), Zipf popularity.
        dict(_linear(256, 4096, 4096, adapters=128, rank=0, routes="zipf"), name="ragged_256"),
        # A short prompt chunk through a merged gate/up projection.
        dict(_linear(300, 24576, 4096, slices=2, adapters=8, rank=16, routes="segments", quant="dq", swiglu=True), name="swiglu_300"),
        # A prefill batch of eight prompts, each with its own adapter.
        dict(_linear(2048, 11008, 4096, adapters=8, rank=32, routes="segments", quant="dq"), name="prefill_2048"),
        # A long prompt through a down projection of the base model, with a bias and no adapters.
        dict(_linear(4096, 4096, 12288, adapters=0, rank=0, bias=True), name="prefill_4096"),
        # Unquantised projections: shrink and expand as two operators over a decode batch ...
        dict(kind="rows", m=64, n=4096, k=4096, slices=1, adapters=32, rank=16, routes="uniform", name="rows_64"),
        # ... and as one update of the base output of a QKV projection over a ragged prompt.
        dict(kind="apply", m=500, n=5120, k=4096, slices=3, adapters=4, rank=16, routes="segments", name="apply_500"),
        # Whole weights back to bf16: a small one, and the largest with double-quantised scales.
        dict(kind="dequant", n=8192, k=1024, quant="fp32", name="dequant_small"),
        dict(kind="dequant", n=24576, k=4096, quant="dq", name="dequant_gate_up"),
    ]


def _between(rng, lo, hi):
    """An integer spread over the logarithm of its range, both ends included."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def _features(rng, lo, hi):
    """A projection width: usually a multiple of 256, now and then only of 64."""
    unit = 64 if rng.random() < 0.25 else 256
    return max(unit, round(_between(rng, lo, hi) / unit) * unit)


def _draw_adapters(rng):
    rank = rng.choice((0, 8, 16, 16, 32, 64))
    adapters = rng.choice((128, 64)) if rank == 0 else rng.choice((1, 4, 8, 16, 32))
    return adapters, rank


def draw(rng):
    kind = rng.choice(("decode", "step", "step", "chunk", "prefill", "prefill", "rows", "apply", "dequant"))
    adapters, rank = _draw_adapters(rng)
    if kind == "step":
        return _step(_between(rng, 1, 64), rng.choice((11008, 12288, 8192)), rng.choice((512, 1024, 4096)),
                     adapters=rng.choice((4, 16, 32)), rank=rng.choice((8, 16, 32)), quant=rng.choice(("fp32", "dq")))
    if kind == "dequant":
        return dict(kind="dequant", n=_features(rng, 512, 24576), k=_features(rng, 512, 4096), quant=rng.choice(("fp32", "dq")))
    if kind in ("rows", "apply"):
        slices = rng.choice((1, 1, 2, 3))
        m = _between(rng, 1, 1024)
        return dict(kind=kind, m=m, n=_features(rng, 1024, 8192), k=_features(rng, 1024, 8192), slices=slices,
                    adapters=adapters, rank=rank, routes=rng.choice(("uniform", "segments")))
    quant = rng.choice(("fp32", "dq"))
    n, k = _features(rng, 1024, 24576), _features(rng, 1024, 12288)
    if kind == "decode":
        exact, quant = rng.random() < 0.25, rng.choice(("fp32", "dq", "nested"))
        return _linear(_between(rng, 1, 64), n, min(k, 8192), slices=rng.choice((1, 1, 3)), adapters=adapters, rank=rank,
                       routes=rng.choice(("uniform", "zipf")), quant=quant, exact=exact, bias=rng.random() < 0.25)
    if kind == "chunk":
        return _linear(_between(rng, 65, 512), n, min(k, 8192), adapters=adapters, rank=rank,
                       routes=rng.choice(("uniform", "zipf", "segments")), quant=quant)
    k = min(k, 6144)
    m = min(_between(rng, 512, 4096), max(512, int(4096 * 4096 * 12288 / (n * k))))
    swiglu = n % 256 == 0 and rng.random() < 0.3
    if rng.random() < 0.25:
        adapters, rank = 0, 0
    return _linear(m, n, k, slices=2 if swiglu else 1, adapters=min(adapters, 16) if rank else 0, rank=rank, routes="segments",
                   quant=quant, swiglu=swiglu, bias=rng.random() < 0.25)


# --------------------------------------------------------------------------
# Inputs
# --------------------------------------------------------------------------


def _dev():
    return torch.device("cuda:0")


def _gen(seed):
    return torch.Generator(device=_dev()).manual_seed(seed)


def _randn(g, *shape, std=1.0):
    return (torch.randn(*shape, generator=g, device=_dev()) * std).bfloat16()


def _weight(g, n, k, quant):
    from loraforge_amd.ops import quantize_nf4

    return quantize_nf4(_randn(g, n, k, std=0.02), compress_statistics=quant != "fp32")


def _ranks(case, cg):
    """Per-adapter ranks (on the host): one rank, or kept ranks drawn from the retained set."""
    if case["rank"]:
        return [case["rank"]] * case["adapters"]
    return [RAGGED_RANKS[i] for i in torch.randint(0, len(RAGGED_RANKS), (case["adapters"],), generator=cg).tolist()]


def _routes(case, cg):
    """int32 slot of every token, on the host (-1: base only)."""
    m, adapters, how = case["m"], case["adapters"], case.get("routes", "uniform")
    if how == "segments":  # contiguous prompts of random lengths, an adapter for each
        parts = min(m, max(1, adapters))
        cuts = torch.sort(torch.randperm(m - 1, generator=cg)[: parts - 1] + 1).values if parts > 1 else torch.empty(0, dtype=torch.int64)
        lengths = torch.diff(torch.cat([torch.tensor([0]), cuts, torch.tensor([m])]))
        return torch.repeat_interleave(torch.arange(parts, dtype=torch.int32), lengths)
    if how == "zipf":
        p = 1.0 / torch.arange(1, adapters + 1, dtype=torch.float64) ** 1.1
        slots = torch.multinomial(p / p.sum(), m, replacement=True, generator=cg).int()
    else:
        slots = torch.randint(0, adapters, (m,), generator=cg, dtype=torch.int32)
    if m > 1:
        slots[torch.rand(m, generator=cg) < NULL_SHARE] = -1
    return slots


def _bounds(n, slices):
    """Output column boundaries of ``slices`` fused projections: even halves, or a QKV-like 3-way split."""
    if slices == 3:
        kv = max(64, n // 10 // 64 * 64)
        return [0, n - 2 * kv, n - kv, n]
    return [0, n] if slices == 1 else [0, n // 2, n]


def _adapters(g, ranks, n, k, bounds, slots):
    """Compact adapter stores: slot g's A is ``[slices * r, K]``, its B ``[N, r]``."""
    from loraforge_amd.ops import LoraBatch

    dev, slices = _dev(), len(bounds) - 1
    r = torch.tensor(ranks, dtype=torch.int64)
    starts = torch.cumsum(r, 0) - r
    i32 = dict(dtype=torch.int32, device=dev)
    return LoraBatch(
        _randn(g, int(r.sum()) * slices * k, std=0.02),
        (starts * slices * k).to(dev),
        _randn(g, int(r.sum()) * n, std=0.02),
        (starts * n).to(dev),
        torch.tensor(ranks, **i32),
        torch.tensor(ranks, **i32),
        torch.full((len(ranks),), 2.0, device=dev),
        slots,
        torch.tensor(bounds, **i32),
        max_rank=max(ranks),
    )


def _segments(slots, rows=16):
    """Tokens grouped by slot into segments of at most ``rows`` tokens (host vectors)."""
    indptr, seg_slots, order = [0], [], []
    for g in sorted(set(slots) - {-1}):
        tokens = [t for t, s in enumerate(slots) if s == g]
        for i in range(0, len(tokens), rows):
            order += tokens[i : i + rows]
            seg_slots.append(g)
            indptr.append(len(order))
    return indptr, seg_slots, order


def _projection(g, cg, m, n, k, slices, case, slots):
    """One quantised projection with its adapters."""
    q, state = _weight(g, n, k, case["quant"])
    ranks = _ranks(case, cg)
    lora = _adapters(g, ranks, n, k, _bounds(n, slices), slots) if ranks else None
    return dict(q=q, state=state, lora=lora, ranks=ranks)


def _inputs(case, seed):
    """Everything a pass reads."""
    g, cg = _gen(seed), torch.Generator().manual_seed(seed)
    s = dict(case=case)
    if case["kind"] == "dequant":
        s["q"], s["state"] = _weight(g, case["n"], case["k"], case["quant"])
        return s
    m = case["m"]
    routes = _routes(case, cg) if case["adapters"] else None
    s["routes"] = None if routes is None else routes.tolist()
    slots = None if routes is None else routes.to(_dev())
    if case["kind"] == "step":
        inter, kv = case["inter"], case["kv"]
        shapes = ((HIDDEN + 2 * kv, HIDDEN, 3), (HIDDEN, HIDDEN, 1), (2 * inter, HIDDEN, 2), (HIDDEN, inter, 1))
        s["x"] = [_randn(g, m, HIDDEN) for _ in range(3)]
        s["layers"] = [_projection(g, cg, m, n, k, slices, case, slots) for n, k, slices in shapes]
        # The fused QKV is split at its real boundaries.
        s["layers"][0]["lora"].slice_offsets = torch.tensor(
            [0, HIDDEN, HIDDEN + kv, HIDDEN + 2 * kv], dtype=torch.int32, device=_dev())
        return s
    n, k = case["n"], case["k"]
    s["x"] = _randn(g, m, k)
    if case["kind"] == "linear":
        s.update(_projection(g, cg, m, n, k, case["slices"], case, slots))
        s["bias"] = _randn(g, n, std=0.5) if case["bias"] else None
        return s
    s["ranks"] = _ranks(case, cg)
    s["y0"] = _randn(g, m, n)
    if case["kind"] == "apply":
        s["lora"] = _adapters(g, s["ranks"], n, k, _bounds(n, case["slices"]), slots)
        return s
    top, slices = max(s["ranks"]), case["slices"]
    s["a"] = _randn(g, case["adapters"], slices * top, k, std=0.02)
    s["lora"] = _adapters(g, s["ranks"], n, 8, _bounds(n, slices), slots)  # its B store and metadata
    return s


# --------------------------------------------------------------------------
# The pass
# --------------------------------------------------------------------------


def _step_pass(s):
    from loraforge_amd.ops import nf4_lora_linear

    qkv, out, up, down = s["layers"]
    a = nf4_lora_linear(s["x"][0], qkv["q"], qkv["state"], lora=qkv["lora"])
    b = nf4_lora_linear(s["x"][1], out["q"], out["state"], lora=out["lora"])
    h = nf4_lora_linear(s["x"][2], up["q"], up["state"], lora=up["lora"], swiglu=True)
    return a, b, h, nf4_lora_linear(h, down["q"], down["state"], lora=down["lora"])


def prepare(case, seed):
    s = _inputs(case, seed)
    dev = _dev()
    if case["kind"] == "step":
        # A server warms a batch size once, captures it and replays the graph from then on.
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _step_pass(s)
        torch.cuda.current_stream().wait_stream(side)
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"], stream=side):
            s["out"] = _step_pass(s)
    elif case["kind"] in ("rows", "apply"):
        s["y"] = s["y0"].clone()
    if case["kind"] == "rows":
        indptr, seg_slots, order = _segments(s["routes"])
        i32 = dict(dtype=torch.int32, device=dev)
        s["z"] = torch.zeros(case["m"], s["a"].shape[1], dtype=torch.bfloat16, device=dev)
        s["segments"] = dict(
            segment_indptr=torch.tensor(indptr, **i32),
            segment_slots=torch.tensor(seg_slots, **i32),
            token_indices=torch.tensor(order, **i32),
            segment_count=torch.tensor([len(seg_slots)], **i32),
        )
    return s


def run(s):
    from loraforge_amd import ops

    case = s["case"]
    kind = case["kind"]
    if kind == "step":
        s["graph"].replay()
        return s["out"]
    if kind == "linear":
        return ops.nf4_lora_linear(
            s["x"], s["q"], s["state"], scales="nested" if case["quant"] == "nested" else None, bias=s["bias"], lora=s["lora"],
            exact=case["exact"], swiglu=case["swiglu"])
    if kind == "dequant":
        if case["quant"] == "fp32":
            return ops.dequantize_nf4(s["q"], s["state"].absmax, s["state"].code, (case["n"], case["k"]))
        return ops.dequantize_nf4_nested(s["q"], s["state"])
    # The base output that the adapters update is new in every pass.
    y, lora = s["y"].copy_(s["y0"]), s["lora"]
    if kind == "apply":
        return ops.lora_apply(s["x"], y, lora)
    ops.row_shrink(s["x"], s["a"], s["z"], lora.token_slots, lora.ranks, num_slices=case["slices"], max_rank=lora.max_rank)
    ops.row_expand(
        s["z"], lora.b_store, y, b_offsets=lora.b_offsets, b_strides=lora.b_strides, ranks=lora.ranks, scales=lora.scales,
        slice_offsets=lora.slice_offsets, **s["segments"])
    return s["z"], y


# --------------------------------------------------------------------------
# Work, tolerance and the values in 64 bits
# --------------------------------------------------------------------------


def _adapters_used(case):
    """Expected number of distinct adapters that a batch routes to."""
    m, adapters, how = case["m"], case["adapters"], case.get("routes", "uniform")
    if how == "segments":
        return min(m, adapters)
    p = [1.0 / i**1.1 if how == "zipf" else 1.0 for i in range(1, adapters + 1)]
    live, total = (1 - NULL_SHARE if m > 1 else 1.0), sum(p)
    return sum(1 - (1 - live * v / total) ** m for v in p)


def _mean_rank(case):
    return case["rank"] or sum(RAGGED_RANKS) / len(RAGGED_RANKS)


def _lora_work(case, n, k, slices):
    if not case["adapters"]:
        return 0, 0
    r = _mean_rank(case)
    live = case["m"] * (1.0 if case["m"] == 1 or case.get("routes") == "segments" else 1 - NULL_SHARE)
    return _adapters_used(case) * 2 * r * (slices * k + n), live * 2 * r * (slices * k + n)


def _weight_bytes(n, k, quant):
    return n * k // 2 + (n * k // 16 if quant == "fp32" else n * k // 64 + n * k // 4096)


def work(case):
    if case["kind"] == "dequant":
        return {"bytes": _weight_bytes(case["n"], case["k"], case["quant"]) + 2 * case["n"] * case["k"], "flops": 0}
    m = case["m"]
    if case["kind"] == "step":
        inter, kv = case["inter"], case["kv"]
        shapes = ((HIDDEN + 2 * kv, HIDDEN, 3, HIDDEN + 2 * kv), (HIDDEN, HIDDEN, 1, HIDDEN), (2 * inter, HIDDEN, 2, inter),
                  (HIDDEN, inter, 1, HIDDEN))
    else:
        n = case["n"]
        shapes = ((n, case["k"], case["slices"], n // 2 if case.get("swiglu") else n),)
    moved = flops = 0
    for n, k, slices, width in shapes:
        b, f = _lora_work(case, n, k, slices)
        moved += b + 2 * m * k + 2 * m * width
        flops += f
        if case["kind"] in ("step", "linear"):
            moved += _weight_bytes(n, k, case["quant"])
            flops += 2 * m * n * k
        else:
            moved += 2 * m * n  # the base output, read before it is written
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    if case["kind"] == "dequant":
        return "exact"
    # bf16 results of fp32 sums, about four times their distance from 64 bits: 0.0018 for the row
    # operators; 0.0032 for a linear, whose decode kernels round the codebook instead of each weight;
    # 0.0044 through SwiGLU; 0.0064 where the down projection follows it.
    if case["kind"] in ("rows", "apply"):
        return {"rel": 0.007}
    if case["kind"] == "step":
        return {"rel": 0.025}
    return {"rel": 0.018 if case["swiglu"] else 0.0125}


def _dequantised(q, state):
    """The weight the packed state stands for: bf16 of codebook value times block scale, as [N, K] in fp64."""
    q = q.reshape(-1)
    nib = torch.stack((q >> 4, q & 15), 1).reshape(-1).long()
    if state.state2 is None:
        scales = state.absmax
    else:
        two = state.state2
        scales = two.code[state.absmax.long()] * two.absmax.repeat_interleave(two.blocksize)[: state.absmax.numel()] + state.offset
    w = (state.code[nib].reshape(-1, 64) * scales.reshape(-1, 1)).bfloat16()
    return w.reshape(tuple(state.shape))


def _delta(x, lora, routes, ranks, n):
    """The LoRA update of every token in fp64; ``x`` fp64 [M, K]."""
    k = x.shape[1]
    y = torch.zeros(x.shape[0], n, dtype=torch.float64, device=x.device)
    bounds = lora.slice_offsets.tolist()
    slices = len(bounds) - 1
    a_at, b_at = lora.a_offsets.tolist(), lora.b_offsets.tolist()
    for g in sorted(set(routes) - {-1}):
        r = ranks[g]
        rows = torch.tensor([t for t, s in enumerate(routes) if s == g], device=x.device)
        a = lora.a_store[a_at[g] : a_at[g] + slices * r * k].reshape(slices, r, k).double()
        b = lora.b_store[b_at[g] : b_at[g] + n * r].reshape(n, r).double()
        for i in range(slices):
            z = x[rows] @ a[i].t()
            y[rows, bounds[i] : bounds[i + 1]] = 2.0 * (z @ b[bounds[i] : bounds[i + 1]].t())
    return y


def _linear_exact(x, p, routes, bias=None, swiglu=False):
    w = _dequantised(p["q"], p["state"])
    y = torch.cat([x @ part.double().t() for part in w.split(4096)], 1)
    if bias is not None:
        y += bias.double()
    if p["lora"] is not None:
        y += _delta(x, p["lora"], routes, p["ranks"], y.shape[1])
    if swiglu:
        gate, up = y.chunk(2, 1)
        y = gate * torch.sigmoid(gate) * up
    return y


def exact(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]
    if kind == "dequant":
        return _dequantised(s["q"], s["state"]).double()
    if kind == "step":
        x = [t.double() for t in s["x"]]
        qkv, out, up, down = s["layers"]
        h = _linear_exact(x[2], up, s["routes"], swiglu=True)
        return (_linear_exact(x[0], qkv, s["routes"]), _linear_exact(x[1], out, s["routes"]), h,
                _linear_exact(h, down, s["routes"]))
    x = s["x"].double()
    if kind == "linear":
        return _linear_exact(x, s, s["routes"], s["bias"], case["swiglu"])
    if kind == "apply":
        return s["y0"].double() + _delta(x, s["lora"], s["routes"], s["ranks"], case["n"])
    # rows: z holds slices * r columns of the token's adapter, the rest stays zero.
    slices, lora, y = case["slices"], s["lora"], s["y0"].double()
    z = torch.zeros(case["m"], s["a"].shape[1], dtype=torch.float64, device=x.device)
    bounds, b_at = lora.slice_offsets.tolist(), lora.b_offsets.tolist()
    for g in sorted(set(s["routes"]) - {-1}):
        r = s["ranks"][g]
        t = torch.tensor([i for i, v in enumerate(s["routes"]) if v == g], device=x.device)
        z[t, : slices * r] = x[t] @ s["a"][g, : slices * r].double().t()
        b = lora.b_store[b_at[g] : b_at[g] + case["n"] * r].reshape(-1, r).double()
        for i in range(slices):
            cols = slice(bounds[i], bounds[i + 1])
            y[t, cols] += 2.0 * (z[t, i * r : (i + 1) * r] @ b[cols].t())
    return z, y
