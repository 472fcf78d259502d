"""The work that users of this package have it do, as timed cases.

- ``decode``: one decode step over a compressed cache: the per-step decode of the packed codes and every layer's
  attention over them, for one conversation or a ragged batch, bit planes or ladder codes.  ``via`` says how the
  program calls it: ``graph`` replays a captured step (a serving loop at a fixed length), ``calls`` makes the
  library's calls with argument blocks built once, ``hook`` goes through ``CompressedContext.attend`` as a Hugging
  Face model's attention does, layer by layer.
- ``score``: a question scored over the codes with its first planes (the ``prog@`` entry point's importance).
- ``project``: the PCA projection of a prefill cache (the coefficients both codecs quantize).
- ``encode``: ``ProgressiveCodec.encode``, a prefill cache to packed planes under a byte budget.
- ``compress``: ``KVTCCodec.compress``, a prefill cache to per-token rungs and the caches rebuilt from them.
- ``restore``: ``kvtc_storage.decode_bytes``, stored bytes on the host to FP16 caches on the GPU.

Caches are synthetic: an i^-1.5 PCA spectrum scaled to unit-variance features, so that the attention scores have
the spread of a trained model's rather than none.  Everything but the package's own plans is made by plain torch
from the seed, and ``exact`` repeats the arithmetic in float64 from the same inputs.
"""

import math
import os
import sys
import types

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for _p in (ROOT, os.path.join(ROOT, "dimmer-kv_amd")):
    if _p not in sys.path:
        sys.path.insert(0, _p)

DEV = "cuda"
GROUP, SINKS, RECENT = 64, 4, 32
KINDS = ("key", "value")
DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
# layers, KV heads, head_dim, query heads, rank of the two model shapes this package is used with
SHAPES = {"1b": (16, 8, 64, 32, 1024), "3b": (28, 8, 128, 24, 2048)}


def _decode(name, shape, tokens, **more):
    layers, kv, dim, heads, rank = SHAPES[shape]
    case = dict(name=name, kind="decode", layers=layers, kv_heads=kv, head_dim=dim, q_heads=heads, rank=rank,
                tokens=tokens, batch=1, spread=1, q_len=1, format="planes", drop=0.12, dtype="bf16", via="calls")
    case.update(more)
    return case


def _codec(name, kind, shape, tokens, **more):
    layers, kv, dim, heads, rank = SHAPES[shape]
    case = dict(name=name, kind=kind, layers=layers, kv_heads=kv, head_dim=dim, q_heads=heads, rank=rank,
                tokens=tokens, dtype="f16")
    case.update(more)
    return case


def listed():
    return [
        # a short chat on a small model: the step is a chain of small launches, so launch latency decides
        _decode("decode-1b-1500", "1b", 1500, drop=0.5, dtype="f32", via="graph"),
        # one document's answer on a small model at the 2-plane floor, called without a graph
        _decode("decode-1b-8k", "1b", 8192, drop=0.95),
        # the headline: a 16K-token conversation on the larger model, 3 % budget, replayed step
        _decode("decode-3b-16k", "3b", 16384, via="graph"),
        # ladder codes answered through a model's attention hook, at a length that fills no tile
        _decode("hook-3b-6k-ladder", "3b", 6001, format="ladder", dtype="f16", via="hook"),
        # a serving batch: 32 conversations of 2K-16K tokens in one fused step
        _decode("decode-3b-ragged-32", "3b", 16384, batch=32, spread=8),
        # the question's own forward: 64 new tokens attend over the long cache through the hook
        _decode("question-3b-16k", "3b", 16384, q_len=64, via="hook"),
        # a short question over a short cache, odd sizes
        _decode("question-1b-3k", "1b", 3001, q_len=13, drop=0.5, dtype="f16", via="hook"),
        # the refinement's question scoring at full size, first two planes
        _decode("score-3b-16k", "3b", 16384, q_len=64) | {"kind": "score", "cap": 2},
        # the projection of a 16K-token prefill's keys (de-rotated, centred, onto the basis)
        _codec("project-3b-16k", "project", "3b", 16384),
        # a whole progressive encode of a medium context, an odd length
        _codec("encode-1b-8k", "encode", "1b", 8191, budget=0.04, floor=1),
        # per-token rungs and rebuilt caches of a medium context
        _codec("compress-3b-4k", "compress", "3b", 4097, budget=0.03),
        # a stored cache read back
        _codec("restore-3b-6k", "restore", "3b", 6000),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the ranges above: either model shape or a few-layer slice of it, any length up to the
    listed ones', every query type, code format and way of calling."""
    shape = rng.choice(["1b", "3b"])
    layers = SHAPES[shape][0]
    kind = rng.choice(["decode"] * 4 + ["question"] * 2 + ["score", "project", "encode", "compress", "restore"])
    few = rng.choice([layers, rng.randint(2, layers)])
    if kind in ("decode", "question", "score"):
        case = _decode("", shape, _log(rng, 300, 16384), layers=few, dtype=rng.choice(sorted(DTYPES)),
                       drop=rng.uniform(0.1, 0.95), via=rng.choice(["graph", "calls", "hook"]))
        if rng.random() < 0.3:
            case["rank"] = 256 * rng.randint(1, case["rank"] // 256)
        if kind == "decode":
            case["q_len"] = rng.choice([1, 1, 1, 1, 2, 3])
            case["format"] = rng.choice(["planes", "planes", "ladder"])
            if case["q_len"] == 1 and case["via"] != "hook" and rng.random() < 0.4:
                case.update(batch=rng.randint(2, 24), spread=rng.choice([1, 4, 8]))
        else:
            case.update(q_len=rng.randint(4, 64), via="hook")
            if kind == "score":
                case.update(kind="score", cap=rng.choice([1, 2, 2, 8]), via="calls")
    else:
        top = {"project": 16384, "encode": 8191, "compress": 4097, "restore": 6000}[kind]
        case = _codec("", kind, shape, _log(rng, 512, top), layers=few)
        if kind == "project":
            case["dtype"] = rng.choice(sorted(DTYPES))
        if kind in ("encode", "compress"):
            # bytes per compressed token and 64-group (3 to 6.5 planes, or the ladder's middle rungs), and the exact tokens
            full, groups = 2 * _features(case), case["rank"] // GROUP
            size = groups * (rng.uniform(28, 56) if kind == "encode" else rng.uniform(26, 48))
            case["budget"] = round((size + 4) / full + (SINKS + RECENT) / case["tokens"], 4)
        if kind == "encode":
            case["floor"] = rng.choice([0, 1])
    case.pop("name")
    return case


# ----------------------------------------------------------------- inputs (plain torch, from the seed alone)

def _gen(seed):
    return torch.Generator(DEV).manual_seed(int(seed) * 7919 + 17)


def _features(case):
    return case["layers"] * case["kv_heads"] * case["head_dim"]


def _scale(case):
    """Component standard deviations: eigenvalues i^-1.5, scaled so that a feature of coef @ basis^T has variance 1."""
    s = torch.arange(1, case["rank"] + 1, device=DEV, dtype=torch.float64).pow(-0.75)
    return (s * math.sqrt(_features(case)) / s.square().sum().sqrt()).float()


def _tables(case, g):
    """Per stream a basis [features, rank] with columns of about unit norm and a mean [features]."""
    f, r = _features(case), case["rank"]
    basis = {k: torch.randn(f, r, generator=g, device=DEV) / math.sqrt(f) for k in KINDS}
    mean = {k: 0.3 * torch.randn(f, generator=g, device=DEV) for k in KINDS}
    return basis, mean


def _rope(case, tokens):
    """float32 cos, sin [tokens, head_dim] (theta 500,000)."""
    d = case["head_dim"]
    inv = 500000.0 ** (-torch.arange(0, d, 2, device=DEV, dtype=torch.float64) / d)
    angle = torch.arange(tokens, device=DEV, dtype=torch.float64)[:, None] * inv[None]
    angle = torch.cat([angle, angle], dim=1)
    return angle.cos().float(), angle.sin().float()


def _lengths(case):
    """Tokens of each conversation of a batch: from tokens / spread to tokens, evenly spread, no two alike."""
    b, top = case["batch"], case["tokens"]
    if b == 1:
        return [top]
    low = max(64, top // case["spread"])
    return [int(low + (top - low) * ((i * 19) % b) / (b - 1)) - i % 5 for i in range(b)]


def _coefficients(case, n, g):
    return torch.randn(n, case["rank"], generator=g, device=DEV) * _scale(case)


def _plane_codes(case, n, g):
    """8-bit codes, fp16 low and span per 64-group, and plane counts: 5 % of the tokens none, the others 2 and more."""
    x = _coefficients(case, n, g).view(n, -1, GROUP)
    low = x.amin(2).half()
    span = (x.amax(2) - low.float()).half()
    code = ((x - low.float()[..., None]) / span.float()[..., None] * 256).floor().clamp(0, 255).to(torch.uint8)
    u = torch.rand(n, generator=g, device=DEV).clamp_min(1e-9)
    planes = 2 + (u.log() / math.log1p(-case["drop"])).floor().clamp(0, 6).long()
    planes[torch.rand(n, generator=g, device=DEV) < 0.05] = 0
    return code, low, span, planes


def _rungs(groups):
    """The bit-width ladder [8, groups] over {0, 2, 4, 8}: finer rungs give more of the leading groups more bits."""
    rows = []
    for r in range(1, 9):
        n8, n4, n2 = groups * r // 16, groups * r // 8, groups * r // 4
        rows.append(([8] * n8 + [4] * n4 + [2] * n2 + [0] * groups)[:groups])
    return torch.tensor(rows, dtype=torch.long)


def _rung_bytes(rungs):
    return [int((row * GROUP // 8).sum() + 4 * (row > 0).sum()) for row in rungs]


def _ladder_quantize(x, widths, dtype):
    """x [n, G, 64] at per-(token, group) ``widths``: levels, fp16 shift and scale (the ladder's definition)."""
    top = (2.0 ** widths.to(dtype) - 1)
    low = x.amin(2).to(torch.float32).half()
    step = ((x.amax(2) - low.to(dtype)) / top.clamp_min(1)).clamp_min(1e-8).to(torch.float32).half()
    level = ((x - low.to(dtype)[..., None]) / step.to(dtype)[..., None]).round()
    level = torch.minimum(level.clamp_min(0), top[..., None])
    coded = widths > 0
    return level * coded[..., None], low * coded, step * coded


def _ladder_codes(case, n, g):
    x = _coefficients(case, n, g).view(n, -1, GROUP)
    rung = torch.randint(2, 7, (n,), generator=g, device=DEV)
    widths = _rungs(case["rank"] // GROUP).to(DEV)[rung]
    level, low, step = _ladder_quantize(x, widths, torch.float32)
    return level.to(torch.uint8), low, step, rung


def _decode_inputs(case, seed):
    g = _gen(seed)
    dt, q_len, layers, kv, d = (case[k] for k in ("dtype", "q_len", "layers", "kv_heads", "head_dim"))
    lengths = _lengths(case)
    basis, mean = _tables(case, g)
    middle = [max(0, n - SINKS - RECENT) for n in lengths]
    codes = {k: (_plane_codes if case["format"] == "planes" else _ladder_codes)(case, sum(middle), g) for k in KINDS}
    exact = [n - m + q_len for n, m in zip(lengths, middle)]
    cache = torch.float32 if case["via"] != "hook" else DTYPES[dt]
    ke, ve = (torch.randn(layers, kv, sum(exact), d, generator=g, device=DEV).to(cache) for _ in KINDS)
    q = (1.5 * torch.randn(layers, case["batch"], case["q_heads"], q_len, d, generator=g, device=DEV)).to(DTYPES[dt])
    positions = torch.cat([torch.arange(SINKS, SINKS + m, device=DEV, dtype=torch.int32) for m in middle])
    mask = None
    if q_len > 1:  # the new tokens are causal among themselves, the other exact tokens seen by all
        mask = torch.zeros(q_len, exact[0], device=DEV)
        mask[:, exact[0] - q_len:] = torch.full((q_len, q_len), float("-inf"), device=DEV).triu(1)
    return types.SimpleNamespace(basis=basis, mean=mean, middle=middle, exact=exact, codes=codes, ke=ke, ve=ve, q=q,
                                 positions=positions, mask=mask, rope=_rope(case, max(lengths) + q_len))


def _cache_inputs(case, seed):
    """A prefill cache (per layer [1, kv_heads, tokens, head_dim], keys rotated), its calibration and weights."""
    g = _gen(seed)
    n, layers, kv, d = case["tokens"], case["layers"], case["kv_heads"], case["head_dim"]
    basis, mean = _tables(case, g)
    cos, sin = _rope(case, n)
    caches = {}
    for k in KINDS:
        x = _coefficients(case, n, g) @ basis[k].T + mean[k] + 0.05 * torch.randn(n, _features(case), generator=g, device=DEV)
        x = x.view(n, layers, kv, d)
        caches[k] = []
        for layer in range(layers):
            t = x[:, layer].transpose(0, 1)
            if k == "key":
                t = t * cos + torch.cat([-t[..., d // 2:], t[..., :d // 2]], -1) * sin
            caches[k].append(t.to(DTYPES[case["dtype"]])[None].contiguous())
    return types.SimpleNamespace(basis=basis, mean=mean, caches=caches, rope=(cos, sin),
                                 weights=torch.rand(n, generator=g, device=DEV) + 0.1)


def _restore_inputs(case, seed):
    """A stored cache as bytes: int32 header, then per stream the rung ids, each rung's codes, shifts and scales
    by width (or fp16 rows for the exact rung), and the exact tokens' fp16 rows."""
    g = _gen(seed)
    n, f, groups = case["tokens"], _features(case), case["rank"] // GROUP
    basis, mean = _tables(case, g)
    start, end = SINKS, n - RECENT
    rungs = _rungs(groups)
    scale = _scale(case).view(groups, GROUP)
    parts = [np.asarray([n, start, end], "<i4").tobytes()]
    kept = {}

    def add(t):
        parts.append(t.contiguous().view(torch.uint8).cpu().numpy().tobytes())
        return t

    for k in KINDS:
        rung = torch.randint(2, 7, (end - start,), generator=g, device=DEV)
        rung[torch.rand(end - start, generator=g, device=DEV) < 0.002] = len(rungs)
        add(rung.to(torch.uint8))
        sections = []
        for r in rung.unique().tolist():
            count = int((rung == r).sum())
            if r == len(rungs):
                sections.append((r, 0, None, add(torch.randn(count, f, generator=g, device=DEV).half())))
                continue
            for width in (2, 4, 8):
                cols = (rungs[r] == width).nonzero().flatten().to(DEV)
                if cols.numel():
                    raw = add(torch.randint(0, 256, (count, cols.numel(), 8 * width), generator=g, device=DEV,
                                            dtype=torch.uint8))
                    spread = scale[cols].mean(1) * (0.8 + 0.4 * torch.rand(count, cols.numel(), generator=g, device=DEV))
                    low = add((-2.5 * spread).half())
                    sections.append((r, width, cols, (raw, low, add((5 * spread / (2 ** width - 1)).half()))))
        kept[k] = (rung, sections, add(torch.randn(n - end + start, f, generator=g, device=DEV).half()))
    return types.SimpleNamespace(basis=basis, mean=mean, data=b"".join(parts), kept=kept, rungs=rungs, span=(start, end))


def _calibration(case, i):
    rungs = _rungs(case["rank"] // GROUP)
    return {"model": "synthetic", "layers": case["layers"], "heads": case["kv_heads"], "head_dim": case["head_dim"],
            "group": GROUP, "sinks": SINKS,
            **{k: {"mean": i.mean[k], "basis": i.basis[k], "rungs": rungs, "rung_bytes": _rung_bytes(rungs)} for k in KINDS}}


def _order(groups):
    """Every group's first plane, then every group's second, ...; rungs at whole planes."""
    planes = torch.tensor([[(p + groups - 1 - g) // groups for g in range(groups)] for p in range(8 * groups + 1)],
                          dtype=torch.uint8)
    sizes = 8.0 * planes.double().sum(1) + 4.0 * (planes > 0).double().sum(1)
    entry = {"planes": planes, "prefix_bytes": sizes, "rungs": [groups * m for m in range(1, 9)]}
    return {"model": "synthetic", "key": dict(entry), "value": dict(entry)}


def _model(case):
    """What the codecs take of a model: its rotary embedding and its head count."""
    def rotary(x, positions):
        cos, sin = _rope(case, int(positions.shape[1]))
        return cos[None], sin[None]

    return types.SimpleNamespace(model=types.SimpleNamespace(rotary_emb=rotary),
                                 config=types.SimpleNamespace(num_attention_heads=case["q_heads"]))


# ----------------------------------------------------------------- prepare and run

def prepare(case, seed):
    kind = case["kind"]
    if kind in ("decode", "score"):
        return _prepare_decode(case, seed)
    state = types.SimpleNamespace(case=case)
    if kind == "restore":
        from kvtc import KVTCCodec
        i = _restore_inputs(case, seed)
        state.codec, state.data = KVTCCodec(_calibration(case, i), DEV, _model(case)), i.data
        return state
    i = _cache_inputs(case, seed)
    state.caches, state.weights, state.rope = i.caches, i.weights, i.rope
    if kind == "compress":
        from kvtc import KVTCCodec
        state.codec = KVTCCodec(_calibration(case, i), DEV, _model(case))
    else:
        from progressive import ProgressiveCodec
        state.codec = ProgressiveCodec(_calibration(case, i), _order(case["rank"] // GROUP), DEV, _model(case))
    return state


def _prepare_decode(case, seed):
    import synth
    from compressed_attention import CompressedContext, ModelTables
    from hot_tier import LadderStream, LadderTables, OrderTables, PackedStream
    from workloads import DecodeWorkload, QuestionStage

    i = _decode_inputs(case, seed)
    layers, kv, d, heads, rank = (case[k] for k in ("layers", "kv_heads", "head_dim", "q_heads", "rank"))
    groups = rank // GROUP
    streams = {}
    if case["format"] == "planes":
        order = _order(groups)["key"]
        table = OrderTables(order["planes"], order["prefix_bytes"], DEV)
        for k in KINDS:
            code, low, span, planes = i.codes[k]
            streams[k] = PackedStream.pack(code, low, span, planes * groups, table, with_cold=False)
    else:
        rungs = _rungs(groups)
        table = LadderTables(rungs, _rung_bytes(rungs), DEV)
        for k in KINDS:
            streams[k] = LadderStream.pack(*i.codes[k], table)
    tables = ModelTables(i.basis["key"], i.basis["value"], i.mean["key"], i.mean["value"], layers, kv, d, *i.rope)
    cu = torch.tensor(np.concatenate([[0], np.cumsum(i.middle)]), dtype=torch.int32)
    context = CompressedContext(tables, streams["key"], streams["value"], i.positions, heads, cu_seqlens=cu)
    state = types.SimpleNamespace(case=case, context=context)
    if case["kind"] == "score":
        past = i.exact[0] - case["q_len"]
        w = types.SimpleNamespace(shape=synth.ModelShape(layers, kv, d, heads, rank), context=context, streams=streams)
        state.question = QuestionStage(w, i.q, i.ke[:, :, :past].contiguous(), i.ke[:, :, past:].contiguous(), 0.01,
                                       plane_cap=case["cap"])
        return state
    if case["via"] == "hook":
        state.q, state.ke, state.ve = i.q, i.ke[:, None], i.ve[:, None]
        state.mask = None if i.mask is None else i.mask[None, None].to(i.q.dtype)
        state.modules = [types.SimpleNamespace(layer_idx=l, num_key_value_groups=heads // kv) for l in range(layers)]
        return state
    outs = torch.empty(layers, case["batch"], case["q_len"], heads, d, dtype=i.q.dtype, device=DEV)
    w = DecodeWorkload("decode", synth.ModelShape(layers, kv, d, heads, rank), context, tables, streams, i.q, i.ke, i.ve,
                       outs, exact_lengths=tuple(i.exact), batch=case["batch"], q_len=case["q_len"])
    w.args = [context.layer_args(l, i.q[l], outs[l], i.ke[l], i.ve[l], i.mask, tuple(i.exact)) for l in range(layers)]
    w.workspace = context.workspace(w.args[0])
    state.work, state.mask = w, i.mask  # the argument blocks hold the mask's address
    if case["via"] == "graph":
        w.capture()
    return state


def run(s):
    case = s.case
    kind = case["kind"]
    if kind == "decode":
        if case["via"] == "graph":
            s.work.graph.replay()
            return s.work.outs
        if case["via"] == "calls":
            s.work.step()
            return s.work.outs
        scaling = case["head_dim"] ** -0.5
        return [s.context.attend(m, s.q[l], s.ke[l], s.ve[l], s.mask, scaling)[0] for l, m in enumerate(s.modules)]
    if kind == "score":
        return s.question.score()
    if kind == "project":
        return s.codec.stream_coefficients("key", s.caches["key"], *s.rope, SINKS, case["tokens"] - RECENT)
    if kind == "encode":
        cache = s.codec.encode(s.caches["key"], s.caches["value"], case["budget"], RECENT, floor_rung=case["floor"])
        out = {"errors": s.codec.last_errors}
        for k in KINDS:
            codes, low, span = s.codec.last_quantized[k]
            out[k] = {"codes": codes, "low": low, "span": span, "pieces": cache.stores[k].packed.pieces}
        return out
    if kind == "compress":
        keys, values, _, _ = s.codec.compress(s.caches["key"], s.caches["value"], case["budget"], RECENT, True,
                                              weights=s.weights, floor_share=1.0)
        return {"keys": keys, "values": values, "choice": [s.codec.last_choice[k] for k in KINDS]}
    import kvtc_storage
    keys, values = kvtc_storage.decode_bytes(s.codec, s.data)
    return {"keys": keys, "values": values}


# ----------------------------------------------------------------- what a pass cannot do without, and how exact it is

def work(case):
    f, r, layers, d = _features(case), case["rank"], case["layers"], case["head_dim"]
    groups, width, basis = r // GROUP, case["kv_heads"] * d, f * r * 2
    if case["kind"] in ("decode", "score"):
        lengths = _lengths(case)
        n = sum(max(0, t - SINKS - RECENT) for t in lengths)
        rows = case["q_heads"] * case["q_len"]
        size = 2 if case["dtype"] != "f32" else 4
        planes = sum((2 + e) * ((1 - case["drop"]) ** e * (case["drop"] if e < 6 else 1)) for e in range(7))
        if case["kind"] == "score":
            planes = min(planes, case["cap"])
        code = groups * 0.95 * (4 + 8 * planes)
        if case["format"] == "ladder":
            code = sum(_rung_bytes(_rungs(groups))[2:7]) / 5
        query = layers * case["batch"] * rows * d * size
        exact = 2 * layers * width * (36 + case["q_len"]) * case["batch"] * (size if case["via"] == "hook" else 4)
        keys = 2 * n * f * r + 2 * n * layers * rows * d
        if case["kind"] == "score":
            return {"bytes": n * code + basis + query + exact / 2 + 4 * n, "flops": keys}
        return {"bytes": 2 * n * code + 2 * basis + 2 * query + exact,
                "flops": keys + 2 * n * layers * rows * r + 2 * layers * case["batch"] * rows * r * d}
    n = case["tokens"] - SINKS - RECENT
    cache = case["tokens"] * f * (4 if case["dtype"] == "f32" else 2)
    project = 2 * n * f * r
    if case["kind"] == "project":
        return {"bytes": cache + 4 * f * r + 4 * n * r, "flops": project}
    if case["kind"] == "encode":
        return {"bytes": 2 * (cache + 4 * f * r + n * (r + 4 * groups + 32)), "flops": 2 * project}
    if case["kind"] == "compress":
        return {"bytes": 2 * (2 * cache + 4 * f * r), "flops": 4 * project}
    stored = n * sum(_rung_bytes(_rungs(groups))[2:7]) / 5
    return {"bytes": 2 * (stored + 4 * f * r + cache), "flops": 2 * project}


def tolerance(case):
    """About four times each kind's measured distance from ``exact``."""
    kind = case["kind"]
    if kind == "decode":  # fp16 operands (5e-4), then the query type's rounding of the output (1.8e-3 in bf16)
        return {"rel": 7e-3 if case["dtype"] == "bf16" else 3e-3, "max": 0.05}
    if kind == "score":  # fp16 keys and probabilities (5e-4)
        return {"rel": 2e-3, "max": 0.02}
    if kind == "project":  # float32 sums of up to 28,672 products (2.5e-6)
        return {"rel": 1e-5, "max": 1e-4}
    if kind == "encode":  # a code, plane count or fp16 bound on an edge may fall either way (7e-5 in the errors)
        return {"rel": 3e-4, "max": 0.05, "differ": 5e-3}
    if kind == "compress":  # FP16 caches; a token on the edge of a rung, or a level on the edge of a code, as well
        return {"rel": 3e-3, "max": 0.99, "differ": 5e-3}
    return {"rel": 1e-3, "max": 1e-2}  # FP16 caches


# ----------------------------------------------------------------- the same in float64

def _rotate(x, cos, sin):
    half = x.shape[-1] // 2
    return x * cos + torch.cat([-x[..., half:], x[..., :half]], -1) * sin


def _plane_values(codes, cap=8):
    code, low, span, planes = codes
    m = planes.clamp_max(cap)[:, None, None]
    idx = code.long() >> (8 - m)
    value = low.double()[..., None] + (idx.double() + 0.5) * span.double()[..., None] / 2.0 ** m
    return torch.where(m > 0, value, 0.0).flatten(1)


def _ladder_values(codes):
    level, low, step, _ = codes
    return (level.double() * step.double()[..., None] + low.double()[..., None]).flatten(1)


def _layer(x, case, layer):
    width = case["kv_heads"] * case["head_dim"]
    return x[layer * width:(layer + 1) * width].double()


def _exact_attention(case, seed):
    i = _decode_inputs(case, seed)
    kv, d, q_len, heads = case["kv_heads"], case["head_dim"], case["q_len"], case["q_heads"]
    cap = case.get("cap", 8)
    coef = {k: _plane_values(i.codes[k], cap) if case["format"] == "planes" else _ladder_values(i.codes[k]) for k in KINDS}
    i.codes.clear()
    cos, sin = (t[i.positions.long()].double()[:, None] for t in i.rope)
    cu, ce = np.concatenate([[0], np.cumsum(i.middle)]), np.concatenate([[0], np.cumsum(i.exact)])
    outs, importance = [], torch.zeros(sum(i.middle), device=DEV, dtype=torch.float64)
    for layer in range(case["layers"]):
        keys = coef["key"] @ _layer(i.basis["key"], case, layer).T + _layer(i.mean["key"], case, layer)
        keys = _rotate(keys.view(-1, kv, d), cos, sin)
        bv, mv = _layer(i.basis["value"], case, layer).view(kv, d, -1), _layer(i.mean["value"], case, layer).view(kv, 1, d)
        out = torch.empty(case["batch"], q_len, heads, d, device=DEV, dtype=torch.float64)
        for b in range(case["batch"]):
            at, ex = slice(int(cu[b]), int(cu[b + 1])), slice(int(ce[b]), int(ce[b + 1]))
            q = i.q[layer, b].double().reshape(kv, -1, d)  # a KV head's query heads, each q_len rows
            s = torch.cat([torch.bmm(q, keys[at].permute(1, 2, 0).contiguous()),
                           torch.bmm(q, i.ke[layer, :, ex].double().transpose(1, 2).contiguous())], -1) * d ** -0.5
            m = i.middle[b]
            if i.mask is not None:
                s[..., m:] += i.mask.double().repeat(heads // kv, 1)
            p = s.softmax(-1)
            if case["kind"] == "score":
                importance[at] += p[..., :m].sum((0, 1))
                continue
            o = torch.bmm((p[..., :m].reshape(-1, m) @ coef["value"][at]).view(kv, -1, case["rank"]),
                          bv.transpose(1, 2).contiguous())
            o = o + p[..., :m].sum(-1, keepdim=True) * mv + torch.bmm(p[..., m:].contiguous(), i.ve[layer, :, ex].double())
            out[b] = o.view(heads, q_len, d).transpose(0, 1)
        outs.append(out)
    if case["kind"] == "score":
        return importance
    return outs if case["via"] == "hook" else torch.stack(outs)


def _projection64(case, i, kind):
    """The middle tokens' coefficients: de-rotated (keys), centred, onto the basis."""
    n, d = case["tokens"], case["head_dim"]
    cos, sin = (t.double() for t in i.rope)
    rows = []
    for t in i.caches[kind]:
        x = t[0].double()
        if kind == "key":
            x = _rotate(x, cos, -sin) / (cos.square() + sin.square())
        rows.append(x.transpose(0, 1).reshape(n, -1))
    x = torch.cat(rows, 1)[SINKS:n - RECENT] - i.mean[kind].double()
    return x @ i.basis[kind].double(), x


def _allocate(errors, sizes, budget):
    """Levels taken per slot: steps in descending worth (made non-increasing) while their bytes fit the budget."""
    step = sizes.double().diff(dim=1)
    worth = ((errors[:, :-1] - errors[:, 1:]).clamp_min(0) / step).cummin(1).values.flatten()
    rank = worth.sort(descending=True, stable=True).indices
    taken = rank[step.flatten()[rank].cumsum(0) <= budget - int(sizes[:, 0].sum())]
    return torch.bincount(taken // step.shape[1], minlength=errors.shape[0])


def _budget_left(case):
    per_token = 4 * _features(case)
    return int(case["budget"] * case["tokens"] * per_token) - (SINKS + RECENT) * per_token


def _exact_encode(case, seed):
    i = _cache_inputs(case, seed)
    out, errors = {}, []
    for k in KINDS:
        c, _ = _projection64(case, i, k)
        x = c.view(c.shape[0], -1, GROUP)
        low = x.amin(2).float().half()
        span = (x.amax(2) - low.double()).float().half()
        code = ((x - low.double()[..., None]) / span.double()[..., None] * 256).floor().clamp(0, 255)
        table = []
        for m in range(1, 9):
            value = low.double()[..., None] + ((code / 2 ** (8 - m)).floor() + 0.5) * span.double()[..., None] / 2 ** m
            table.append((x - value).square().sum((1, 2)))
        errors.append(torch.stack(table, 1) / c.square().sum(1).mean())
        out[k] = {"codes": None, "low": low.double(), "span": span.double(), "pieces": None}
    return {"errors": torch.cat(errors), **out}


def _exact_caches(case, kind, matrix, originals, rope, span):
    start, end = span
    x = matrix.view(matrix.shape[0], case["layers"], case["kv_heads"], case["head_dim"])
    out = []
    for layer, whole in enumerate(originals):
        whole = whole.double().clone()
        t = x[:, layer].transpose(0, 1)
        whole[..., start:end, :] = _rotate(t, rope[0][start:end].double(), rope[1][start:end].double()) if kind == "key" else t
        out.append(whole)
    return out


def _exact_compress(case, seed):
    i = _cache_inputs(case, seed)
    groups, span = case["rank"] // GROUP, (SINKS, case["tokens"] - RECENT)
    rungs = _rungs(groups).to(DEV)
    sizes = torch.tensor(_rung_bytes(rungs.cpu()) + [2 * _features(case)], device=DEV)
    middle, left = span[1] - span[0], _budget_left(case)
    first = max([r for r in range(len(sizes)) if 2 * middle * int(sizes[r]) <= left], default=0)
    importance = i.weights[span[0]:span[1]].double()
    importance = importance / importance.mean()
    errors, coefs = [], {}
    for k in KINDS:
        c, x = _projection64(case, i, k)
        blocks = c.view(middle, groups, GROUP)
        per_width = {0: blocks.square().sum(2)}
        coded = {0: torch.zeros_like(blocks)}
        for w in (2, 4, 8):
            level, low, step = _ladder_quantize(blocks, torch.full((middle, groups), w, device=DEV), torch.float64)
            coded[w] = level * step.double()[..., None] + low.double()[..., None]
            per_width[w] = (blocks - coded[w]).square().sum(2)
        table = [sum(per_width[int(w)][:, g] for g, w in enumerate(row)) for row in rungs.cpu().tolist()]
        e = torch.stack(table + [torch.zeros_like(table[0])], 1) / x.square().sum(1).mean()
        errors.append((e * importance[:, None])[:, first:])
        coefs[k] = (c, coded)
    choice = _allocate(torch.cat(errors), sizes[first:].expand(2 * middle, -1), left) + first
    out = {"choice": [None, None]}
    for j, (k, name) in enumerate((("key", "keys"), ("value", "values"))):
        picked = choice[j * middle:(j + 1) * middle]
        c, coded = coefs[k]
        widths = rungs[picked.clamp_max(len(rungs) - 1)]
        value = sum(coded[w] * (widths == w)[..., None] for w in (0, 2, 4, 8)).flatten(1)
        value = torch.where((picked == len(rungs))[:, None], c, value)
        matrix = value @ i.basis[k].double().T + i.mean[k].double()
        out[name] = _exact_caches(case, k, matrix, i.caches[k], i.rope, span)
    return out


def _exact_restore(case, seed):
    i = _restore_inputs(case, seed)
    n, f, (start, end) = case["tokens"], _features(case), i.span
    rope = _rope(case, n)
    out = {}
    for k, name in (("key", "keys"), ("value", "values")):
        rung, sections, exact = i.kept[k]
        value = torch.zeros(end - start, case["rank"] // GROUP, GROUP, device=DEV, dtype=torch.float64)
        for r, width, cols, part in sections:
            if cols is None:
                continue
            raw, low, step = part
            per = 8 // width  # codes per byte, the first in the low bits
            codes = (raw.long()[..., None] >> (width * torch.arange(per, device=DEV))) & (2 ** width - 1)
            rows = (rung == r).nonzero()
            value[rows, cols] = codes.flatten(2).double() * step.double()[..., None] + low.double()[..., None]
        matrix = value.flatten(1) @ i.basis[k].double().T + i.mean[k].double()
        for r, width, cols, part in sections:
            if cols is None:
                matrix[rung == r] = part.double()
        whole = torch.zeros(n, f, device=DEV, dtype=torch.float64)
        whole[:start], whole[end:] = exact[:start].double(), exact[start:].double()
        whole = whole.view(n, case["layers"], case["kv_heads"], -1).permute(1, 2, 0, 3)
        out[name] = _exact_caches(case, k, matrix, [t[None] for t in whole], rope, i.span)
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind in ("decode", "score"):
        return _exact_attention(case, seed)
    if kind == "project":
        i = _cache_inputs(case, seed)
        return _projection64(case, i, "key")[0]
    return {"encode": _exact_encode, "compress": _exact_compress, "restore": _exact_restore}[kind](case, seed)
