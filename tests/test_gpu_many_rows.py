"""Attention with more query rows per KV head than a decode step has (a question's forward, several new tokens):
every form of K2 (128-row workgroups of a tile quarter, half and whole tile; 256-row workgroups), both heights of
the value product, row counts that fill no block, and ragged batches, against the oracle at the attention bar."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import synth
from helpers import assert_close, assert_sensitive, build_case, gpu_attend, gpu_context, oracle_attend, value_mean_base

pytestmark = pytest.mark.gpu
DEV = "cuda"
SHAPES = {"1b": synth.ModelShape(2, 8, 64, 32, 1024), "3b": synth.ModelShape(2, 8, 128, 24, 2048),
          "small": synth.ModelShape(2, 4, 64, 8, 256)}


@pytest.mark.parametrize("name,tokens,q_len,dtype", [
    ("1b", 290, 2, "float32"),     # one full tile; a quarter tile per workgroup, 64 rows
    ("1b", 1500, 13, "float16"),   # 416 rows: 128-row products, blocks of 52 rows per head
    ("small", 37, 70, "bfloat16"),  # one compressed token, one 256-component column of workgroups
    ("1b", 9000, 3, "bfloat16"),   # half a tile per workgroup
    ("3b", 700, 70, "bfloat16"),   # 210 rows per head
    ("3b", 8400, 2, "float32"),    # a tile per workgroup, 48 rows
    ("3b", 13000, 5, "float16"),   # 256-row workgroups, 120 rows
])
def test_many_rows_match_oracle(name, tokens, q_len, dtype):
    shape = SHAPES[name]
    print(f"[case] many rows {name} T={tokens} q_len={q_len} {dtype}", flush=True)
    case = build_case(shape, tokens, seed=77, query_scale=100.0, q_len=q_len, query_dtype=getattr(torch, dtype))
    ctx, _, _ = gpu_context(case)
    got = gpu_attend(case, ctx, 1)
    ref, base = oracle_attend(case, 1), value_mean_base(case, 1)
    if tokens > 1000:
        queries, case.queries = case.queries, torch.zeros_like(case.queries)
        assert_sensitive(ref, oracle_attend(case, 1), base, what="zero query")
        case.queries = queries
    err, fro = assert_close(got, ref, what=f"{name} {tokens} {q_len}", base=base)
    assert np.array_equal(got, gpu_attend(case, ctx, 1))
    print(f"  max abs err {err:.2e}, rel fro {fro:.2e}", flush=True)


def test_many_rows_ragged_batch_and_negative_scale():
    from compressed_attention import CompressedContext, ModelTables
    from hot_tier import OrderTables, PackedStream

    shape, q_len, lengths = SHAPES["1b"], 7, (900, 36, 290, 2600)
    print(f"[case] many rows, ragged {lengths}", flush=True)
    basis = {k: synth.orthonormal_basis(shape.features, shape.rank, 31 + i) for i, k in enumerate(("key", "value"))}
    mean = {k: torch.randn(shape.features, generator=torch.Generator().manual_seed(33)) * 0.01 for k in ("key", "value")}
    cases = [build_case(shape, t, seed=40 + i, query_scale=100.0, q_len=q_len, basis=basis, mean=mean,
                        rope_rows=max(lengths) + q_len) for i, t in enumerate(lengths)]
    for c in cases:
        c.mask = None  # a batch has no mask
    first = cases[0]
    tables = ModelTables(basis["key"].to(DEV), basis["value"].to(DEV), mean["key"].to(DEV), mean["value"].to(DEV),
                         shape.layers, shape.kv_heads, shape.head_dim, first.cos.to(DEV), first.sin.to(DEV))
    order = OrderTables(first.order.planes, first.order.prefix_bytes, DEV)
    streams = {}
    for kind in ("key", "value"):
        cat = lambda f: torch.from_numpy(np.concatenate([getattr(c, f)[kind] for c in cases])).to(DEV)  # noqa: E731
        streams[kind] = PackedStream.pack(cat("codes"), cat("low"), cat("span"), cat("pieces"), order)
    cu = torch.tensor(np.concatenate([[0], np.cumsum([c.ctx.middle for c in cases])]), dtype=torch.int32)
    ctx = CompressedContext(tables, streams["key"], streams["value"],
                            torch.from_numpy(np.concatenate([c.positions for c in cases])), shape.q_heads, cu_seqlens=cu)
    q = torch.cat([c.queries[0] for c in cases]).to(DEV).contiguous()
    ke, ve = (torch.cat([getattr(c, f)[0] for c in cases], dim=1).to(DEV).contiguous() for f in ("key_exact", "value_exact"))
    lens = tuple(c.key_exact.shape[2] for c in cases)

    def run(query, scaling):
        out = torch.empty(len(cases), q_len, shape.q_heads, shape.head_dim, device=DEV)
        ctx.run_layer(ctx.layer_args(0, query, out, ke, ve, None, lens, scaling))
        torch.cuda.synchronize()
        return out

    out = run(q, shape.head_dim ** -0.5)
    for b, c in enumerate(cases):
        assert_close(out[b:b + 1].cpu().numpy(), oracle_attend(c, 0), what=f"sequence {b}", base=value_mean_base(c, 0))
    # negated twice: the same scores but for the matrix unit's last bit (its sums are not symmetric under negation),
    # which can move a weight by one fp16 rounding, 2^-11 of itself and so at most that of the largest output
    other = run(-q, -shape.head_dim ** -0.5)
    assert float((out - other).abs().max()) <= 2.0 ** -11 * float(out.abs().max())


def test_prepared_codes_serve_few_and_many_rows():
    """One decode of the codes serves layers with one and with several query positions, in either order."""
    case = build_case(SHAPES["1b"], 700, seed=5, query_scale=50.0, q_len=6)
    ctx, _, _ = gpu_context(case)
    want = gpu_attend(case, ctx, 1)
    one = build_case(SHAPES["1b"], 700, seed=5, query_scale=50.0, q_len=1)
    few = gpu_attend(one, ctx, 1)
    ctx._prepared = None
    assert np.array_equal(few, gpu_attend(one, ctx, 1)) and np.array_equal(want, gpu_attend(case, ctx, 1))


def test_value_lines_follow_decodes_and_few_row_layers():
    """The values' operand lines are kept between many-row layers: a few-row layer on the same workspace (whose areas
    overlap them) and a new decode after the codes changed both make the next many-row layer convert again."""
    shape = SHAPES["1b"]
    many = build_case(shape, 1500, seed=9, query_scale=50.0, q_len=9)
    one = build_case(shape, 1500, seed=9, query_scale=50.0, q_len=1)
    ctx, _, streams = gpu_context(many, refine_capacity=200)
    want = [gpu_attend(many, ctx, layer) for layer in (0, 1)]
    few = gpu_attend(one, ctx, 1)  # overwrites part of the workspace, no decode of the codes
    assert np.array_equal(gpu_attend(many, ctx, 1), want[1]) and np.array_equal(gpu_attend(one, ctx, 1), few)
    streams["value"].refine(torch.arange(0, 1400, 7, device=DEV)[:200])
    changed = gpu_attend(many, ctx, 1)
    assert not np.array_equal(changed, want[1])
    case = build_case(shape, 1500, seed=9, query_scale=50.0, q_len=9)
    fresh, _, again = gpu_context(case, refine_capacity=200)
    again["value"].refine(torch.arange(0, 1400, 7, device=DEV)[:200])
    assert np.array_equal(changed, gpu_attend(case, fresh, 1))


@pytest.mark.parametrize("name,tokens", [("1b", 300), ("3b", 13000)])  # 128-row and 256-row workgroups, a ragged last tile
def test_many_rows_with_zero_scale(name, tokens):
    """A scale of 0: every token weighs the same, as zero queries make it (the same kernels, finite scores of 0)."""
    print(f"[case] many rows, scale 0, {name} T={tokens}", flush=True)
    case = build_case(SHAPES[name], tokens, seed=8, query_scale=50.0, q_len=5)
    ctx, _, _ = gpu_context(case)
    case.mask = None
    ke, ve = (getattr(case, f)[0].to(DEV).contiguous() for f in ("key_exact", "value_exact"))

    def run(query, scaling):
        out = torch.empty(1, 5, case.shape.q_heads, case.shape.head_dim, device=DEV)
        ctx.run_layer(ctx.layer_args(0, query, out, ke, ve, None, None, scaling))
        torch.cuda.synchronize()
        return out

    query = case.queries[0].to(DEV).contiguous()
    got, want = run(query, 0.0), run(torch.zeros_like(query), case.shape.head_dim ** -0.5)
    assert torch.isfinite(got).all()
    # the weights are equal in both; their common power of two may differ
    assert torch.allclose(got, want, rtol=1e-5, atol=1e-6 * float(want.abs().max()))


@pytest.mark.parametrize("shape,lengths", [
    (synth.ModelShape(2, 8, 64, 40, 512), (700,)),                       # 5 query heads per KV head, one more than few rows
    (synth.ModelShape(1, 8, 128, 64, 512), (4500,)),                     # 8, half a tile per workgroup
    (synth.ModelShape(1, 4, 64, 32, 256), (500, 36, 37, 1300, 292, 293)),  # 8, sequences of no token, one, a tile and one more
])
def test_one_query_token_of_many_heads(shape, lengths):
    """An ordinary decode step of a model with more than 4 query heads per KV head, single and ragged."""
    from compressed_attention import CompressedContext, ModelTables
    from hot_tier import OrderTables, PackedStream

    print(f"[case] one query token, {shape.q_heads}/{shape.kv_heads} heads, {lengths}", flush=True)
    basis = {k: synth.orthonormal_basis(shape.features, shape.rank, 51 + i) for i, k in enumerate(("key", "value"))}
    mean = {k: torch.randn(shape.features, generator=torch.Generator().manual_seed(53)) * 0.01 for k in ("key", "value")}
    cases = [build_case(shape, t, seed=60 + i, query_scale=100.0, q_len=1, basis=basis, mean=mean,
                        rope_rows=max(lengths) + 1) for i, t in enumerate(lengths)]
    for c in cases:
        c.mask = None
    first = cases[0]
    tables = ModelTables(basis["key"].to(DEV), basis["value"].to(DEV), mean["key"].to(DEV), mean["value"].to(DEV),
                         shape.layers, shape.kv_heads, shape.head_dim, first.cos.to(DEV), first.sin.to(DEV))
    order = OrderTables(first.order.planes, first.order.prefix_bytes, DEV)
    streams = {}
    for kind in ("key", "value"):
        cat = lambda f: torch.from_numpy(np.concatenate([getattr(c, f)[kind] for c in cases])).to(DEV)  # noqa: E731
        streams[kind] = PackedStream.pack(cat("codes"), cat("low"), cat("span"), cat("pieces"), order)
    cu = torch.tensor(np.concatenate([[0], np.cumsum([c.ctx.middle for c in cases])]), dtype=torch.int32)
    ctx = CompressedContext(tables, streams["key"], streams["value"],
                            torch.from_numpy(np.concatenate([c.positions for c in cases])), shape.q_heads, cu_seqlens=cu)
    layer = shape.layers - 1
    q = torch.cat([c.queries[layer] for c in cases]).to(DEV).contiguous()
    ke, ve = (torch.cat([getattr(c, f)[layer] for c in cases], dim=1).to(DEV).contiguous() for f in ("key_exact", "value_exact"))
    out = torch.empty(len(cases), 1, shape.q_heads, shape.head_dim, device=DEV)
    ctx.run_layer(ctx.layer_args(layer, q, out, ke, ve, None, tuple(c.key_exact.shape[2] for c in cases), shape.head_dim ** -0.5))
    torch.cuda.synchronize()
    for b, c in enumerate(cases):
        base = value_mean_base(c, layer) if c.ctx.middle else 0.0
        assert_close(out[b:b + 1].cpu().numpy(), oracle_attend(c, layer), what=f"sequence {b}", base=base)
