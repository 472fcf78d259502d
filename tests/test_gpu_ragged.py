"""Ragged batches past one wave's worth of sequences (the tile lookup takes 64 at a time): every sequence of the batch
against the oracle, with sequences of no compressed token, of one, of a whole tile and of one more."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import synth
from helpers import assert_close, build_case, oracle_attend, value_mean_base

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("batch,q_len", [(63, 1), (64, 1), (65, 1), (130, 3)])
def test_ragged_batch_matches_oracle(batch, q_len):
    from compressed_attention import CompressedContext, ModelTables
    from hot_tier import OrderTables, PackedStream

    shape = synth.ModelShape(1, 4, 64, 8, 256)
    print(f"[case] ragged batch of {batch}, q_len {q_len}", flush=True)
    lengths = [36 + (0, 1, 256, 257, 40, 511)[i % 6] for i in range(batch)]
    basis = {k: synth.orthonormal_basis(shape.features, shape.rank, 31 + i) for i, k in enumerate(("key", "value"))}
    mean = {k: torch.randn(shape.features, generator=torch.Generator().manual_seed(33)) * 0.01 for k in ("key", "value")}
    kinds = {t: build_case(shape, t, seed=40 + t, query_scale=100.0, q_len=q_len, basis=basis, mean=mean, rope_rows=600)
             for t in set(lengths)}
    cases = [kinds[t] for t in lengths]
    for c in kinds.values():
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
    out = torch.empty(batch, q_len, shape.q_heads, shape.head_dim, device=DEV)
    ctx.run_layer(ctx.layer_args(0, q, out, ke, ve, None, tuple(c.key_exact.shape[2] for c in cases), shape.head_dim ** -0.5))
    torch.cuda.synchronize()
    want = {t: oracle_attend(c, 0) for t, c in kinds.items()}
    for b, (t, c) in enumerate(zip(lengths, cases)):
        base = value_mean_base(c, 0) if c.ctx.middle else 0.0
        assert_close(out[b:b + 1].cpu().numpy(), want[t], what=f"sequence {b} of {t}", base=base)
