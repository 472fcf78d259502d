"""The progressive encoder's HIP passes (dkv_quantize8_rungs, the bit-plane pack) against the table they replace and
the oracle's planes, at group counts that fill no quad of groups and buffers that start at any element."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import synth

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("groups,tokens,rungs", [(1, 1, 1), (4, 257, 7), (7, 130, 16), (16, 33, 17), (32, 66, 128)])
def test_rung_errors_match_table(groups, tokens, rungs):
    import progressive

    print(f"[case] rung errors G={groups} n={tokens} R={rungs}", flush=True)
    g = torch.Generator(DEV).manual_seed(groups)
    flat = torch.randn(tokens * 64 * groups + 1, generator=g, device=DEV)
    for coef in (flat[:-1].view(tokens, -1), flat[1:].view(tokens, -1)):  # the second 4 bytes off
        coef = coef * torch.logspace(1, -3, 64 * groups, device=DEV) if coef.data_ptr() % 16 == 0 else coef
        if coef.data_ptr() % 16 == 0:
            coef[0, :64] = 0.25  # a group of equal values
            coef[-1, -1] = float("nan")
        planes = torch.randint(0, 9, (rungs, groups), generator=g, device=DEV, dtype=torch.uint8)
        codes, low, span, errors, energy = progressive._quantize8_rungs(coef, planes)
        codes_t, low_t, span_t, table = progressive._quantize8_hip(coef, 64, True)
        assert torch.equal(codes, codes_t)
        assert torch.equal(low.view(torch.int16), low_t.view(torch.int16))
        assert torch.equal(span.view(torch.int16), span_t.view(torch.int16))
        want = torch.gather(table.double(), 2, planes.long().T.expand(tokens, -1, -1)).sum(1)
        # at most `groups` roundings of 2^-24 of a positive sum
        assert torch.allclose(errors.double(), want, rtol=groups * 2.0 ** -24, atol=0.0, equal_nan=True)
        # 64 groups squares, each rounded, and their sum
        assert torch.allclose(energy.double(), coef.double().square().sum(1), rtol=65 * groups * 2.0 ** -24, atol=0.0,
                              equal_nan=True)


@pytest.mark.parametrize("groups,tokens,shift", [(4, 1, 0), (7, 65, 3), (16, 300, 1)])
def test_pack_any_alignment(groups, tokens, shift):
    """Hot and cold tiers of random piece counts, read back bit for bit: the hot planes dequantize to the codes'
    top planes, and after a refine of every token to all of them."""
    import progressive
    from hot_tier import OrderTables, PackedStream

    print(f"[case] pack G={groups} n={tokens} at byte {shift}", flush=True)
    g = torch.Generator(DEV).manual_seed(tokens)
    sequence = [x for m in range(8) for x in np.random.default_rng(m).permutation(groups).tolist()]
    order = progressive.order_from_sequence(sequence, groups)
    flat = torch.randint(0, 256, (tokens * groups * 64 + 4,), generator=g, device=DEV, dtype=torch.uint8)
    codes = flat[shift:shift + tokens * groups * 64].view(tokens, groups, 64)
    low = torch.randn(tokens, groups, generator=g, device=DEV).half()
    span = torch.rand(tokens, groups, generator=g, device=DEV).half() + 0.5
    pieces = torch.randint(0, 8 * groups + 1, (tokens,), generator=g, device=DEV, dtype=torch.int16)
    packed = PackedStream.pack(codes, low, span, pieces, OrderTables(order.planes, order.prefix_bytes, DEV),
                               refine_capacity=tokens)
    planes = order.planes.to(DEV)[pieces.long()]
    assert torch.equal(packed.dequantize(), progressive.dequantize(codes, low, span, planes))
    packed.refine(torch.arange(tokens, device=DEV))
    assert torch.equal(packed.dequantize(), progressive.dequantize(codes, low, span, torch.full((1, groups), 8, device=DEV)))


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("layers,heads,tokens,dim,start,end", [(2, 3, 50, 64, 4, 18), (130, 1, 9, 8, 0, 8), (1, 8, 40, 128, 5, 40)])
def test_outside_tokens_match_cat(layers, heads, tokens, dim, start, end, dtype):
    """More layers than one launch takes, no sinks, no recent window."""
    import dkv_hip

    print(f"[case] outside tokens L={layers} H={heads} T={tokens} D={dim} {start}..{end} {dtype}", flush=True)
    g = torch.Generator(DEV).manual_seed(layers)
    caches = [torch.randn(1, heads, tokens, dim, generator=g, device=DEV).to(dtype) for _ in range(layers)]
    got = dkv_hip.outside_tokens(caches, start, end - start)
    assert torch.equal(got, torch.stack([torch.cat([t[..., :start, :], t[..., end:, :]], dim=2) for t in caches]))
