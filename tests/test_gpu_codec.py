"""The kvtc codec's HIP passes (dkv_ladder_errors, dkv_ladder_code, dkv_rows_to_caches, dkv_copy_tokens) against the
torch arithmetic they replace, which stays as the path of every other device and layout."""

from __future__ import annotations

import pytest
import torch

import synth

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _codec(shape, seed=3):
    import kvtc

    ctx = synth.make_context(shape, 300, seed=seed)
    return kvtc.KVTCCodec(synth.kvtc_checkpoint(ctx), DEV, synth.RopeModel(shape, DEV))


@pytest.mark.parametrize("groups,tokens,rungs", [(4, 1, 8), (16, 257, 8), (7, 130, 3), (32, 70, 40)])
def test_ladder_passes_match_torch(groups, tokens, rungs, monkeypatch):
    """Groups that fill no quad, one token, more than 16 rungs; a group of equal values and one of huge range."""
    import kvtc

    print(f"[case] ladder passes G={groups} n={tokens} R={rungs}", flush=True)
    codec = _codec(synth.ModelShape(2, 8, 64, 32, 1024))
    g = torch.Generator(DEV).manual_seed(groups)
    stream = codec.streams["key"]
    stream.rungs = torch.tensor([0, 2, 4, 8], device=DEV)[torch.randint(0, 4, (rungs, groups), generator=g, device=DEV)]
    stream.rung_bytes = [1] * rungs
    coef = torch.randn(tokens, 64 * groups, generator=g, device=DEV) * torch.logspace(1, -3, 64 * groups, device=DEV)
    coef[0, :64] *= 300  # up to about 13,000 (an fp16 shift holds 65,504; past it both give NaN)
    picked = torch.randint(-1, rungs + 1, (tokens,), generator=g, device=DEV)
    errors = codec.rung_errors(coef, "key")
    counts = torch.bincount(picked + 1, minlength=rungs + 2).tolist()
    decoded, (codes, low, scale) = codec._code_stream("key", coef, picked, counts)
    monkeypatch.setattr(kvtc, "_plain_gpu", lambda *t: False)
    want = codec.rung_errors(coef, "key")
    # sums of 64 G squares, each computed alike: at most 64 G roundings of 2^-24 of the (positive) sum
    assert torch.allclose(errors, want, rtol=64 * groups * 2.0 ** -24, atol=0.0)
    decoded_t, (codes_t, low_t, scale_t) = codec._code_stream("key", coef, picked, counts)
    assert torch.equal(decoded, decoded_t) and torch.equal(codes, codes_t)
    assert torch.equal(low.view(torch.int16), low_t.view(torch.int16))
    assert torch.equal(scale.view(torch.int16), scale_t.view(torch.int16))


def test_ladder_errors_of_degenerate_groups():
    """A constant group's step rounds to 0 in fp16 (levels 0/0): NaN errors, as the torch arithmetic gives; a NaN or
    an infinity makes its token's errors non-finite and no other's."""
    codec = _codec(synth.ModelShape(2, 8, 64, 32, 1024))
    coef = torch.randn(6, 1024, generator=torch.Generator(DEV).manual_seed(1), device=DEV)
    coef[1, :64] = 0.25
    coef[3, 70], coef[4, 80] = float("nan"), float("inf")
    errors = codec.rung_errors(coef, "key")
    assert torch.isfinite(errors[[0, 2, 5]]).all()
    used = codec.streams["key"].rungs[:, :2] > 0
    assert torch.isnan(errors[1][used[:, 0]]).all() and torch.isnan(errors[3]).all()
    assert not torch.isfinite(errors[4]).any()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shape,tokens,span", [(synth.ModelShape(2, 8, 64, 32, 1024), 41, (4, 9)),
                                               (synth.ModelShape(3, 2, 128, 24, 2048), 33, (0, 33)),
                                               (synth.ModelShape(1, 3, 8, 3, 64), 5, (2, 4))])
def test_rebuilt_caches_match_from_matrix(shape, tokens, span, dtype, monkeypatch):
    """Rows back into caches, keys rotated, the tokens outside the span bit for bit the originals'."""
    import kvtc

    codec = _codec(synth.ModelShape(2, 8, 64, 32, 1024))
    codec.layers, codec.heads, codec.head_dim = shape.layers, shape.kv_heads, shape.head_dim
    g = torch.Generator(DEV).manual_seed(tokens)
    rows = torch.randn(span[1] - span[0], shape.features, generator=g, device=DEV)
    originals = [torch.randn(1, shape.kv_heads, tokens, shape.head_dim, generator=g, device=DEV).to(dtype)
                 for _ in range(shape.layers)]
    originals[0] = originals[0].transpose(1, 2).contiguous().transpose(1, 2)  # one in another memory order
    cos, sin = (torch.randn(tokens, shape.head_dim, generator=g, device=DEV) for _ in range(2))
    monkeypatch.setattr(kvtc, "inverse_transform", lambda *a: rows.clone())
    for kind in ("key", "value"):
        got = codec._rebuilt_caches(kind, None, originals, span, cos, sin)
        with monkeypatch.context() as m:
            m.setattr(kvtc, "_plain_caches", lambda t: False)
            want = codec._rebuilt_caches(kind, None, originals, span, cos, sin)
        for a, b in zip(got, want):
            assert a.dtype == b.dtype == dtype and torch.equal(a, b)


@pytest.mark.parametrize("groups,tokens", [(1, 1), (7, 33), (32, 130)])
def test_live_groups_match_torch(groups, tokens):
    """Unused groups, one whose only entry is the last row's last, one of negative zeros, a NaN; and the coefficients of
    ladder codes bit for bit."""
    import dkv_hip

    print(f"[case] live groups G={groups} n={tokens}", flush=True)
    g = torch.Generator(DEV).manual_seed(groups)
    coef = torch.randn(tokens, groups * 64, generator=g, device=DEV)
    for k in range(groups):
        if k % 3 != 1:
            coef[:, k * 64:(k + 1) * 64] = -0.0 if k % 2 else 0.0
    coef[-1, -1] = float("nan") if groups == 7 else 2.0
    want = coef.reshape(tokens, -1, 64).ne(0).any(dim=2).any(dim=0)
    assert torch.equal(dkv_hip.live_groups(coef), want)
    codes = torch.randint(0, 256, (tokens, groups, 64), generator=g, device=DEV, dtype=torch.uint8)
    low, scale = (torch.randn(tokens, groups, generator=g, device=DEV).half() for _ in range(2))
    codes[:, 0], low[:, 0] = 0, 0.0
    values = codes.float() * scale.float().unsqueeze(2) + low.float().unsqueeze(2)
    got = torch.empty(tokens, groups * 64, device=DEV)
    live = dkv_hip.live_groups(got, codes, low, scale)
    assert torch.equal(got.view(torch.int32), values.reshape(tokens, -1).view(torch.int32))
    assert torch.equal(live, values.ne(0).any(dim=2).any(dim=0))
