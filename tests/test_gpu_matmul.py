"""The float32 product on the fp16 matrix cores (dkv_matmul_f32) against float64.

Bound: hi + lo holds an element to 2^-22 of itself and the dropped lo lo is below 2^-22 of a product, so the
split costs at most 3 * 2^-22 of sum |a b|; each of the 3 K / 16 fp32 accumulations rounds by at most 2^-24 of
sum |a b|, and the scaling, the sum over k ranges and the bias by a few more."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _pair(m, n, k, kn, seed):
    g = torch.Generator(DEV).manual_seed(seed)
    a = torch.randn(m, k, generator=g, device=DEV)
    b = torch.randn(k, n, generator=g, device=DEV) if kn else torch.randn(n, k, generator=g, device=DEV).t()
    return a, b, torch.randn(n, generator=g, device=DEV)


def _check(got, a, b, bias=None):
    ref = a.double() @ b.double()
    size = a.double().abs() @ b.double().abs()
    if bias is not None:
        ref, size = ref + bias.double(), size + bias.double().abs()
    bound = (3 * 2.0 ** -22 + (3 * a.shape[1] / 16 + 24) * 2.0 ** -24) * size
    worst = float(((got.double() - ref).abs() / bound.clamp_min(1e-300)).max())
    assert got.shape == ref.shape and worst <= 1.0, worst
    return float((got.double() - ref).norm() / ref.norm()), float((torch.matmul(a, b).double() - a.double() @ b.double()).norm()
                                                                  / (a.double() @ b.double()).norm())


@pytest.mark.parametrize("kn", [True, False])
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (37, 65, 63), (256, 256, 64), (257, 255, 65), (300, 513, 130),
                                   (511, 512, 4099), (64, 100, 40000)])
def test_matmul_against_float64(m, n, k, kn):
    import dkv_hip

    a, b, bias = _pair(m, n, k, kn, m + n + k)
    print(f"[case] matmul {m} x {n} x {k} kn={kn}", flush=True)
    _check(dkv_hip.matmul_f32(a, b), a, b)
    mine, lib = _check(dkv_hip.matmul_f32(a, b, bias), a, b, bias)
    if k >= 1000:  # long sums: closer to float64 than the library's float32 product
        assert mine <= lib


def test_matmul_rows_of_any_scale_strides_and_specials():
    """Rows over the whole float32 range keep float32's relative accuracy; unaligned and strided operands are
    read as they lie; infinities and NaN come out where torch puts them."""
    import dkv_hip

    a, b, _ = _pair(300, 200, 256, True, 5)
    wide = a * torch.logspace(-37, 30, 300, device=DEV)[:, None]
    _check(dkv_hip.matmul_f32(wide, b), wide, b)
    big = torch.randn(300, 261, device=DEV)
    part = big[:, 3:259]  # rows 1,044 bytes apart, from an address that is no multiple of 16
    _check(dkv_hip.matmul_f32(part, b[:, 7:150]), part, b[:, 7:150])
    assert (dkv_hip.matmul_f32(torch.zeros_like(a), b) == 0).all()
    a[5, 3], a[7, 9], b[4, 11] = float("inf"), float("nan"), float("-inf")
    got, want = dkv_hip.matmul_f32(a, b), a @ b
    for same in (torch.isnan, torch.isposinf, torch.isneginf):
        assert torch.equal(same(got), same(want))
    fine = torch.isfinite(want)
    assert torch.allclose(got[fine], want[fine], rtol=1e-4, atol=1e-4)


def test_float_product_route():
    """Small products, watched ones and other types stay with torch, bit for bit."""
    import kvtc

    a, b, bias = _pair(128, 64, 512, True, 6)
    assert torch.equal(kvtc.float_product(a, b, bias), a @ b + bias)
    a, b, bias = _pair(3000, 2048, 1024, True, 7)
    assert a.shape[0] * a.shape[1] * b.shape[1] >= kvtc.SPLIT_PRODUCT_MIN
    got = kvtc.float_product(a, b, bias)
    assert not torch.equal(got, a @ b + bias)
    _check(got, a, b, bias)
    weight = b.clone().requires_grad_(True)
    assert torch.equal(kvtc.float_product(a, weight), a @ weight) and kvtc.float_product(a, weight).requires_grad
    with torch.autocast("cuda", dtype=torch.float16):
        assert kvtc.float_product(a, b).dtype == torch.float16
    assert kvtc.float_product(a.half(), b.half()).dtype == torch.float16
    out, tangent = torch.func.jvp(lambda x: kvtc.float_product(x, b), (a,), (a,))
    assert torch.equal(out, a @ b) and torch.equal(tangent, a @ b)


@pytest.mark.parametrize("layers,heads,dim,rank,dtype,start,end,kind", [
    (2, 8, 64, 256, torch.float16, 4, 269, "key"),       # 1,024 columns: idle threads, a row tile and a remainder
    (28, 8, 128, 192, torch.bfloat16, 0, 33, "key"),     # 28,672 columns, no sinks, 192 of 256 basis columns
    (16, 8, 64, 1024, torch.float32, 4, 260, "value"),   # 8,192 columns: every thread of the small workgroup
    (3, 5, 48, 130, torch.float16, 2, 300, "value"),     # 720 columns: no whole block of 64
])
def test_projection_from_caches_matches_rows(layers, heads, dim, rank, dtype, start, end, kind):
    """dkv_project_caches equals dkv_matmul_f32 of dkv_centered_rows' rows bit for bit (same pieces, same sums), also
    in a row with an infinity, and its energies are the rows' (at most `columns` roundings of a positive sum)."""
    import dkv_hip

    tokens, width = end + 7, layers * heads * dim
    print(f"[case] projection from caches {layers}x{heads}x{dim} rank {rank} {dtype} {start}..{end} {kind}", flush=True)
    g = torch.Generator(DEV).manual_seed(rank)
    caches = [torch.randn(1, heads, tokens, dim, generator=g, device=DEV).to(dtype) for _ in range(layers)]
    caches[1][0, 1, start + 5, 3] = float("inf")
    mean = torch.randn(width, generator=g, device=DEV)
    cos, sin = (torch.randn(tokens, dim, generator=g, device=DEV) for _ in range(2)) if kind == "key" else (None, None)
    basis = torch.randn(width, rank, generator=g, device=DEV) / width ** 0.5
    rows = torch.empty(end - start, width, device=DEV)
    dkv_hip.centered_rows(caches, cos, sin, mean, start, end, rows)
    for b in (basis, basis.T.contiguous().T):
        got, energy = dkv_hip.project_caches(caches, cos, sin, mean, start, end, b, True)
        assert torch.equal(torch.nan_to_num(got), torch.nan_to_num(dkv_hip.matmul_f32(rows, b)))
    assert torch.allclose(energy.double(), rows.double().square().sum(1), rtol=width * 2.0 ** -24, atol=0.0)


def _same_specials(got, want):
    for same in (torch.isnan, torch.isposinf, torch.isneginf):
        assert torch.equal(same(got), same(want))
    fine = torch.isfinite(want)
    assert torch.allclose(got[fine], want[fine], rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("kn", [True, False])
@pytest.mark.parametrize("rows,columns", [("all", 0), (0, "all"), (65, 129), (1, 0), (0, 1)])
def test_matmul_flagged_rows_and_columns(rows, columns, kn):
    """Rows of A and columns of B with infinities or NaN, from one (a tile of one row) to all of them, with a bias:
    where torch puts them, the other outputs untouched."""
    import dkv_hip

    m, n, k = 200, 300, 1100
    print(f"[case] matmul flagged rows {rows}, columns {columns} kn={kn}", flush=True)
    a, b, bias = _pair(m, n, k, kn, 11)
    specials = torch.tensor([float("inf"), float("-inf"), float("nan")], device=DEV)
    for i in range(m if rows == "all" else rows):
        a[i if rows == "all" else 3 * i, (7 * i) % k] = specials[i % 3]
    for i in range(n if columns == "all" else columns):
        b[(5 * i) % k, i if columns == "all" else 2 * i] = specials[(i + 1) % 3]
    _same_specials(dkv_hip.matmul_f32(a, b, bias), torch.matmul(a, b) + bias)


def test_projection_from_caches_with_every_row_flagged():
    """A NaN in the mean reaches every row: all outputs NaN, and no slower than a few of the product (by one workgroup per 64
    rows, a thread per output and all of K in turn, it was hundreds of them)."""
    import dkv_hip

    layers, heads, dim, rank, end = 16, 8, 64, 1024, 2052
    print("[case] projection from caches, every row flagged", flush=True)
    g = torch.Generator(DEV).manual_seed(3)
    caches = [torch.randn(1, heads, end + 3, dim, generator=g, device=DEV).half() for _ in range(layers)]
    mean = torch.zeros(layers * heads * dim, device=DEV)
    cos, sin = (torch.randn(end + 3, dim, generator=g, device=DEV) for _ in range(2))
    basis = torch.randn(layers * heads * dim, rank, generator=g, device=DEV)

    def timed():
        best = 1e9
        for _ in range(3):
            t0, t1 = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            t0.record()
            out, _ = dkv_hip.project_caches(caches, cos, sin, mean, 4, end, basis, False)
            t1.record()
            t1.synchronize()
            best = min(best, t0.elapsed_time(t1))
        return out, best

    out, plain = timed()
    assert torch.isfinite(out).all()
    mean[77] = float("nan")
    out, flagged = timed()
    print(f"  {1e3 * plain:.0f} us, every row flagged {1e3 * flagged:.0f} us", flush=True)
    assert torch.isnan(out).all() and flagged < 4 * plain


@pytest.mark.parametrize("above", [2.0 ** 12, 2.0 ** 18, 2.0 ** 26])
def test_matmul_outliers_inside_rows_and_columns(above):
    """One element of every row of A and of every column of B far above the rest, each against a zero: an element is
    held to 2^-39 of its row's largest where 2^-22 of itself is less, so each side adds 2^-39 max |a| sum |b| at most."""
    import dkv_hip

    m, n, k = 200, 260, 1024
    print(f"[case] matmul outliers of {above:.0f}", flush=True)
    a, b, _ = _pair(m, n, k, True, 21)
    a[:, 5] *= above
    b[5] = 0.0
    b[9] *= above
    a[:, 9] = 0.0
    got, ref = dkv_hip.matmul_f32(a, b).double(), a.double() @ b.double()
    aa, bb = a.double().abs(), b.double().abs()
    bound = (3 * 2.0 ** -22 + (3 * k / 16 + 24) * 2.0 ** -24) * (aa @ bb)
    bound += 2.0 ** -39 * (aa.amax(1, keepdim=True) * bb.sum(0) + aa.sum(1, keepdim=True) * bb.amax(0))
    assert ((got - ref).abs() <= bound).all()
    if above <= 2.0 ** 12:  # within the range where the pieces hold every element
        assert float((got - ref).norm()) <= float((torch.matmul(a, b).double() - ref).norm())


@pytest.mark.parametrize("m,n,k", [(1, 70, 300), (70, 90, 1), (70, 1, 300), (1, 1, 300)])
def test_matmul_strides_of_single_rows_and_columns(m, n, k):
    """A dimension of one element has any stride, and contiguous() leaves it."""
    import dkv_hip

    print(f"[case] matmul single {m} x {n} x {k}", flush=True)
    a, b, _ = _pair(m, n, k, True, 31)
    wide = torch.randn(m + k, 2 * (n + k), device=DEV)
    views_a = [a, a.t().contiguous().t(), torch.as_strided(wide, (m, k), (1, 1)) if m == 1 else a]
    views_b = [b, b.t().contiguous().t(), torch.as_strided(wide, (k, n), (3, 1)) if k == 1 else b]
    for x in views_a:
        for y in views_b:
            _check(dkv_hip.matmul_f32(x, y), x, y)
