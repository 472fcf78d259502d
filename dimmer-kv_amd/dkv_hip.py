"""ctypes binding of libdimmerkv_hip.so (the C ABI declared in include/dimmerkv.h).

The library is loaded from this directory.  There is no fallback: if the
library is missing, or a tensor is not on a GPU, the call raises.  Return
codes map to the reference's exception types (scripts/kvtc.py:226-227,
289-290 ValueError; scripts/progressive.py:189-190 AssertionError;
scripts/methods.py:136-137 RuntimeError).
"""

from __future__ import annotations

import contextlib
import ctypes
from pathlib import Path

import torch

HERE = Path(__file__).resolve().parent
LIB_PATH = HERE / "libdimmerkv_hip.so"
ABI_VERSION = 3

DKV_F32, DKV_F16, DKV_BF16 = 0, 1, 2
DKV_FMT_PLANES, DKV_FMT_LADDER = 0, 1
_DTYPE = {torch.float32: DKV_F32, torch.float16: DKV_F16, torch.bfloat16: DKV_BF16}

EXPORTS = [
    "dkv_abi_version", "dkv_last_error", "dkv_pack_planes", "dkv_pack_ladder", "dkv_unpack_dequant", "dkv_dequantize_codes",
    "dkv_prepare_key_basis", "dkv_prepare_value_basis", "dkv_attend_workspace_bytes", "dkv_attend_prepare",
    "dkv_attend_layer",
    "dkv_attend_scores", "dkv_attend_values",
    "dkv_score_workspace_bytes", "dkv_score_begin", "dkv_score_layer", "dkv_topk_workspace_bytes", "dkv_topk",
    "dkv_gather_cold", "dkv_refine_rows", "dkv_wire_pack", "dkv_wire_unpack", "dkv_attend_layer_noalloc",
    "dkv_quantize8", "dkv_quantize8_rungs", "dkv_centered_rows", "dkv_matmul_f32_workspace_bytes", "dkv_matmul_f32",
    "dkv_ladder_errors", "dkv_ladder_code", "dkv_rows_to_caches", "dkv_copy_tokens", "dkv_outside_tokens", "dkv_project_caches", "dkv_live_groups",
]
NOALLOC_MAX_BYTES = 64 << 20  # DKV_NOALLOC_MAX_BYTES: the static workspace of dkv_attend_layer_noalloc

c_i32, c_i64, c_f32, c_vp, c_sz = ctypes.c_int32, ctypes.c_int64, ctypes.c_float, ctypes.c_void_p, ctypes.c_size_t


class Order(ctypes.Structure):
    _fields_ = [("groups", c_i32), ("pieces", c_i32), ("planes", c_vp), ("seg_off", c_vp), ("cold_off", c_vp),
                ("prefix_bytes", c_vp)]


class Ladder(ctypes.Structure):
    _fields_ = [("groups", c_i32), ("rungs", c_i32), ("bits", c_vp), ("seg_off", c_vp), ("rung_bytes", c_vp)]


class Stream(ctypes.Structure):
    _fields_ = [("blob", c_vp), ("tok_off", c_vp), ("pieces", c_vp), ("order", Order), ("format", c_i32),
                ("ladder", Ladder)]


class Wire(ctypes.Structure):
    """Where each (rung, width) section of the byte-storage layout lies (dkv_wire_t)."""
    _fields_ = [("section", c_vp), ("count", c_vp), ("rank", c_vp), ("slot", c_vp), ("nwidth", c_vp),
                ("bytes", c_i64)]


class AttendArgs(ctypes.Structure):
    _fields_ = [
        ("batch", c_i32), ("q_len", c_i32),
        ("layers", c_i32), ("layer", c_i32), ("kv_heads", c_i32), ("head_dim", c_i32), ("q_heads", c_i32),
        ("rank", c_i32),
        ("scaling", c_f32),
        ("key", Stream), ("value", Stream),
        ("cu_seqlens", c_vp), ("cu_seqlens_host", c_vp), ("positions", c_vp),
        ("key_basis", c_vp), ("value_basis", c_vp), ("mean_k", c_vp), ("mean_v", c_vp),
        ("rope_cos", c_vp), ("rope_sin", c_vp), ("rope_rows", c_i32),
        ("query", c_vp), ("query_dtype", c_i32),
        ("cu_exact", c_vp), ("cu_exact_host", c_vp), ("key_exact", c_vp), ("value_exact", c_vp), ("mask", c_vp),
        ("out", c_vp), ("out_dtype", c_i32), ("exact_dtype", c_i32),
    ]


class DkvError(RuntimeError):
    pass


_lib = None


def lib() -> ctypes.CDLL:
    """Load the HIP library once; raise loudly if it has not been built."""
    global _lib
    if _lib is None:
        if not LIB_PATH.exists():
            raise RuntimeError(f"{LIB_PATH} is missing: build it with __graft_entry__.build() "
                               "(python dimmer-kv_amd/build_lib.py); there is no CPU fallback")
        handle = ctypes.CDLL(str(LIB_PATH))
        handle.dkv_abi_version.restype = c_i32
        handle.dkv_last_error.restype = ctypes.c_char_p
        for name in ("dkv_attend_workspace_bytes", "dkv_score_workspace_bytes", "dkv_topk_workspace_bytes",
                     "dkv_matmul_f32_workspace_bytes"):
            getattr(handle, name).restype = c_sz
        handle.dkv_topk_workspace_bytes.argtypes = [c_i32]
        if handle.dkv_abi_version() != ABI_VERSION:
            raise RuntimeError(f"{LIB_PATH} has ABI {handle.dkv_abi_version()}, expected {ABI_VERSION}")
        _lib = handle
    return _lib


def _check(rc: int, what: str) -> None:
    if rc == 0:
        return
    msg = f"{what}: {lib().dkv_last_error().decode()} (code {rc})"
    if rc in (-1, -2):
        raise ValueError(msg)
    if rc == -5:
        raise AssertionError(msg)
    raise DkvError(msg)


def addr(t: torch.Tensor) -> int:
    """Address of ``t``'s first element.  torch reports 0 for every empty tensor; an empty view of an
    allocation gets the address its storage gives it, so arrays of zero tokens still pass the C ABI's
    non-null checks (nothing is read through them)."""
    if t.numel():
        return t.data_ptr()
    return t.untyped_storage().data_ptr() + t.storage_offset() * t.element_size()


def ptr(t: torch.Tensor | None) -> int | None:
    if t is None:
        return None
    if not t.is_cuda:
        raise ValueError("dimmer-kv HIP kernels need GPU tensors (no CPU path)")
    if not t.is_contiguous():
        raise ValueError("dimmer-kv HIP kernels need contiguous tensors")
    return addr(t)


try:  # the raw handle of the current stream, without a Python stream object per call
    from torch._C import _cuda_getCurrentRawStream as _raw_stream, _cuda_getDevice as _current_device
except ImportError:  # pragma: no cover - older torch
    _raw_stream = _current_device = None


def stream_handle() -> int:
    """The current HIP stream of the current device (what torch.cuda.current_stream().cuda_stream gives)."""
    if _raw_stream is not None:
        return _raw_stream(_current_device())
    return torch.cuda.current_stream().cuda_stream


_HERE = contextlib.nullcontext()


def _on_device_of(t: torch.Tensor):
    """``t``'s GPU as the current device: ``stream_handle`` is then the stream that orders the work on its memory."""
    return _HERE if _current_device is not None and t.get_device() == _current_device() else torch.cuda.device(t.device)


def dtype_code(dtype: torch.dtype) -> int:
    if dtype not in _DTYPE:
        raise ValueError(f"unsupported dtype {dtype}")
    return _DTYPE[dtype]


def _expect(what: str, device, *expected) -> None:
    """Refuse tensors that a kernel would read or write past: each (tensor, name, dtype, shape), a first length of None
    for any.  Lists of caches are their callers' to compare (kvtc._plain_caches, or made alike)."""
    for t, name, dtype, shape in expected:
        have, want = t.shape, shape
        if want[0] is None and len(have) == len(want):
            have, want = have[1:], want[1:]
        if have != want or t.dtype != dtype or t.device != device:
            raise ValueError(f"{what}: {name} must be {dtype} {list(shape)} on {device} "
                             f"(got {t.dtype} {list(t.shape)} on {t.device})")


# ----------------------------------------------------------------- wrappers

def pack_planes(codes, low, span, pieces, order: Order, hot, hot_off, cold=None, cold_off=None) -> None:
    n = codes.shape[0]
    _check(lib().dkv_pack_planes(c_vp(ptr(codes)), c_vp(ptr(low)), c_vp(ptr(span)), c_vp(ptr(pieces)), c_i32(n),
                                 order, c_vp(ptr(hot)), c_vp(ptr(hot_off)), c_vp(ptr(cold)), c_vp(ptr(cold_off)),
                                 c_vp(stream_handle())), "dkv_pack_planes")


def pack_ladder(codes, low, scale, rung, ladder: Ladder, blob, tok_off) -> None:
    n = codes.shape[0]
    _check(lib().dkv_pack_ladder(c_vp(ptr(codes)), c_vp(ptr(low)), c_vp(ptr(scale)), c_vp(ptr(rung)), c_i32(n),
                                 ladder, c_vp(ptr(blob)), c_vp(ptr(tok_off)), c_vp(stream_handle())),
           "dkv_pack_ladder")


def wire_pack(codes, low, scale, rung, ladder: Ladder, wire: Wire, out) -> None:
    """codes u8 [n, G, 64], shifts/scales (int16 views of fp16) [n, G], rung int16 [n] -> storage sections."""
    _check(lib().dkv_wire_pack(c_vp(ptr(codes)), c_vp(ptr(low)), c_vp(ptr(scale)), c_vp(ptr(rung)),
                               c_i32(rung.numel()), ladder, wire, c_vp(ptr(out)), c_vp(stream_handle())),
           "dkv_wire_pack")


def wire_unpack(data, rung, ladder: Ladder, wire: Wire, codes, low, scale) -> None:
    """Storage sections -> codes u8 [n, G, 64], shifts/scales (int16 views of fp16) [n, G]."""
    _check(lib().dkv_wire_unpack(c_vp(ptr(data)), c_vp(ptr(rung)), c_i32(rung.numel()), ladder, wire,
                                 c_vp(ptr(codes)), c_vp(ptr(low)), c_vp(ptr(scale)), c_vp(stream_handle())),
           "dkv_wire_unpack")


def unpack_dequant(stream: Stream, t0: int, nt: int, out: torch.Tensor) -> None:
    _check(lib().dkv_unpack_dequant(ctypes.byref(stream), c_i32(t0), c_i32(nt), c_vp(ptr(out)),
                                    c_i32(dtype_code(out.dtype)), c_vp(stream_handle())), "dkv_unpack_dequant")


def centered_rows(tensors, cos, sin, mean, start: int, end: int, out) -> None:
    """Per-layer caches [1, H, T, D] (fp16/bf16/fp32, one device) -> out f32 [end - start, L*H*D]:
    the token-matrix rows start..end - 1 minus ``mean``, keys de-rotated when cos/sin are given."""
    first = tensors[0]
    if first.dtype not in _DTYPE:
        raise ValueError(f"centered_rows: cache dtype {first.dtype} not supported")
    if first.dim() != 4 or first.shape[0] != 1:
        raise ValueError(f"centered_rows: caches must be [1, heads, tokens, head_dim] (got {tuple(first.shape)})")
    if any(t.shape != first.shape or t.dtype != first.dtype or t.device != first.device or not t.is_contiguous()
           for t in tensors):
        raise ValueError("centered_rows: the layers' caches must be contiguous and share shape, dtype and device")
    _, heads, tokens, head_dim = first.shape
    width = len(tensors) * heads * head_dim
    if not 0 <= start <= end <= tokens:
        raise ValueError(f"centered_rows: need 0 <= start <= end <= {tokens} (got {start}, {end})")

    def need(t, name, ok_shape, want):
        if (t is None or t.dtype != torch.float32 or t.device != first.device or not t.is_contiguous()
                or not ok_shape(tuple(t.shape))):
            got = "None" if t is None else f"{t.dtype} {tuple(t.shape)} on {t.device}"
            raise ValueError(f"centered_rows: {name} must be a contiguous float32 tensor {want} on {first.device} "
                             f"(got {got})")

    if (cos is None) != (sin is None):
        raise ValueError("centered_rows: give both cos and sin (keys) or neither (values)")
    if cos is not None:
        for t, name in ((cos, "cos"), (sin, "sin")):
            need(t, name, lambda sh: len(sh) == 2 and sh[0] >= end and sh[1] == head_dim,
                 f"[>= {end} positions, {head_dim}]")
    need(mean, "mean", lambda sh: sh == (width,), f"[{width}]")
    need(out, "out", lambda sh: sh == (end - start, width), f"[{end - start}, {width}]")
    ptrs = torch.tensor([ptr(t) for t in tensors], dtype=torch.int64).to(first.device)
    with _on_device_of(first):
        _check(lib().dkv_centered_rows(c_vp(ptr(ptrs)), c_i32(_DTYPE[first.dtype]), c_i32(len(tensors)), c_i32(heads),
                                       c_i32(tokens), c_i32(head_dim), c_vp(ptr(cos)), c_vp(ptr(sin)), c_vp(ptr(mean)),
                                       c_i32(start), c_i32(end), c_vp(ptr(out)), c_vp(stream_handle())),
               "dkv_centered_rows")


def ladder_errors(coef, bits) -> torch.Tensor:
    """coef f32 [n, 64G], bits u8 [R, G] -> squared quantization error of every token at every rung [n, R]."""
    rungs, groups = bits.shape
    _expect("ladder_errors", coef.device, (coef, "coef", torch.float32, (None, 64 * groups)),
            (bits, "bits", torch.uint8, (rungs, groups)))
    errors = torch.empty(coef.shape[0], rungs, dtype=torch.float32, device=coef.device)
    with _on_device_of(coef):
        _check(lib().dkv_ladder_errors(c_vp(ptr(coef)), c_i32(coef.shape[0]), c_i32(groups), c_vp(ptr(bits)), c_i32(rungs),
                                       c_vp(ptr(errors)), c_vp(stream_handle())), "dkv_ladder_errors")
    return errors


def ladder_code(coef, bits, level):
    """coef f32 [n, 64G] at each token's level (int64 [n]: a rung of bits u8 [R, G], R as it is, -1 dropped) ->
    decoded f32 [n, 64G], codes u8 [n, G, 64], low and scale f16 [n, G]."""
    (n, features), (rungs, groups) = coef.shape, bits.shape
    _expect("ladder_code", coef.device, (coef, "coef", torch.float32, (n, 64 * groups)),
            (bits, "bits", torch.uint8, (rungs, groups)), (level, "level", torch.int64, (n,)))
    decoded = torch.empty_like(coef)
    codes = torch.empty(n, groups, features // groups, dtype=torch.uint8, device=coef.device)
    low = torch.empty(n, groups, dtype=torch.float16, device=coef.device)
    scale = torch.empty_like(low)
    with _on_device_of(coef):
        _check(lib().dkv_ladder_code(c_vp(ptr(coef)), c_i32(n), c_i32(groups), c_vp(ptr(bits)), c_i32(rungs), c_vp(ptr(level)),
                                     c_vp(ptr(decoded)), c_vp(ptr(codes)), c_vp(ptr(low)), c_vp(ptr(scale)),
                                     c_vp(stream_handle())), "dkv_ladder_code")
    return decoded, codes, low, scale


def to_device(values, dtype, device) -> torch.Tensor:
    """A small host list (or tensor) on ``device`` without waiting for the GPU's earlier work: from pinned memory,
    as a pageable copy synchronizes the stream."""
    host = torch.as_tensor(values, dtype=dtype)
    if torch.device(device).type != "cuda" or host.is_cuda or host.numel() == 0:
        return host.to(device)
    return host.pin_memory().to(device, non_blocking=True)


def _pointer_table(tensors) -> torch.Tensor:
    return to_device([ptr(t) for t in tensors], torch.int64, tensors[0].device)


def rows_to_caches(rows, caches, first: int, gap_start: int, gap_len: int, cos=None, sin=None) -> None:
    """Token-matrix rows f32 [n, L*H*D] into per-layer caches [1, H, T, D] (contiguous, one dtype): row i is token
    first + i, plus gap_len from token gap_start on; keys are rotated when cos / sin [T, D] are given."""
    head = caches[0]
    _, heads, tokens, dim = head.shape
    _expect("rows_to_caches", head.device, (rows, "rows", torch.float32, (None, len(caches) * heads * dim)),
            *((t, "cos and sin", torch.float32, (tokens, dim)) for t in (cos, sin) if t is not None))
    table = _pointer_table(caches)
    with _on_device_of(head):
        _check(lib().dkv_rows_to_caches(c_vp(ptr(rows)), c_i32(rows.shape[0]), c_i32(first), c_i32(gap_start), c_i32(gap_len),
                                        c_vp(ptr(table)), c_i32(dtype_code(head.dtype)), c_i32(len(caches)), c_i32(heads),
                                        c_i32(tokens), c_i32(dim), c_vp(ptr(cos)), c_vp(ptr(sin)), c_vp(stream_handle())),
               "dkv_rows_to_caches")


def copy_tokens(src, dst, skip: int, skip_len: int) -> None:
    """Every token outside [skip, skip + skip_len) of per-layer caches [1, H, T, D] (contiguous, one dtype) into others."""
    if len(dst) != len(src):
        raise ValueError(f"copy_tokens: dst must be {len(src)} caches (got {len(dst)})")
    _expect("copy_tokens", src[0].device, (dst[0], "dst", src[0].dtype, src[0].shape))
    _, heads, tokens, dim = src[0].shape
    a, b = _pointer_table(src), _pointer_table(dst)
    with _on_device_of(src[0]):
        _check(lib().dkv_copy_tokens(c_vp(ptr(a)), c_vp(ptr(b)), c_i32(dtype_code(src[0].dtype)), c_i32(len(src)), c_i32(heads),
                                     c_i32(tokens), c_i32(dim), c_i32(skip), c_i32(skip_len), c_vp(stream_handle())),
               "dkv_copy_tokens")


def outside_tokens(src, skip: int, skip_len: int) -> torch.Tensor:
    """Every token outside [skip, skip + skip_len) of per-layer caches [1, H, T, D] (contiguous, one dtype):
    [L, 1, H, T - skip_len, D]."""
    _, heads, tokens, dim = src[0].shape
    out = torch.empty(len(src), 1, heads, tokens - skip_len, dim, dtype=src[0].dtype, device=src[0].device)
    table = (c_i64 * len(src))(*[ptr(t) for t in src])
    with _on_device_of(out):
        _check(lib().dkv_outside_tokens(table, c_vp(ptr(out)), c_i32(dtype_code(out.dtype)), c_i32(len(src)), c_i32(heads),
                                        c_i32(tokens), c_i32(dim), c_i32(skip), c_i32(skip_len), c_vp(stream_handle())),
               "dkv_outside_tokens")
    return out


def matmul_f32(a: torch.Tensor, b: torch.Tensor, bias: torch.Tensor | None = None) -> torch.Tensor:
    """a [M, K] @ b [K, N] (+ bias [N]) for float32 GPU matrices, on the fp16 matrix cores with float32's
    accuracy (dkv_matmul_f32).  ``a`` has unit stride along its rows, ``b`` along either dimension (the
    transpose of a row-major [N, K] is read as it lies)."""
    for t, name, dims in ((a, "a", 2), (b, "b", 2), (bias, "bias", 1)):
        if t is not None and (t.dtype != torch.float32 or not t.is_cuda or t.device != a.device or t.dim() != dims):
            raise ValueError(f"matmul_f32: {name} must be a float32 GPU tensor of {dims} dimensions")
    (m, k), (kb, n) = a.shape, b.shape
    if k != kb or (bias is not None and bias.shape[0] != n) or min(m, n, k) == 0:
        raise ValueError(f"matmul_f32: shapes {tuple(a.shape)} @ {tuple(b.shape)} do not match")
    if a.stride(1) != 1 or a.stride(0) < k:
        a = a.contiguous()
    kn = b.stride(1) == 1 and b.stride(0) >= n
    if not kn and not (b.stride(0) == 1 and b.stride(1) >= k):
        b, kn = b.contiguous(), True
    # (a dimension of one element may have any stride, contiguous() or not)
    lda, ldb = max(a.stride(0), k), max(b.stride(0), n) if kn else max(b.stride(1), k)
    if bias is not None:
        bias = bias.contiguous()
    out = torch.empty(m, n, dtype=torch.float32, device=a.device)
    need = lib().dkv_matmul_f32_workspace_bytes(c_i64(m), c_i64(n), c_i64(k))
    if need == 0:
        _check(-2, "dkv_matmul_f32_workspace_bytes")
    workspace = torch.empty(need, dtype=torch.uint8, device=a.device)
    with _on_device_of(a):
        _check(lib().dkv_matmul_f32(c_vp(a.data_ptr()), c_i64(lda), c_vp(b.data_ptr()), c_i64(ldb), c_i32(kn),
                                    c_vp(ptr(bias)), c_i64(m), c_i64(n), c_i64(k), c_vp(ptr(out)), c_i64(n),
                                    c_vp(ptr(workspace)), c_sz(need), c_vp(stream_handle())), "dkv_matmul_f32")
    return out


def live_groups(coef, codes=None, low=None, scale=None) -> torch.Tensor:
    """bool [G]: the 64-wide groups of coef f32 [n, 64G] that some row uses.  With ladder codes u8 [n, G, 64], low and scale
    f16 [n, G], coef is written first: code * scale + low."""
    n, groups = coef.shape[0], coef.shape[1] // 64
    _expect("live_groups", coef.device, (coef, "coef", torch.float32, (n, 64 * groups)))
    if codes is not None:
        _expect("live_groups", coef.device, (codes, "codes", torch.uint8, (n, groups, 64)),
                *((t, "low and scale", torch.float16, (n, groups)) for t in (low, scale)))
    live = torch.zeros(groups, dtype=torch.int32, device=coef.device)
    with _on_device_of(coef):
        _check(lib().dkv_live_groups(c_vp(ptr(codes)), c_vp(ptr(low)), c_vp(ptr(scale)), c_vp(ptr(coef)), c_i64(n), c_i32(groups),
                                     c_vp(ptr(live)), c_vp(stream_handle())), "dkv_live_groups")
    return live.bool()


def project_caches(tensors, cos, sin, mean, start: int, end: int, basis, with_energy: bool):
    """Centred rows of per-layer caches [1, H, T, D] times basis f32 [L*H*D, rank]: f32 [end - start, rank], and the rows'
    energies [end - start] or None (dkv_project_caches; contiguous 16-byte aligned tensors, cos and sin for keys)."""
    first = tensors[0]
    _, heads, tokens, dim = first.shape
    (k, n), m = basis.shape, end - start
    if (k != len(tensors) * heads * dim or mean.shape != (k,)
            or any(t is not None and (t.shape[0] < end or t.shape[1:] != (dim,)) for t in (cos, sin))):
        raise ValueError(f"project_caches: basis and mean must be of {len(tensors) * heads * dim} columns, cos and sin of "
                         f"{end} tokens and {dim} dimensions")
    kn = basis.stride(1) == 1 and basis.stride(0) >= n
    if not kn and not (basis.stride(0) == 1 and basis.stride(1) >= k):
        basis, kn = basis.contiguous(), True
    out = torch.empty(m, n, dtype=torch.float32, device=first.device)
    energy = torch.empty(m, dtype=torch.float32, device=first.device) if with_energy else None
    need = lib().dkv_matmul_f32_workspace_bytes(c_i64(m), c_i64(n), c_i64(k))
    if need == 0:
        _check(-2, "dkv_matmul_f32_workspace_bytes")
    workspace = torch.empty(need, dtype=torch.uint8, device=first.device)
    table = _pointer_table(tensors)
    with _on_device_of(first):
        _check(lib().dkv_project_caches(c_vp(ptr(table)), c_i32(dtype_code(first.dtype)), c_i32(len(tensors)), c_i32(heads),
                                        c_i32(tokens), c_i32(dim), c_vp(ptr(cos)), c_vp(ptr(sin)), c_vp(ptr(mean)),
                                        c_i32(start), c_i32(end), c_vp(basis.data_ptr()),
                                        c_i64(max(basis.stride(0), n) if kn else max(basis.stride(1), k)), c_i32(kn), c_i64(n), c_vp(ptr(out)),
                                        c_i64(n), c_vp(ptr(energy)), c_vp(ptr(workspace)), c_sz(need), c_vp(stream_handle())),
               "dkv_project_caches")
    return out, energy


def quantize8(coef, codes, low, span, errors=None) -> None:
    """coef f32 [n, 64G] -> codes u8 [n, G, 64], low/span f16 bits [n, G], errors f32 [n, G, 9] or None."""
    n, groups = codes.shape[0], codes.shape[1]
    with _on_device_of(codes):
        _check(lib().dkv_quantize8(c_vp(ptr(coef)), c_i32(n), c_i32(groups), c_vp(ptr(codes)), c_vp(ptr(low)),
                                   c_vp(ptr(span)), c_vp(ptr(errors)), c_vp(stream_handle())), "dkv_quantize8")


def quantize8_rungs(coef, planes, codes, low, span, errors, energy) -> None:
    """coef f32 [n, 64G], planes u8 [R, G] -> codes, low, span as quantize8's, errors f32 [n, R], energy f32 [n]."""
    n, groups = codes.shape[0], codes.shape[1]
    if coef.shape != (n, 64 * groups) or errors.shape != (n, planes.shape[0]) or planes.shape[1:] != (groups,):
        raise ValueError(f"quantize8_rungs: coef must be [{n}, {64 * groups}], planes [rungs, {groups}], errors [{n}, rungs]")
    with _on_device_of(codes):
        _check(lib().dkv_quantize8_rungs(c_vp(ptr(coef)), c_i32(n), c_i32(groups), c_vp(ptr(planes)), c_i32(planes.shape[0]),
                                         c_vp(ptr(codes)), c_vp(ptr(low)), c_vp(ptr(span)), c_vp(ptr(errors)),
                                         c_vp(ptr(energy)), c_vp(stream_handle())), "dkv_quantize8_rungs")


def dequantize_codes(codes, low, span, planes, out) -> None:
    n, groups = codes.shape[0], codes.shape[1]
    _check(lib().dkv_dequantize_codes(c_vp(ptr(codes)), c_vp(ptr(low)), c_vp(ptr(span)), c_vp(ptr(planes)),
                                      c_i32(planes.shape[0]), c_i32(n), c_i32(groups), c_vp(ptr(out)),
                                      c_vp(stream_handle())), "dkv_dequantize_codes")


def prepare_key_basis(basis, layers, kv_heads, head_dim, rank, out) -> None:
    _check(lib().dkv_prepare_key_basis(c_vp(ptr(basis)), c_i32(layers), c_i32(kv_heads), c_i32(head_dim),
                                       c_i32(rank), c_vp(ptr(out)), c_vp(stream_handle())), "dkv_prepare_key_basis")


def prepare_value_basis(basis, layers, kv_heads, head_dim, rank, out) -> None:
    _check(lib().dkv_prepare_value_basis(c_vp(ptr(basis)), c_i32(layers), c_i32(kv_heads), c_i32(head_dim),
                                         c_i32(rank), c_vp(ptr(out)), c_vp(stream_handle())),
           "dkv_prepare_value_basis")


def attend_workspace_bytes(args: AttendArgs) -> int:
    n = lib().dkv_attend_workspace_bytes(ctypes.byref(args))
    if n == 0:
        _check(-2, "dkv_attend_workspace_bytes")
    return n


def attend_prepare(args: AttendArgs, workspace: torch.Tensor, plane_cap: int = 8, values: bool = True) -> None:
    """K1 into the workspace: every token's key codes decoded (to ``plane_cap`` planes) for K2, and
    the value codes for K3 unless ``values`` is False (question scoring reads keys only)."""
    if not values:
        args = AttendArgs.from_buffer_copy(args)
        args.value = Stream()  # no value blob: the library decodes the keys alone
    _check(lib().dkv_attend_prepare(ctypes.byref(args), c_i32(plane_cap), c_vp(ptr(workspace)),
                                    c_sz(workspace.numel()), c_vp(stream_handle())), "dkv_attend_prepare")


def attend_layer(args: AttendArgs, workspace: torch.Tensor) -> None:
    _check(lib().dkv_attend_layer(ctypes.byref(args), c_vp(ptr(workspace)), c_sz(workspace.numel()),
                                  c_vp(stream_handle())), "dkv_attend_layer")


def attend_layer_noalloc(args: AttendArgs) -> None:
    """K1 decode + one layer with the library's static workspace (no allocation anywhere, for
    callers that cannot allocate).  Contexts whose workspace exceeds NOALLOC_MAX_BYTES are refused;
    calls that overlap on one GPU share that workspace and race."""
    _check(lib().dkv_attend_layer_noalloc(ctypes.byref(args), c_vp(stream_handle())), "dkv_attend_layer_noalloc")


def attend_scores(args: AttendArgs, workspace: torch.Tensor) -> None:
    _check(lib().dkv_attend_scores(ctypes.byref(args), c_vp(ptr(workspace)), c_sz(workspace.numel()),
                                   c_vp(stream_handle())), "dkv_attend_scores")


def attend_values(args: AttendArgs, workspace: torch.Tensor) -> None:
    _check(lib().dkv_attend_values(ctypes.byref(args), c_vp(ptr(workspace)), c_sz(workspace.numel()),
                                   c_vp(stream_handle())), "dkv_attend_values")


def score_workspace_bytes(args: AttendArgs) -> int:
    n = lib().dkv_score_workspace_bytes(ctypes.byref(args))
    if n == 0:
        _check(-2, "dkv_score_workspace_bytes")
    return n


def score_begin(importance: torch.Tensor) -> None:
    _check(lib().dkv_score_begin(c_vp(ptr(importance)), c_i32(importance.numel()), c_vp(stream_handle())),
           "dkv_score_begin")


def score_layer(args: AttendArgs, key_question: torch.Tensor, importance: torch.Tensor,
                workspace: torch.Tensor) -> None:
    _check(lib().dkv_score_layer(ctypes.byref(args), c_vp(ptr(key_question)), c_vp(ptr(importance)),
                                 c_vp(ptr(workspace)), c_sz(workspace.numel()), c_vp(stream_handle())),
           "dkv_score_layer")


def topk(scores: torch.Tensor, k: int, out: torch.Tensor) -> None:
    _check(lib().dkv_topk(c_vp(ptr(scores)), c_i32(scores.numel()), c_i32(k), c_vp(ptr(out)), c_vp(None), c_sz(0),
                          c_vp(stream_handle())), "dkv_topk")


def refine_rows(stream: Stream, n: int, cold, cold_tok_off, rows, refined_base_off: int, blob, tok_off, pieces,
                owner, version: int, fetched) -> None:
    """K4c over any token list on the device (dkv_refine_rows): ``fetched`` [2] int64, zero on entry,
    gets the reference's byte count and the out-of-range flag."""
    k = rows.numel()
    refined_ptr = ptr(blob) + refined_base_off
    _check(lib().dkv_refine_rows(ctypes.byref(stream), c_i32(n), c_vp(ptr(cold)), c_vp(ptr(cold_tok_off)),
                                 c_vp(ptr(rows)), c_i32(k), c_vp(refined_ptr), c_i64(refined_base_off),
                                 c_vp(ptr(tok_off)), c_vp(ptr(pieces)), c_vp(ptr(owner)), c_i32(version),
                                 c_vp(ptr(fetched)), c_vp(stream_handle())), "dkv_refine_rows")


def gather_cold(stream: Stream, cold, cold_tok_off, idx, refined_base_off: int, blob, tok_off, pieces) -> None:
    k = idx.numel()
    refined_ptr = ptr(blob) + refined_base_off
    _check(lib().dkv_gather_cold(ctypes.byref(stream), c_vp(ptr(cold)), c_vp(ptr(cold_tok_off)), c_vp(ptr(idx)),
                                 c_i32(k), c_vp(refined_ptr), c_i64(refined_base_off), c_vp(ptr(tok_off)),
                                 c_vp(ptr(pieces)), c_vp(stream_handle())), "dkv_gather_cold")
