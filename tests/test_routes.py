"""What the HIP entry points of the codecs promise callers whose calls were tensor operations before (CPU): the device
and stream they launch on, the calls they leave to torch, and what they refuse.  No kernel runs: a stub stands in for
the library and records what would be launched."""

from __future__ import annotations

import pytest
import torch

import dkv_hip


class Launches:
    """Stands in for the library; ``log`` holds (entry point, current device at the call, its stream argument)."""

    def __init__(self, monkeypatch):
        self.log, self.current = [], "elsewhere"
        outer = self

        class Device:
            def __init__(self, device):
                self.device = device

            def __enter__(self):
                self.before, outer.current = outer.current, str(self.device)

            def __exit__(self, *exc):
                outer.current = self.before

        monkeypatch.setattr(torch.cuda, "device", Device)
        monkeypatch.setattr(dkv_hip, "_current_device", lambda: 5)  # CPU tensors say -1
        monkeypatch.setattr(dkv_hip, "lib", lambda: self)
        monkeypatch.setattr(dkv_hip, "ptr", lambda t: None if t is None else t.data_ptr())
        monkeypatch.setattr(dkv_hip, "stream_handle", lambda: hash(self.current) & 0xFFFF)

    def __getattr__(self, name):
        if not name.startswith("dkv_"):
            raise AttributeError(name)

        def call(*args):
            if name.endswith("workspace_bytes"):
                return 256
            self.log.append((name, self.current, args[-1].value))
            return 0

        return call


def _wrapped_calls():
    coef, bits = torch.zeros(3, 128), torch.zeros(4, 2, dtype=torch.uint8)
    codes = torch.zeros(3, 2, 64, dtype=torch.uint8)
    low, scale = (torch.zeros(3, 2, dtype=torch.float16) for _ in range(2))
    caches = [torch.zeros(1, 2, 5, 64) for _ in range(2)]
    cos, mean = torch.ones(5, 64), torch.zeros(256)
    return {
        "dkv_ladder_errors": lambda: dkv_hip.ladder_errors(coef, bits),
        "dkv_ladder_code": lambda: dkv_hip.ladder_code(coef, bits, torch.zeros(3, dtype=torch.int64)),
        "dkv_live_groups": lambda: dkv_hip.live_groups(coef, codes, low, scale),
        "dkv_rows_to_caches": lambda: dkv_hip.rows_to_caches(torch.zeros(3, 256), caches, 1, 5, 0, cos, cos),
        "dkv_copy_tokens": lambda: dkv_hip.copy_tokens(caches, [c.clone() for c in caches], 1, 3),
        "dkv_outside_tokens": lambda: dkv_hip.outside_tokens(caches, 1, 3),
        "dkv_centered_rows": lambda: dkv_hip.centered_rows(caches, cos, cos, mean, 1, 4, torch.empty(3, 256)),
        "dkv_quantize8": lambda: dkv_hip.quantize8(coef, codes, low, scale),
        "dkv_quantize8_rungs": lambda: dkv_hip.quantize8_rungs(coef, bits, codes, low, scale, torch.zeros(3, 4), torch.zeros(3)),
    }


@pytest.mark.parametrize("name", list(_wrapped_calls()))
def test_kernels_launch_on_their_tensors_device(name, monkeypatch):
    """A codec on a GPU that is not the current one: the launch goes to that GPU's stream, which orders it behind the
    work that wrote the tensors."""
    launches = Launches(monkeypatch)
    _wrapped_calls()[name]()
    assert launches.log == [(name, "cpu", hash("cpu") & 0xFFFF)]
    assert launches.current == "elsewhere"


def _codec(layers=2, heads=2, dim=64, rank=64):
    import kvtc
    import synth

    shape = synth.ModelShape(layers, heads, dim, heads, rank)
    return kvtc.KVTCCodec(synth.kvtc_checkpoint(synth.make_context(shape, 60, seed=2)), "cpu", synth.RopeModel(shape))


@pytest.mark.parametrize("change", ["wide rows", "narrow rows", "narrow tables", "short tables", "heads", "short span"])
def test_rebuilt_caches_of_other_shapes_are_left_to_torch(change, monkeypatch):
    """rows_to_caches takes its strides from the caches: rows or tables of another width would be read out of range."""
    import kvtc

    launches = Launches(monkeypatch)
    monkeypatch.setattr(kvtc, "_plain_gpu", lambda *t: True)
    codec, tokens, span = _codec(), 20, (4, 12)
    features = 256 + 64 * (change == "wide rows") - 64 * (change == "narrow rows")
    rows = torch.zeros(span[1] - span[0] - (change == "short span"), features)
    cos = torch.ones(tokens - (change == "short tables"), 32 if change == "narrow tables" else 64)
    caches = [torch.zeros(1, 4 if change == "heads" else 2, tokens, 64) for _ in range(2)]
    monkeypatch.setattr(kvtc, "inverse_transform", lambda *a: rows)
    with pytest.raises(RuntimeError):
        codec._rebuilt_caches("key", None, caches, span, cos, cos)
    assert launches.log == []


def test_compress_of_other_shapes_raises_as_torch_does(monkeypatch):
    """Caches of other heads than the calibration's: torch's broadcast error, not the binding's."""
    import kvtc

    monkeypatch.setattr(kvtc, "_plain_gpu", lambda *t: True)
    codec = _codec()
    monkeypatch.setattr(codec, "centered", lambda *a: pytest.fail("the kernel's route"))
    caches = [torch.randn(1, 4, 40, 64) for _ in range(2)]
    with pytest.raises(RuntimeError):
        codec.compress(caches, caches, 0.3, 8, True)


def test_bindings_refuse_shapes_they_would_read_past():
    """On the host, before a pointer is taken (CPU tensors pass the shape checks and are refused as host memory)."""
    f, u8, f16, i64 = torch.float32, torch.uint8, torch.float16, torch.int64
    z = lambda *shape, dtype=f: torch.zeros(*shape, dtype=dtype)  # noqa: E731
    caches, other = [z(1, 2, 5, 64) for _ in range(2)], [z(1, 2, 5, 64), z(1, 2, 4, 64)]
    for call in (
        lambda: dkv_hip.ladder_errors(z(3, 192), z(4, 2, dtype=u8)),
        lambda: dkv_hip.ladder_errors(z(3, 128), z(4, 2)),
        lambda: dkv_hip.ladder_code(z(3, 128), z(4, 2, dtype=u8), z(2, dtype=i64)),
        lambda: dkv_hip.rows_to_caches(z(3, 255), caches, 1, 5, 0),
        lambda: dkv_hip.rows_to_caches(z(3, 256), caches, 1, 5, 0, z(5, 32), z(5, 32)),
        lambda: dkv_hip.copy_tokens(caches, other[1:] * 2, 1, 3),
        lambda: dkv_hip.copy_tokens(caches, caches[:1], 1, 3),
        lambda: dkv_hip.live_groups(z(3, 100)),
        lambda: dkv_hip.live_groups(z(3, 128), z(2, 2, 64, dtype=u8), z(3, 2, dtype=f16), z(3, 2, dtype=f16)),
        lambda: dkv_hip.quantize8_rungs(z(3, 128), z(4, 3, dtype=u8), z(3, 2, 64, dtype=u8), z(3, 2), z(3, 2), z(3, 4), z(3)),
        lambda: dkv_hip.project_caches(caches, None, None, z(256), 1, 4, z(255, 8), False),
        lambda: dkv_hip.project_caches(caches, None, None, z(255), 1, 4, z(256, 8), False),
        lambda: dkv_hip.project_caches(caches, z(5, 32), z(5, 32), z(256), 1, 4, z(256, 8), False),
    ):
        with pytest.raises(ValueError, match="must be"):
            call()


def test_ladder_kernels_need_a_size_for_every_rung(monkeypatch):
    """The exact level follows the last sized rung; the kernels take it to follow the last row of widths."""
    import kvtc

    monkeypatch.setattr(kvtc, "_plain_gpu", lambda *t: True)
    codec = _codec()
    coef = torch.zeros(3, 64)
    assert codec._ladder_on_gpu(coef, "key")
    codec.streams["key"].rung_bytes = codec.streams["key"].rung_bytes[:-1]
    assert not codec._ladder_on_gpu(coef, "key")


def test_recorded_calls_are_left_to_torch():
    """A trace of a call must hold its operations: a kernel's output would be a constant in it."""
    import kvtc
    from torch.fx.experimental.proxy_tensor import make_fx
    from torch.utils.flop_counter import FlopCounterMode

    seen = []

    def watched(x):
        seen.append(kvtc._watched())
        return x + 1

    x = torch.ones(2)
    watched(x)
    torch.jit.trace(watched, x, check_trace=False)
    make_fx(watched)(x)
    with FlopCounterMode(display=False):
        watched(x)
    torch.func.vmap(watched)(x)
    torch.func.jvp(watched, (x,), (x,))
    torch.compile(watched, backend="eager")(x)
    watched(x)
    assert seen[0] is False and seen[-1] is False and len(seen) >= 8 and all(seen[1:-1])


@pytest.mark.parametrize("rows,k,n,row_major,pays", [
    (103, 28672, 2048, True, False), (128, 28672, 2048, True, False), (256, 28672, 2048, True, True),
    (400, 4096, 4096, True, False), (480, 4096, 4096, True, True), (700, 8192, 1024, True, False),
    (960, 8192, 1024, True, True), (256, 8192, 8192, True, False), (480, 8192, 8192, True, True),
    (128, 2048, 28672, False, False), (192, 2048, 28672, False, False), (256, 2048, 28672, False, True),
    (500, 1024, 8192, False, False), (720, 1024, 8192, False, True)])
def test_split_products_where_they_measured_faster(rows, k, n, row_major, pays):
    """Both sides of the line, at sizes timed against the library: few rows against a large basis are the library's."""
    import kvtc

    assert kvtc.split_pays(rows, k, n, row_major) is pays


def test_launches_past_their_threads_are_left_to_torch(monkeypatch):
    """Half a million tokens of a large model and more: sizes only, of one element expanded."""
    import kvtc

    monkeypatch.setattr(kvtc, "_plain_gpu", lambda *t: True)
    one = torch.zeros(1)
    for tokens, fits in ((599_186, True), (599_187, False)):
        like = one.half().expand(1, 8, tokens, 128)
        assert kvtc.fit_caches(one.expand(tokens, 28672), like, 28, (0, tokens), ()) is fits
    assert kvtc.split_pays(2**21 - 1, 64, 64, True) and not kvtc.split_pays(2**21, 64, 64, True)
    codec = _codec(rank=64)
    assert codec._ladder_on_gpu(one.expand(2**28 - 1, 64), "key") and not codec._ladder_on_gpu(one.expand(2**28, 64), "key")


def test_launch_on_the_current_device_enters_nothing(monkeypatch):
    launches = Launches(monkeypatch)
    monkeypatch.setattr(dkv_hip, "_current_device", lambda: -1)
    dkv_hip.ladder_errors(torch.zeros(3, 128), torch.zeros(4, 2, dtype=torch.uint8))
    assert launches.log == [("dkv_ladder_errors", "elsewhere", hash("elsewhere") & 0xFFFF)]


@pytest.mark.parametrize("kind,dtype", [("key", torch.float16), ("value", torch.bfloat16), ("key", torch.float32)])
def test_rebuilt_caches_that_fit_take_the_kernels(kind, dtype, monkeypatch):
    import kvtc

    launches = Launches(monkeypatch)
    monkeypatch.setattr(kvtc, "_plain_gpu", lambda *t: True)
    codec, tokens, span = _codec(), 20, (4, 12)
    monkeypatch.setattr(kvtc, "inverse_transform", lambda *a: torch.zeros(8, 256))
    caches = [torch.zeros(1, 2, tokens, 64, dtype=dtype) for _ in range(2)]
    cos = torch.ones(tokens, 64)
    out = codec._rebuilt_caches(kind, None, caches, span, cos, cos)
    assert [t.shape for t in out] == [t.shape for t in caches] and all(t.dtype == dtype for t in out)
    assert [name for name, *_ in launches.log] == ["dkv_rows_to_caches", "dkv_copy_tokens"]
