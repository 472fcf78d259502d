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
