"""Layer kernels on another device than the current one, on the host: device
tensors stand in as CPU ones, the library as a stub that notes the current
device and the stream of each call."""

from __future__ import annotations

import importlib
from contextlib import ExitStack, contextmanager
from unittest.mock import patch

import pytest

torch = pytest.importorskip("torch")

import tensorsmith_hip as ts  # noqa: E402
from tensorsmith_hip import _lib, nn  # noqa: E402
from tensorsmith_hip.nn import functional as F  # noqa: E402

D = importlib.import_module("tensorsmith_hip.device")


class Stub:
    """Every entry point; the queries give 256 bytes, the launches succeed."""

    def __init__(self):
        self.current, self.calls = 0, []

    def __getattr__(self, name):
        if name.endswith("_workspace"):
            return lambda *a: 256
        return lambda *a: self.calls.append((name, self.current, a[-1])) or 0

    @contextmanager
    def device(self, index):
        before, self.current = self.current, index
        yield
        self.current = before


@pytest.mark.parametrize("index", [0, 1])
def test_layers_launch_on_their_tensors_device(index):
    lib = Stub()
    with ExitStack() as stack:
        for patched in (patch.object(D.Device, "torch", torch.device("cpu")),
                        patch.object(D, "is_available", lambda value: True),
                        patch.object(D, "current_stream", lambda dev: 0x100 + dev.index),
                        patch.object(torch.cuda, "current_device", lambda: lib.current),
                        patch.object(torch.cuda, "device", lib.device),
                        patch.object(_lib, "load", lambda: lib)):
            stack.enter_context(patched)
        dev = f"hip:{index}"
        draw = lambda *s: ts.Tensor(torch.randn(s).half(), device=dev, requires_grad=True)
        w, gate, up = draw(64), draw(4, 64), draw(4, 64)
        F.rms_norm(draw(4, 64), w).backward(draw(4, 64))
        F.layer_norm(draw(4, 64), w, draw(64)).backward(draw(4, 64))
        F._silu_mul(gate, up).backward(draw(4, 64))
        F.linear(draw(4, 64), draw(64, 64))
        F.linear(draw(4096, 64), draw(64, 64)).backward(draw(4096, 64))
        block = nn.TransformerDecoderBlock(256, 4, 512, device=dev).eval()
        block.to(dtype="float16")
        cache = block.attention.new_cache(1, 256, dtype="float16")
        cache.length = 200
        with ts.no_grad():
            block(draw(1, 1, 256), cache=cache)
    names = {name for name, _, _ in lib.calls}
    assert names == {"tsattn_norm_forward", "tsattn_norm_backward", "tsattn_silu_mul", "tsattn_silu_mul_backward",
                     "tsattn_rows_linear", "tsattn_linear_wgrad", "tsattn_cached_step"}
    for name, current, stream in lib.calls:
        assert (current, getattr(stream, "value", stream)) == (index, 0x100 + index), name
    assert lib.current == 0
