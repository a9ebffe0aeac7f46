"""Which blocks the cached step in one call takes, on the host: device tensors
stand in as CPU ones and the library as a stub that only counts its calls."""

from __future__ import annotations

import importlib
from contextlib import ExitStack
from types import SimpleNamespace
from unittest.mock import patch

import pytest

torch = pytest.importorskip("torch")

import tensorsmith_hip as ts  # noqa: E402
from tensorsmith_hip import _lib, nn  # noqa: E402

D = importlib.import_module("tensorsmith_hip.device")
T = importlib.import_module("tensorsmith_hip.nn.transformer")
Module = importlib.import_module("tensorsmith_hip.nn.module").Module


@pytest.fixture
def stub():
    calls = []
    lib = SimpleNamespace(tsattn_cached_step_workspace=lambda desc: 256,
                          tsattn_cached_step=lambda *a: calls.append(a) or 0)
    with ExitStack() as stack:
        for patched in (patch.object(D.Device, "torch", torch.device("cpu")),
                        patch.object(D, "is_available", lambda value: True),
                        patch.object(D, "current_stream", lambda dev: 0),
                        patch.object(torch.cuda, "current_device", lambda: 0),
                        patch.object(_lib, "load", lambda: lib)):
            stack.enter_context(patched)
        yield calls


class Half(Module):
    def forward(self, input):
        return input * 0.5


class Scaled(nn.Dropout):
    def forward(self, input):
        return super().forward(input) * 0.5


def _instance(layer):
    layer.forward = lambda input: input * 0.5
    return layer


def _block():
    block = nn.TransformerDecoderBlock(256, 4, 512, num_kv_heads=2, dropout=0.1, device="hip").eval()
    block.to(dtype="float16")
    return block


def _step(block, whole=True):
    cache = block.attention.new_cache(1, 256, dtype="float16")
    cache.length = 200
    x = ts.Tensor(torch.randn(1, 1, 256).half(), device="hip")
    out = T._cached_step(x, block.attention, cache, block=block if whole else None)
    assert cache.length == 200 + (out is not None)
    return out


def test_a_plain_block_is_one_call(stub):
    block = _block()
    assert _step(block) is not None and len(stub) == 1
    assert _step(block, whole=False) is not None and len(stub) == 2  # the attention layer alone


@pytest.mark.parametrize("where", ["residual_dropout", "ffn.dropout"])
@pytest.mark.parametrize("layer", [lambda: Half(), lambda: Scaled(0.1), lambda: _instance(nn.Dropout(0.1)),
                                   lambda: nn.Dropout(1.5)], ids=["module", "subclass", "instance", "bad p"])
def test_whatever_stands_in_a_dropouts_place_is_run(stub, where, layer):
    block = _block()
    setattr(block.ffn if where == "ffn.dropout" else block, "dropout" if where == "ffn.dropout" else where,
            layer().eval())
    assert _step(block) is None and not stub


def test_a_dropout_that_drops_is_run(stub):
    block = _block()
    block.ffn.dropout.train()
    assert _step(block) is None and not stub
    block.ffn.dropout.p = 0.0
    assert _step(block) is not None


@pytest.mark.parametrize("cls,name", [(Module, "__call__"), (nn.Linear, "forward"), (nn.RMSNorm, "forward"),
                                      (nn.SwiGLU, "forward"), (nn.Dropout, "forward"),
                                      (nn.MultiHeadAttention, "forward"), (nn.KVCache, "_project_append"),
                                      (nn.KVCache, "get")], ids=lambda v: getattr(v, "__name__", v))
def test_a_method_replaced_on_its_class_is_run(stub, cls, name):
    block = _block()
    original = getattr(cls, name)
    with patch.object(cls, name, lambda self, *a, **k: original(self, *a, **k)):
        assert _step(block) is None and not stub
    assert _step(block) is not None
