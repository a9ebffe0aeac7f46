"""Launches and scratch as the host code asks for them: device tensors stand in as
CPU ones, the library as a stub that notes each call, the current device and the
stream."""

from __future__ import annotations

import importlib
from contextlib import ExitStack, contextmanager
from unittest.mock import patch

import pytest

torch = pytest.importorskip("torch")

import tensorsmith_hip as ts  # noqa: E402
from tensorsmith_hip import _lib, nn  # noqa: E402
from tensorsmith_hip.nn import functional as F  # noqa: E402

A = importlib.import_module("tensorsmith_hip.nn.attention")
D = importlib.import_module("tensorsmith_hip.device")


class Stub:
    """Every entry point; the queries give 256 bytes, the launches succeed."""

    def __init__(self):
        self.current, self.calls, self.asked, self.args = 0, [], [], {}

    def __getattr__(self, name):
        if name.endswith("_workspace"):
            return lambda *a: self.asked.append(name) or 256
        return lambda *a: self.args.update({name: a}) or self.calls.append((name, self.current, a[-1])) or 0

    @contextmanager
    def device(self, index):
        before, self.current = self.current, index
        yield
        self.current = before


@pytest.fixture
def lib():
    lib = Stub()
    with ExitStack() as stack:
        for patched in (patch.object(D.Device, "torch", torch.device("cpu")),
                        patch.object(D, "is_available", lambda value: True),
                        patch.object(D, "current_stream", lambda dev: 0x100 + dev.index),
                        patch.object(A, "current_stream", lambda dev: 0x100 + dev.index),
                        patch.object(torch.cuda, "current_device", lambda: lib.current),
                        patch.object(torch.cuda, "device", lib.device),
                        patch.object(_lib, "load", lambda: lib)):
            stack.enter_context(patched)
        yield lib


@pytest.mark.parametrize("index", [0, 1])
def test_layers_launch_on_their_tensors_device(lib, index):
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


def _attend(dtype=torch.float16, heads=2, s=2000, mask=None, dropout=0.0, q_len=16, causal=True):
    q, k, v = (ts.Tensor(torch.randn(1, heads, n, 64).to(dtype), device="hip") for n in (q_len, s, s))
    mask = None if mask is None else ts.Tensor(mask, device="hip")
    return nn.scaled_dot_product_attention(q, k, v, mask, dropout, causal and dropout == 0.0,
                                           causal_offset=s - q_len if causal and dropout == 0.0 else 0)


def test_split_scratch_is_asked_for_where_a_forward_can_split(lib):
    _attend()
    _attend(mask=torch.ones(1, 1, 1, 2000, dtype=torch.bool))  # key padding
    assert lib.asked.count("tsattn_sdpa_forward_workspace") == 2
    for kw in (dict(dtype=torch.float32), dict(dropout=0.5), dict(mask=torch.ones(16, 2000, dtype=torch.bool)),
               dict(mask=torch.ones(16, 2000)), dict(heads=257), dict(heads=129, q_len=129), dict(s=1500)):
        _attend(**kw)
    assert lib.asked.count("tsattn_sdpa_forward_workspace") == 2
    assert [name for name, _, _ in lib.calls].count("tsattn_sdpa_forward_split") == 9


@pytest.mark.parametrize("dims,q_len,kv_len,causal,offset,pays", [
    # a split call is 21 - 24 us of host time: over fewer keys the unsplit kernel is through before
    ((128, 128), 16, 1181, False, 0, False), ((128, 128), 16, 1182, False, 0, True),
    ((64, 64), 16, 1565, True, 1549, False), ((64, 64), 16, 1566, True, 1550, True),
    ((32, 32), 16, 1757, False, 0, False), ((32, 32), 16, 1758, False, 0, True),
    ((64, 128), 16, 1373, False, 0, False), ((128, 64), 16, 1374, False, 0, True),
    # a causal window that ends before the keys do
    ((128, 128), 1000, 8000, True, 0, False), ((128, 128), 1000, 8000, True, 182, True)])
def test_splits_that_their_host_time_hides(dims, q_len, kv_len, causal, offset, pays):
    p = _lib.Problem()
    p.dtype, p.batch, p.heads_q, p.heads_kv = _lib.BF16, 1, 4, 4
    p.len_q, p.len_kv, p.dim_qk, p.dim_v = q_len, kv_len, *dims
    p.is_causal, p.causal_offset, p.mask_kind = int(causal), offset, _lib.MASK_NONE
    assert A._split_pays(p) == pays


def test_without_room_for_scratch_the_unsplit_paths_run(lib):
    """Split forwards and weight gradients take scratch that the paths before them
    did not: memory that has no room for it still runs those."""
    empty = torch.empty

    def full(*a, **kw):
        if kw.get("dtype") == torch.uint8:
            raise torch.OutOfMemoryError
        return empty(*a, **kw)

    x, w = (ts.Tensor(torch.randn(s).half(), device="hip", requires_grad=True) for s in ((4096, 64), (64, 64)))
    out = F.linear(x, w)
    with patch.object(torch, "empty", full):
        _attend()
        out.backward(ts.Tensor(torch.ones(4096, 64).half(), device="hip"))
    assert not any(name == "tsattn_linear_wgrad" for name, _, _ in lib.calls)
    assert lib.args["tsattn_sdpa_forward_split"][7:9] == (None, 0)  # workspace and its bytes
    want = torch.ones(64, 4096).double() @ x._data.double()
    assert ((w.grad._data.double() - want).norm() / want.norm()).item() <= 2e-3


def test_layers_outside_the_kernels_take_the_plain_path(lib):
    """Host time is what bounds small layers: without autocast a linear layer enters no
    cast context, and what the kernels' first condition rules out asks nothing more."""
    def refuse(*a, **kw):
        raise AssertionError("asked")

    draw = lambda *s: ts.Tensor(torch.randn(s), device="hip", requires_grad=True)
    with patch.object(F, "no_grad", refuse), patch.object(F, "_rows_pays", refuse), \
            patch.object(F, "_wgrad_pays", refuse), patch.object(F, "_code", refuse):
        F.linear(draw(3, 100), draw(50, 100), draw(50)).backward(draw(3, 50))
        F.linear(draw(5000, 8), draw(8, 8)).backward(draw(5000, 8))
        F.rms_norm(draw(5, 100), draw(100)).backward(draw(5, 100))
    assert not lib.calls and not lib.asked
