"""Few-row linear layers and the cached step that runs on them.

``tsattn_rows_linear`` / ``_swiglu`` against float64 at the edges of their
split (one row, a full and a second row block, a K that ends inside a
64-column chunk, fewer chunks than accumulators, an output that ends inside a
32-channel tile); a decoder block's cached step in one call against the same
layers run one by one.  Bound: one rounding to the dtype per op and the fp32
sums (relative 2^-11 / 2^-8 of the result's scale a rounding).
"""

from __future__ import annotations

import ctypes
import importlib
from unittest.mock import patch

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():  # pragma: no cover - CPU containers
    pytest.skip("no GPU", allow_module_level=True)

import tensorsmith_hip as ts  # noqa: E402
from tensorsmith_hip import _lib, nn  # noqa: E402
from tensorsmith_hip.nn import functional as F  # noqa: E402

T = importlib.import_module("tensorsmith_hip.nn.transformer")
ULP = {torch.float16: 2.0**-11, torch.bfloat16: 2.0**-8}
CODE = {torch.float16: _lib.F16, torch.bfloat16: _lib.BF16}


def _stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def _close(got, want, dtype, roundings):
    scale = want.abs() + want.square().mean().sqrt()
    err = ((got.double() - want).abs() / scale).max().item()
    assert err <= roundings * ULP[dtype] + 2e-6, (err, roundings * ULP[dtype])


SHAPES = [(1, 8, 4), (1, 64, 32), (5, 200, 36), (32, 1000, 100), (33, 512, 2048), (64, 4096, 96), (3, 2048, 16388)]


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows,k,n", SHAPES)
def test_rows_linear_matches_float64(rows, k, n, dt):
    print("rows linear", rows, k, n, dt, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(k + n)
    draw = lambda *s: torch.randn(s, generator=gen, device="cuda").to(dt)
    x, w, b, res = draw(rows, k + 8)[:, :k], draw(n, k), draw(n), draw(rows, n)
    lib = _lib.load()
    for bias, residual in ((None, None), (b, None), (b, res)):
        out = torch.full((rows, n + 4), 7.0, dtype=dt, device="cuda")
        _lib.check(lib.tsattn_rows_linear(
            CODE[dt], rows, k, n, x.data_ptr(), x.stride(0), w.data_ptr(),
            None if bias is None else bias.data_ptr(), None if residual is None else residual.data_ptr(), n,
            out.data_ptr(), n + 4, _stream()), "rows linear")
        want = x.double() @ w.double().t()
        if bias is not None:
            want = want + b.double()
        if residual is not None:
            want = want + res.double()
        _close(out[:, :n], want, dt, 3)
        assert (out[:, n:] == 7).all()
    u = draw(n, k)
    out = torch.empty(rows, n, dtype=dt, device="cuda")
    _lib.check(lib.tsattn_rows_swiglu(CODE[dt], rows, k, n, x.data_ptr(), x.stride(0), w.data_ptr(), u.data_ptr(),
                                      out.data_ptr(), n, _stream()), "rows swiglu")
    gate, up = ((x.double() @ m.double().t()).to(dt).double() for m in (w, u))
    _close(out, gate * torch.sigmoid(gate) * up, dt, 4)


def test_rows_linear_refuses_what_it_does_not_take():
    x, w, out = (torch.zeros(64, 64, dtype=torch.float16, device="cuda") for _ in range(3))
    lib = _lib.load()
    call = lambda rows, k, n, xp=x.data_ptr(): lib.tsattn_rows_linear(
        _lib.F16, rows, k, n, xp, 64, w.data_ptr(), None, None, 0, out.data_ptr(), 64, _stream())
    assert call(65, 64, 64) == _lib.ERR_UNSUPPORTED
    assert call(4, 60, 64) == _lib.ERR_UNSUPPORTED
    assert call(4, 64, 62) == _lib.ERR_UNSUPPORTED
    assert call(4, 64, 64, x.data_ptr() + 2) == _lib.ERR_UNSUPPORTED
    assert call(0, 64, 64) == _lib.ERR_INVALID
    # layers outside it keep their results
    odd = torch.randn(3, 50, device="cuda").half()
    wo = torch.randn(7, 50, device="cuda").half()
    got = F.linear(ts.Tensor(odd, device="hip"), ts.Tensor(wo, device="hip"))._data
    _close(got, odd.double() @ wo.double().t(), torch.float16, 2)


STEPS = [
    # (dtype, embed, heads, kv heads, batch, tokens, past, int8)
    ("float16", 256, 4, 2, 3, 1, 140, False),
    ("bfloat16", 512, 4, 1, 2, 2, 127, False),
    ("float16", 256, 2, 2, 33, 1, 128, False),
    ("bfloat16", 512, 4, 2, 2, 1, 300, True),
    ("float16", 256, 4, 4, 2, 3, 150, True),
]


@pytest.mark.parametrize("case", STEPS, ids=lambda c: "-".join(map(str, c)))
def test_block_step_in_one_call_matches_the_layers(case):
    dtype, embed, heads, kv_heads, batch, tokens, past, int8 = case
    print("block step", case, flush=True)
    ts.seed(3)
    dt = getattr(torch, dtype)
    block = nn.TransformerDecoderBlock(embed, heads, 2 * embed, num_kv_heads=kv_heads, device="hip").eval()
    block.to(dtype=dtype)
    dim = embed // heads
    gen = torch.Generator(device="cuda").manual_seed(past)
    draw = lambda *s: ts.Tensor(torch.randn(s, generator=gen, device="cuda").to(dt), device="hip")
    k, v, x = draw(batch, kv_heads, past, dim), draw(batch, kv_heads, past, dim), draw(batch, tokens, embed)
    got = {}
    for name in ("call", "layers"):
        cache = block.attention.new_cache(batch, 512, dtype=dtype, quantized=int8)
        with ts.no_grad():
            cache.append(k, v)
            _lib.profile_reset()
            _lib.profile_enable(True)
            if name == "call":
                out = block(x, cache=cache)
            else:
                # a wrapped cache method sends the block through its layers
                original = nn.KVCache._project_append
                with patch.object(nn.KVCache, "_project_append", lambda self, *a: original(self, *a)):
                    out = block(x, cache=cache)
            _lib.profile_enable(False)
        probes = _lib.profile_read()
        assert ("rows_swiglu" in probes) == (name == "call"), sorted(probes)
        assert cache.length == past + tokens
        got[name] = (out._data, [t[:, :, past:past + tokens] for t in cache.storage if t is not None])
    # both cache the same rows bit for bit: the projections sum in the same order
    for a, b in zip(got["call"][1], got["layers"][1]):
        assert torch.equal(a, b)
    _close(got["call"][0], got["layers"][0].double(), dt, 8)


MHA_STEPS = [
    # (dtype, embed, heads, kv heads, batch, tokens, past, int8, bias, rotary, causal)
    ("float16", 256, 4, 2, 3, 1, 140, False, True, True, True),
    ("bfloat16", 256, 2, 1, 2, 3, 130, False, True, False, False),
    ("float16", 512, 4, 4, 1, 4, 128, False, False, True, False),
    ("float16", 256, 4, 2, 2, 1, 200, True, True, True, True),
    ("bfloat16", 512, 4, 2, 2, 2, 150, True, True, False, False),
    ("float16", 256, 2, 2, 33, 1, 127, True, False, False, True),
]


@pytest.mark.parametrize("case", MHA_STEPS, ids=lambda c: "-".join(map(str, c)))
def test_attention_step_in_one_call_matches_the_layers(case):
    """The attention layer alone: projection biases (of three weights side by side
    over int8 caches), no rotation, tokens that see each other both ways."""
    dtype, embed, heads, kv_heads, batch, tokens, past, int8, bias, rotary, causal = case
    print("attention step", case, flush=True)
    ts.seed(4)
    dt = getattr(torch, dtype)
    mha = nn.MultiHeadAttention(embed, heads, num_kv_heads=kv_heads, bias=bias, rotary=rotary, device="hip").eval()
    mha.to(dtype=dtype)
    gen = torch.Generator(device="cuda").manual_seed(past)
    draw = lambda *s: ts.Tensor(torch.randn(s, generator=gen, device="cuda").to(dt), device="hip")
    k, v, x = (draw(batch, kv_heads, past, embed // heads), draw(batch, kv_heads, past, embed // heads),
               draw(batch, tokens, embed))
    got, original, steps = {}, nn.KVCache._project_append, []
    step = T._cached_step
    for name in ("call", "layers"):
        cache = mha.new_cache(batch, 256, dtype=dtype, quantized=int8)
        with (ts.no_grad(), patch.object(T, "_cached_step", lambda *a, **kw: steps.append(step(*a, **kw)) or steps[-1]),
              patch.object(nn.KVCache, "_project_append",
                           original if name == "call" else lambda self, *a: original(self, *a))):
            cache.append(k, v)
            out = mha(x, cache=cache, is_causal=causal)
        assert (steps.pop() is None) == (name == "layers")
        assert cache.length == past + tokens
        got[name] = (out._data, [t[:, :, past:past + tokens] for t in cache.storage if t is not None])
    for a, b in zip(got["call"][1], got["layers"][1]):
        assert torch.equal(a, b)
    _close(got["call"][0], got["layers"][0].double(), dt, 6)


def test_block_step_leaves_replaced_layers_alone():
    """A block whose layer was replaced runs that layer."""
    class Doubled(nn.RMSNorm):
        def forward(self, input):
            return super().forward(input) * 2.0

    block = nn.TransformerDecoderBlock(256, 4, 512, device="hip").eval()
    block.to(dtype="float16")
    cache = block.attention.new_cache(1, 256, dtype="float16")
    x = ts.Tensor(torch.randn(1, 200, 256, device="cuda").half(), device="hip")
    one = ts.Tensor(torch.randn(1, 1, 256, device="cuda").half(), device="hip")
    with ts.no_grad():
        block(x, cache=cache)
        plain = block(one, cache=cache)
        cache.truncate(200)
        norm = Doubled(256, device="hip")
        norm.to(dtype="float16")
        block.ffn_norm = norm
        changed = block(one, cache=cache)
        cache.truncate(200)
        with pytest.raises(ValueError, match="capacity"):
            block(x, cache=cache)
    assert not torch.equal(plain._data, changed._data)
    assert cache.length == 200


def test_rows_of_a_large_tensor_and_bad_eps_stay_with_the_layers():
    """The last position of a long batch (a row stride past the kernel's 32-bit
    offsets) is multiplied all the same; a norm's eps is checked in a cached step."""
    far = torch.empty(2, 2**20, 512, dtype=torch.float16, device="cuda")[:, -1]
    far.copy_(torch.randn(2, 512, device="cuda"))
    w = torch.randn(64, 512, device="cuda").half()
    assert (far.shape[0] * far.stride(0) + 512) * 2 >= 2**31
    got = F.linear(ts.Tensor(far, device="hip"), ts.Tensor(w, device="hip"))._data
    _close(got, far.double() @ w.double().t(), torch.float16, 2)
    block = nn.TransformerDecoderBlock(256, 4, 512, device="hip").eval()
    block.to(dtype="float16")
    cache = block.attention.new_cache(1, 256, dtype="float16")
    x = ts.Tensor(torch.randn(1, 200, 256, device="cuda").half(), device="hip")
    with ts.no_grad():
        block(x, cache=cache)
        block.ffn_norm.eps = 0.0
        with pytest.raises(ValueError, match="eps"):
            block(x[:, :1], cache=cache)
