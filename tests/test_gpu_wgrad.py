"""The split weight-gradient kernel against float64.

Edges: fewer tokens than one stage, a split that ends inside a stage, more
splits than one reducing pass, eight and four splits of many tiles, outputs one
piece past a tile and smaller than one, strided operands; and F.linear's VJP on both sides of the rule.  Bound:
one rounding to the dtype and the fp32 sums.
"""

from __future__ import annotations

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():  # pragma: no cover - CPU containers
    pytest.skip("no GPU", allow_module_level=True)

import tensorsmith_hip as ts  # noqa: E402
from tensorsmith_hip import _lib  # noqa: E402
from tensorsmith_hip.nn import functional as F  # noqa: E402

ULP = {torch.float16: 2.0**-11, torch.bfloat16: 2.0**-8}
CODE = {torch.float16: _lib.F16, torch.bfloat16: _lib.BF16}


def _close(got, want, dtype, tokens):
    # fp32 partial sums of `tokens` products: 2^-24 sqrt(tokens) of the sum's scale
    scale = want.abs() + want.square().mean().sqrt()
    err = ((got.double() - want).abs() / scale).max().item()
    assert err <= ULP[dtype] + 2.0**-22 * tokens**0.5, err


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("tokens,m,n", [(1, 8, 8), (33, 136, 120), (161, 128, 264), (1000, 256, 128),
                                        (4097, 512, 72), (9000, 64, 136), (1300, 776, 904), (600, 1160, 1032)])
def test_wgrad_matches_float64(tokens, m, n, dt):
    print("wgrad", tokens, m, n, dt, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(tokens)
    g = torch.randn(tokens, m + 16, generator=gen, device="cuda").to(dt)[:, 8:8 + m]
    x = torch.randn(tokens, n + 8, generator=gen, device="cuda").to(dt)[:, :n]
    lib = _lib.load()
    nbytes = lib.tsattn_linear_wgrad_workspace(tokens, m, n)
    ws = torch.full((nbytes,), 255, dtype=torch.uint8, device="cuda")  # NaN bytes: every partial is written
    out, wide = (torch.empty(m, n, dtype=t, device="cuda") for t in (dt, torch.float32))
    for to, code in ((out, CODE[dt]), (wide, _lib.F32)):
        _lib.check(lib.tsattn_linear_wgrad(CODE[dt], code, tokens, m, n, g.data_ptr(), g.stride(0), x.data_ptr(),
                                           x.stride(0), to.data_ptr(), ws.data_ptr(), nbytes,
                                           torch.cuda.current_stream().cuda_stream), "wgrad")
    _close(out, g.double().t() @ x.double(), dt, tokens)
    assert torch.equal(wide, out.float())  # the rounded sums, widened


@pytest.mark.parametrize("rows,out_features", [((4, 1024), 264), ((3, 1365), 264), ((4096,), 100)])
def test_linear_vjp_on_both_sides_of_the_rule(rows, out_features):
    gen = torch.Generator(device="cuda").manual_seed(out_features)
    x = torch.randn(*rows, 136, generator=gen, device="cuda").half()
    w = torch.randn(out_features, 136, generator=gen, device="cuda").half()
    g = torch.randn(*rows, out_features, generator=gen, device="cuda").half()
    tx, tw = (ts.Tensor(t, device="hip", requires_grad=True) for t in (x, w))
    _lib.profile_reset()
    _lib.profile_enable(True)
    F.linear(tx, tw).backward(ts.Tensor(g, device="hip"))
    torch.cuda.synchronize()
    _lib.profile_enable(False)
    tokens = x.numel() // 136
    assert ("wgrad" in _lib.profile_read()) == (tokens >= 4096 and out_features % 8 == 0)
    g64, x64 = g.double().reshape(tokens, -1), x.double().reshape(tokens, -1)
    _close(tw.grad._data, g64.t() @ x64, torch.float16, tokens)
    _close(tx.grad._data.reshape(tokens, -1), g64 @ w.double(), torch.float16, out_features)
