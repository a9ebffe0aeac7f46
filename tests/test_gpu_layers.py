"""The norm and SwiGLU kernels against the same chains in float64.

Sizes at the edges of the kernels' split: one 8-element piece, a row that ends
inside a wave's first step, the last size of the wave form (2048) and the first
past it, the largest row; one row, and more rows than one pass of the grid.
The bound is the rounding of the results to their dtype (relative 2^-24 / 2^-11
/ 2^-8, plus the fp32 sums' 1e-6), with the VJP's products of two such values.
"""

from __future__ import annotations

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():  # pragma: no cover - CPU containers
    pytest.skip("no GPU", allow_module_level=True)

import tensorsmith_hip as ts  # noqa: E402
from tensorsmith_hip.nn import functional as F  # noqa: E402

EPS = {torch.float32: 2.0**-23, torch.float16: 2.0**-10, torch.bfloat16: 2.0**-7}


def _close(got, want, dtype, what, sums=1):
    got, want = got.double().cpu(), want.double().cpu()
    scale = want.abs() + want.square().mean().sqrt()
    err = ((got - want).abs() / scale.clamp_min(1e-30)).max().item()
    bound = EPS[dtype] + 4e-6 * sums
    assert err <= bound, (what, err, bound)


NORM_CASES = [
    # (rows shape, dim, x dtype, w dtype, rms)
    ((3,), 8, torch.float32, torch.float32, True),
    ((1, 1), 136, torch.float16, torch.float16, True),
    ((5, 7), 512, torch.float32, torch.float32, True),
    ((2, 2100), 512, torch.float32, torch.float32, False),
    ((9001,), 64, torch.bfloat16, torch.float32, True),
    ((33,), 2048, torch.float16, torch.float32, False),
    ((33,), 2056, torch.bfloat16, torch.bfloat16, True),
    ((1030,), 4096, torch.float16, torch.float16, False),
    ((6,), 8192, torch.float32, torch.float32, True),
]


@pytest.mark.parametrize("case", NORM_CASES, ids=lambda c: f"{'x'.join(map(str, c[0]))}x{c[1]}-{c[4]}")
def test_norm_matches_float64(case):
    lead, dim, xd, wd, rms = case
    print("norm", case, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(dim)
    draw = lambda shape, dt: torch.randn(shape, generator=gen, device="cuda").to(dt)
    x, g = draw((*lead, dim), xd) + 0.25, draw((*lead, dim), xd)
    w, b = draw((dim,), wd) + 1, draw((dim,), wd)
    tx, tw, tb = (ts.Tensor(t, device="hip", requires_grad=True) for t in (x, w, b))
    out = F.rms_norm(tx, tw) if rms else F.layer_norm(tx, tw, tb)
    assert out._op == ("rms_norm" if rms else "layer_norm")
    out.backward(ts.Tensor(g, device="hip"))
    x64, w64, b64 = (t.double().requires_grad_() for t in (x, w, b))
    if rms:
        ref = x64 / (x64.square().mean(-1, keepdim=True) + 1e-6).sqrt() * w64
    else:
        ref = torch.nn.functional.layer_norm(x64, (dim,), w64, b64, 1e-5)
    ref.backward(g.double())
    _close(out._data, ref, xd, "out")
    _close(tx.grad._data, x64.grad, xd, "dx", 2)
    _close(tw.grad._data, w64.grad, wd, "dw", 2)
    if not rms:
        _close(tb.grad._data, b64.grad, wd, "db", 2)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape", [(1, 8), (3, 24), (7, 2048), (4100, 520)])
def test_silu_mul_matches_the_two_ops(shape, dtype):
    """Bit for bit the product's rounding; silu within one rounding of torch's."""
    gen = torch.Generator(device="cuda").manual_seed(shape[1])
    x, u, g = (torch.randn(shape, generator=gen, device="cuda").to(dtype) * 3 for _ in range(3))
    x.view(-1)[:4] = torch.tensor([float("inf"), float("-inf"), 90.0, -90.0], device="cuda").to(dtype)
    leaves = [[ts.Tensor(t, device="hip", requires_grad=True) for t in (x, u)] for _ in range(2)]
    fused = F._silu_mul(*leaves[0])
    plain = F.silu(leaves[1][0]) * leaves[1][1]
    assert fused._op == "silu_mul"
    for out in (fused, plain):
        out.backward(ts.Tensor(g, device="hip"))
    pairs = [(fused._data, plain._data)] + [(a.grad._data, b.grad._data) for a, b in zip(*leaves)]
    for got, want in pairs:
        assert torch.equal(torch.isnan(got), torch.isnan(want))
        fine = torch.isfinite(want)
        assert torch.equal(got[~fine & ~torch.isnan(want)], want[~fine & ~torch.isnan(want)])
        _close(got[fine], want[fine], dtype, "silu_mul", 1)


def test_operands_outside_the_kernels():
    """Odd row lengths, strided and empty inputs keep working."""
    x = torch.randn(4, 6, 100, device="cuda")
    w = torch.ones(101, device="cuda")
    odd = torch.randn(3, 101, device="cuda")
    got = F.rms_norm(ts.Tensor(odd, device="hip"), ts.Tensor(w, device="hip"))._data
    want = odd / (odd.square().mean(-1, keepdim=True) + 1e-6).sqrt()
    np.testing.assert_allclose(got.cpu(), want.cpu(), rtol=1e-5, atol=1e-6)
    sliced = x[:, -1:, 2:98]
    got = F.rms_norm(ts.Tensor(sliced, device="hip"), ts.Tensor(w[:96], device="hip"))._data
    want = sliced / (sliced.square().mean(-1, keepdim=True) + 1e-6).sqrt()
    np.testing.assert_allclose(got.cpu(), want.cpu(), rtol=1e-5, atol=1e-6)
    empty = F.rms_norm(ts.Tensor(torch.empty(0, 96, device="cuda"), device="hip"),
                       ts.Tensor(w[:96], device="hip"))
    assert empty.shape == (0, 96)
