"""16-bit forward with masks whose rows start 4- but not 16-byte aligned: read as
16-byte pieces, the last of which passes the end of the mask.  Against float64,
the last row on its own; bound: the 16-bit rounding of the probabilities and the
result (2-norm)."""

from __future__ import annotations

import math

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():  # pragma: no cover - CPU containers
    pytest.skip("no GPU", allow_module_level=True)

import abi  # noqa: E402
from tensorsmith_hip import _lib  # noqa: E402

CASES = [(1, 2, 1, 335, 335, 128, "float32"), (2, 3, 3, 130, 301, 64, "float32"), (1, 2, 2, 97, 31, 32, "float32"),
         (1, 2, 2, 200, 334, 128, "float16"), (1, 2, 2, 200, 34, 64, "bfloat16"), (2, 2, 1, 300, 300, 64, "bool"),
         (1, 2, 2, 100, 36, 128, "bool")]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c)))
def test_forward_with_unaligned_mask_rows(case):
    b, hq, hkv, sq, sk, d, kind = case
    print("mask rows", case, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(sk)
    draw = lambda *s: torch.randn(s, generator=gen, device="cuda").bfloat16()
    q, k, v = draw(b, hq, sq, d), draw(b, hkv, sk, d), draw(b, hkv, sk, d)
    if kind == "bool":
        mask = torch.rand(b, 1, sq, sk, generator=gen, device="cuda") < 0.6
    else:
        mask = torch.randn(1, hq, sq, sk, generator=gen, device="cuda").to(getattr(torch, kind))
    out, lse, path = abi.forward(q, k, v, mask=mask)
    assert path == _lib.PATH_MFMA
    rep = hq // hkv
    x = q.double() @ k.double().repeat_interleave(rep, 1).transpose(-1, -2).contiguous() / math.sqrt(d)
    x = x.masked_fill(~mask, -math.inf) if kind == "bool" else x + mask.double()
    want = torch.softmax(x, -1).nan_to_num(0) @ v.double().repeat_interleave(rep, 1)
    for part in (slice(None), slice(-1, None)):
        got, ref = out.double()[:, :, part], want[:, :, part]
        assert ((got - ref).norm() / ref.norm()).item() <= 8e-3
    seen = torch.logsumexp(x, -1)
    assert (lse.double() - seen)[torch.isfinite(seen)].abs().max().item() <= 2e-5
