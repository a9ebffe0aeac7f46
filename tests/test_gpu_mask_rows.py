"""16-bit attention with masks whose rows start 4- but not 16-byte aligned: read as
16-byte pieces, the last of which passes the end of the mask (in the middle of
four bytes, where the rows are padded ones).  Against float64, the forward's last
row on its own; bound: the 16-bit rounding of the probabilities, dS and the
results (2-norm)."""

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


# (..., mask dtype, keys a stored mask row is longer)
GRADS = [(1, 4, 1, 335, 335, 128, "float32", 0), (1, 4, 1, 300, 300, 64, "bool", 0), (1, 4, 2, 300, 308, 128, "bool", 0),
         (1, 2, 1, 600, 334, 128, "float16", 0), (2, 2, 2, 130, 301, 64, "bool", 7), (1, 2, 2, 97, 333, 64, "float16", 1),
         (1, 2, 2, 65, 31, 32, "bool", 1)]


@pytest.mark.parametrize("case", GRADS, ids=lambda c: "-".join(map(str, c)))
def test_gradients_with_unaligned_mask_rows(case):
    b, hq, hkv, sq, sk, d, kind, pad = case
    print("mask rows, gradients", case, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(sk)
    draw = lambda *s: (torch.randn(s, generator=gen, device="cuda") * 0.7).half()
    q, k, v, g = draw(b, hq, sq, d), draw(b, hkv, sk, d), draw(b, hkv, sk, d), draw(b, hq, sq, d)
    if kind == "bool":
        mask = torch.rand(b, 1, sq, sk + pad, generator=gen, device="cuda") < 0.6
    else:
        mask = torch.randn(1, hq, sq, sk + pad, generator=gen, device="cuda").to(getattr(torch, kind))
    mask = mask[..., :sk]
    # the last row's outcome is its last key's alone, the last element of the mask
    mask[:, :, -1, :-1] = False if kind == "bool" else 0
    mask[:, :, -1, -1] = True if kind == "bool" else 20
    out, lse, path = abi.forward(q, k, v, mask=mask)
    assert path == _lib.PATH_MFMA
    got = abi.backward(q, k, v, out, g, lse, mask=mask)[:3]
    t = lambda m: m.transpose(-1, -2).contiguous()
    rep, scale = hq // hkv, 1 / math.sqrt(d)
    qd, kd, vd, gd = (a.double() for a in (q, k.repeat_interleave(rep, 1), v.repeat_interleave(rep, 1), g))
    x = qd @ t(kd) * scale
    x = x.masked_fill(~mask, -math.inf) if kind == "bool" else x + mask.double()
    p = torch.softmax(x, -1).nan_to_num(0)
    dp = gd @ t(vd)
    ds = p * (dp - (p * dp).sum(-1, keepdim=True))
    group = lambda m: m.unflatten(1, (hkv, rep)).sum(2)
    want = ds @ kd * scale, group(t(ds) @ qd * scale), group(t(p) @ gd)
    for name, a, ref in zip(("last row", "dq", "dk", "dv"), (out[:, :, -1], *got), ((p @ vd)[:, :, -1], *want)):
        assert ((a.double() - ref).norm() / ref.norm()).item() <= 2e-3, name
