"""dK / dV of problems with few key blocks: each block's query tiles over several
workgroups, against the unsplit kernel and float64.

Cases at the edges of the split: two parts of the smallest size, parts that begin
inside a query head, causal key blocks with fewer tiles than parts, rows that see
no key, key blocks past a key length (parts without a tile), ragged ends, unequal
head dims, masks whose rows start 4- but not 16-byte aligned (read as 16-byte
pieces, the last of which passes the mask's end), folded rotation.  The partial
sums are fp32 and rounded once, so the split results are as far from float64 as
the unsplit ones.
"""

from __future__ import annotations

import ctypes
import math

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():  # pragma: no cover - CPU containers
    pytest.skip("no GPU", allow_module_level=True)

import abi  # noqa: E402
import tensorsmith_hip as ts  # noqa: E402
from tensorsmith_hip import _lib, nn  # noqa: E402

# 16-bit P, dS and results: a rounding each, 2-norm
REL = {torch.float16: 2e-3, torch.bfloat16: 1.5e-2}
F16, BF16 = torch.float16, torch.bfloat16

CASES = [
    # (B, Hq, Hkv, Sq, Sk, Dqk, Dv, dtype, causal, mask)
    (1, 4, 1, 256, 256, 128, 128, BF16, True, None),
    (1, 8, 1, 1000, 1000, 64, 64, F16, True, None),
    (2, 2, 2, 1030, 515, 32, 32, BF16, False, None),
    (1, 4, 2, 700, 650, 128, 64, F16, True, None),
    (2, 4, 1, 520, 600, 64, 128, BF16, False, "lengths"),
    (1, 4, 1, 335, 335, 128, 128, BF16, True, "add-f32"),
    (1, 4, 1, 335, 301, 64, 64, F16, False, "add-f32"),
    (1, 4, 1, 300, 300, 64, 64, F16, False, "bool"),
    (1, 4, 1, 300, 308, 128, 128, BF16, True, "bool"),
    (1, 2, 1, 600, 334, 128, 128, BF16, False, "add-f16"),
]


def _reference(q, k, v, g, seen, bias):
    rep = q.shape[1] // k.shape[1]
    qd, kd, vd, gd = (t.double() for t in (q, k.repeat_interleave(rep, 1), v.repeat_interleave(rep, 1), g))
    scale = 1 / math.sqrt(q.shape[-1])
    t = lambda m: m.transpose(-1, -2).contiguous()
    x = qd @ t(kd) * scale
    if bias is not None:
        x = x + bias.double()
    x = x.masked_fill(~seen, -math.inf)
    top = x.amax(-1, keepdim=True)
    e = torch.exp(x - torch.where(torch.isfinite(top), top, 0.0))
    p = e / e.sum(-1, keepdim=True).clamp_min(1e-300)
    dp = gd @ t(vd)
    ds = p * (dp - (p * dp).sum(-1, keepdim=True))
    group = lambda m: m.unflatten(1, (k.shape[1], rep)).sum(2)
    return ds @ kd * scale, group(t(ds) @ qd * scale), group(t(p) @ gd)


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(x).split(".")[-1] for x in c))
def test_backward_parts(case):
    b, hq, hkv, sq, sk, dqk, dv, dt, causal, mkind = case
    print("backward parts", case, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(sq + sk)
    draw = lambda *s: (torch.randn(s, generator=gen, device="cuda") * 0.7).to(dt)
    q, k, v, g = draw(b, hq, sq, dqk), draw(b, hkv, sk, dqk), draw(b, hkv, sk, dv), draw(b, hq, sq, dv)
    off = sk - sq if causal else 0
    kw, bias = dict(causal=causal, offset=off), None
    seen = torch.ones(b, 1, sq, sk, dtype=torch.bool, device="cuda")
    if mkind == "lengths":
        keys = torch.arange(sk, device="cuda")[None] < torch.tensor([[sk], [130]], device="cuda")
        kv_len, kv_prefix = abi.key_lengths(keys)
        seen = seen & keys[:, None, None, :]
        kw.update(mask=keys[:, None, None, :], kv_len=kv_len, kv_prefix=kv_prefix)
    elif mkind == "bool":
        mask = torch.rand(b, 1, sq, sk, generator=gen, device="cuda") < 0.6
        mask[:, :, 5] = False
        seen = seen & mask
        kw.update(mask=mask)
    elif mkind:
        bias = torch.randn(1, hq, sq, sk, generator=gen, device="cuda")
        bias = bias if mkind == "add-f32" else bias.half()
        bias[:, :, 7, :40] = -math.inf
        kw.update(mask=bias)
    if causal:
        seen = seen & (torch.arange(sk, device="cuda")[None] <= torch.arange(sq, device="cuda")[:, None] + off)
    out, lse, path = abi.forward(q, k, v, **kw)
    assert path == _lib.PATH_MFMA
    p = abi.problem(q, k, v, **kw)
    need = _lib.load().tsattn_sdpa_backward_workspace(ctypes.byref(p))
    want = _reference(q, k, v, g, seen, bias)
    split = abi.backward(q, k, v, out, g, lse, **kw)[:3]
    # a byte less than the parts need: the unsplit kernel
    plain = abi.backward(q, k, v, out, g, lse, ws_bytes=need - 1, **kw)[:3]
    assert torch.equal(split[0], plain[0])  # dQ: the same dS, bit for bit
    differ = False
    for name, got, ref, exact in zip(("dq", "dk", "dv"), split, plain, want):
        rel = lambda a: ((a.double() - exact).norm() / exact.norm()).item()
        assert rel(got) <= REL[dt] and rel(got) <= 1.05 * rel(ref) + 1e-5, (name, rel(got), rel(ref))
        differ |= not torch.equal(got, ref)
    assert differ  # the sums' order changed: both forms ran
    if mkind == "lengths":
        assert (split[1][1, :, 130:] == 0).all() and (split[2][1, :, 130:] == 0).all()


def test_backward_parts_rotate_the_key_gradients_back():
    """With the rotation folded in: the gradients of rotating first, to a rounding."""
    got = []
    for fold in (True, False):
        gen = torch.Generator(device="cuda").manual_seed(4)
        draw = lambda *s: ts.Tensor((torch.randn(s, generator=gen, device="cuda")).half(), device="hip",
                                    requires_grad=True)
        q, k, v = draw(1, 4, 300, 64), draw(1, 1, 300, 64), draw(1, 1, 300, 64)
        up = torch.randn(1, 4, 300, 64, generator=gen, device="cuda").half()
        a, c = (q, k) if fold else (nn.rotary_embedding(q, 0), nn.rotary_embedding(k, 0))
        out = nn.scaled_dot_product_attention(a, c, v, is_causal=True, enable_gqa=True,
                                              _rope=(0, 0, 10000.0) if fold else None)
        out.backward(ts.Tensor(up, device="hip"))
        got.append([t.grad._data.double() for t in (q, k, v)])
    for a, c in zip(*got):
        assert ((a - c).norm() / c.norm()).item() <= 2e-3
