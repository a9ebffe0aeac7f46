"""The key-split 16-bit forward against the unsplit one and against float64.

Cases at the edges of the split: the smallest number of tiles a part gets,
causal blocks whose early rows leave later parts empty, a ragged last key and
row, key-padding lengths (a row that sees nothing) and a key mask with holes,
grouped heads, strided caches, unequal head dims, folded rotation.  The parts
are combined in fp32, so both forwards are within the rounding of the 16-bit
probabilities (the unsplit kernel's own) of each other, and equally far from
float64.
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
from tensorsmith_hip import _lib  # noqa: E402

REL = {torch.float16: 1e-3, torch.bfloat16: 8e-3}  # 2 roundings of 16-bit values, 2-norm

CASES = [
    # (B, Hq, Hkv, Sq, Sk, Dqk, Dv, dtype, causal, mask)
    (1, 2, 1, 130, 1024, 128, 128, torch.bfloat16, True, None),
    (1, 1, 1, 1, 1025, 64, 64, torch.float16, True, None),
    (2, 2, 2, 33, 2047, 32, 32, torch.bfloat16, False, None),
    (1, 3, 3, 1500, 1500, 64, 64, torch.float16, True, None),
    (3, 2, 2, 100, 1100, 128, 128, torch.float16, False, "lengths"),
    (2, 2, 1, 200, 1300, 64, 64, torch.bfloat16, True, "holes"),
    (1, 2, 2, 260, 1111, 128, 64, torch.bfloat16, True, None),
    (1, 2, 2, 260, 1111, 64, 128, torch.float16, False, None),
]


def _split_forward(q, k, v, rope=None, **kw):
    lib = _lib.load()
    p = abi.problem(q, k, v, **kw)
    out = torch.full(q.shape[:3] + (v.shape[3],), 7.0, dtype=q.dtype, device=q.device)
    lse = torch.full(q.shape[:3], 7.0, dtype=torch.float32, device=q.device)
    nbytes = lib.tsattn_sdpa_forward_workspace(ctypes.byref(p))
    assert nbytes > 0
    ws = torch.full((nbytes,), 255, dtype=torch.uint8, device=q.device)  # NaN: every partial is written
    _lib.check(lib.tsattn_sdpa_forward_split(
        ctypes.byref(p), rope, abi.view(q), abi.view(k), abi.view(v), abi.view(out),
        ctypes.c_void_p(lse.data_ptr()), ctypes.c_void_p(ws.data_ptr()), nbytes, abi.stream()), "split forward")
    return out, lse


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(x).split(".")[-1] for x in c))
def test_split_forward(case):
    b, hq, hkv, sq, sk, dqk, dv, dt, causal, mkind = case
    print("split forward", case, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(sk)
    draw = lambda *s: (torch.randn(s, generator=gen, device="cuda") * 0.7).to(dt)
    q, k, v = draw(b, hq, sq, dqk), draw(b, hkv, sk + 9, dqk)[:, :, :sk], draw(b, hkv, sk + 9, dv)[:, :, :sk]
    off = sk - sq if causal else 0
    kw, seen = dict(causal=causal, offset=off), torch.ones(b, 1, 1, sk, dtype=torch.bool, device="cuda")
    if mkind:
        lens = torch.tensor([sk, 0, 517][:b] if mkind == "lengths" else [sk, 700][:b], device="cuda")
        keys = torch.arange(sk, device="cuda")[None] < lens[:, None]
        if mkind == "holes":
            keys[:, 40:300:3] = False
        kv_len, kv_prefix = abi.key_lengths(keys)
        seen = keys[:, None, None, :]
        kw.update(mask=seen, kv_len=kv_len, kv_prefix=kv_prefix)
    out, lse = _split_forward(q, k, v, **kw)
    plain, lse_p, path = abi.forward(q, k, v, **kw)
    assert path == _lib.PATH_MFMA
    rep = hq // hkv
    x = q.double() @ k.double().repeat_interleave(rep, 1).transpose(-1, -2).contiguous() / math.sqrt(dqk)
    if causal:
        ok = torch.arange(sk, device="cuda")[None] <= torch.arange(sq, device="cuda")[:, None] + off
        seen = seen & ok
    x = x.masked_fill(~seen, -math.inf)
    want_lse = torch.logsumexp(x, -1)
    p = torch.exp(x - want_lse.clamp_min(-1e300)[..., None])
    want = p @ v.double().repeat_interleave(rep, 1)
    rel = lambda a: ((a.double() - want).norm() / want.norm()).item()
    assert rel(out) <= REL[dt] and rel(out) <= 1.2 * rel(plain) + 1e-5, (rel(out), rel(plain))
    live = torch.isfinite(want_lse)
    assert torch.equal(torch.isneginf(lse), ~live) and torch.equal(torch.isneginf(lse_p), ~live)
    assert (lse[live].double() - want_lse[live]).abs().max() <= 2e-5
    assert (out[~live] == 0).all()


def test_split_forward_folds_the_rotation():
    """With a descriptor: the unsplit folded forward's rotated queries, bit for bit."""
    from tensorsmith_hip.nn.attention import rope_tables

    q, k, v = (torch.randn(1, 2, s, 64, device="cuda").half() for s in (130, 1200, 1200))
    cos, sin = rope_tables(10000.0, 64, torch.float16, q.device, 1200)
    outs = []
    for split in (True, False):
        rot = torch.empty(1, 2, 130, 64, dtype=torch.float16, device="cuda")
        d = _lib.RopeDesc()
        d.cos, d.sin, d.rotary_dim, d.q_pos0, d.k_pos0 = cos.data_ptr(), sin.data_ptr(), 64, 1070, 0
        d.q_rotated = rot.data_ptr()
        if split:
            out, lse = _split_forward(q, k, v, rope=ctypes.byref(d), causal=True, offset=1070)
        else:
            p = abi.problem(q, k, v, causal=True, offset=1070)
            out, lse = torch.empty_like(q), torch.empty(1, 2, 130, device="cuda")
            _lib.check(_lib.load().tsattn_sdpa_forward_rope(
                ctypes.byref(p), ctypes.byref(d), abi.view(q), abi.view(k), abi.view(v), abi.view(out),
                ctypes.c_void_p(lse.data_ptr()), abi.stream()), "rope forward")
        torch.cuda.synchronize()
        outs.append((out, lse, rot))
    assert torch.equal(outs[0][2], outs[1][2])
    assert ((outs[0][0].double() - outs[1][0].double()).norm() / outs[1][0].double().norm()).item() <= 1e-3
    assert (outs[0][1] - outs[1][1]).abs().max().item() <= 2e-5
