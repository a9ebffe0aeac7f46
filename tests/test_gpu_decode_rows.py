"""The matrix-core decode split kernel (2 .. 8 query rows per KV head) against
attention in float64.

Sizes at the edges of its work split: a cache that ends one key before, at and
after a 32-key tile and a wave's second tile, splits shorter than one tile per
wave, every row count the routing sends here, caches whose rows are not
contiguous ([B,S,H,D] memory), general and key-padding masks, an empty row.
The bound is the rounding of the result to its dtype: the probabilities enter
the value product with all their bits and the sums are fp32, so 4e-6 of the row's
largest value (sums over up to 700 keys) on top of half an ulp.
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

ULP = {torch.float16: 2.0**-11, torch.bfloat16: 2.0**-8}

CASES = [
    # (B, Hkv, rep, Sq, keys, D, dtype, split, layout, mask)
    (2, 2, 2, 1, 31, 64, torch.float16, 0, "bhsd", None),
    (1, 3, 4, 1, 33, 128, torch.bfloat16, 0, "bhsd", None),
    (3, 2, 8, 1, 641, 128, torch.float16, 0, "bhsd", None),
    (2, 2, 1, 5, 200, 128, torch.bfloat16, 40, "bhsd", None),
    (2, 1, 3, 2, 257, 64, torch.bfloat16, 96, "bshd", None),
    (1, 2, 7, 1, 320, 256, torch.float16, 0, "bhsd", None),
    (2, 2, 2, 3, 130, 256, torch.bfloat16, 33, "bshd", None),
    (3, 2, 4, 1, 300, 128, torch.float16, 0, "bhsd", "lengths"),
    (2, 2, 4, 1, 300, 64, torch.bfloat16, 64, "bhsd", "bool"),
    (2, 2, 2, 2, 190, 128, torch.float16, 0, "bhsd", "additive"),
]


def _reference(q, k, v, causal_off, mask):
    rep = q.shape[1] // k.shape[1]
    k, v = (t.double().repeat_interleave(rep, dim=1) for t in (k, v))
    x = q.double() @ k.transpose(-1, -2).contiguous() / math.sqrt(q.shape[-1])
    n, sq = k.shape[2], q.shape[2]
    seen = torch.arange(n, device=q.device)[None, :] <= torch.arange(sq, device=q.device)[:, None] + causal_off
    x = x.masked_fill(~seen, -math.inf)
    if mask is not None:
        x = x.masked_fill(~mask, -math.inf) if mask.dtype == torch.bool else x + mask.double()
    p = torch.exp(x - x.amax(-1, keepdim=True).clamp_min(-1e300))
    return (p @ v) / p.sum(-1, keepdim=True).clamp_min(1e-300)


def _check(got, want, dtype):
    scale = want.abs().amax(-1, keepdim=True).clamp_min(1e-30)
    err = (got.double() - want).abs() - ULP[dtype] * want.abs()
    assert (err / scale).max().item() <= 4e-6, (err / scale).max().item()


def _probed(run):
    _lib.profile_reset()
    _lib.profile_enable(True)
    out = run()
    torch.cuda.synchronize()
    _lib.profile_enable(False)
    return out, _lib.profile_read()


def _caches(gen, b, h, n, d, layout):
    out = []
    for _ in range(2):
        t = torch.randn((b, n + 7, h, d) if layout == "bshd" else (b, h, n + 7, d), generator=gen, device="cuda")
        out.append(t.transpose(1, 2) if layout == "bshd" else t)
    return out


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(x).split(".")[-1] for x in c))
def test_decode_rows_match_float64(case):
    b, hkv, rep, sq, n, d, dt, split, layout, mkind = case
    print("decode rows", case, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(n + d)
    q = torch.randn(b, hkv * rep, sq, d, generator=gen, device="cuda").to(dt)
    k, v = (t.to(dt)[:, :, :n] for t in _caches(gen, b, hkv, n, d, layout))
    kw, mask = dict(causal=True, offset=n - sq), None
    if mkind == "lengths":
        lens = torch.tensor([n, 0, n - 37][:b], dtype=torch.int32, device="cuda")
        kw["kv_len"] = lens
        mask = (torch.arange(n, device="cuda")[None] < lens[:, None])[:, None, None]
    elif mkind == "bool":
        mask = torch.rand(b, hkv * rep, 1, n, generator=gen, device="cuda") > 0.4
        mask[0, 1] = False  # a row that sees nothing
        kw["mask"] = mask
    elif mkind == "additive":
        mask = torch.randn(b, 1, sq, n, generator=gen, device="cuda")
        mask[..., 32:96] = -math.inf
        kw["mask"] = mask
    got, probes = _probed(lambda: abi.decode(q, k, v, split_len=split, **kw))
    assert "decode_mfma" in probes and "decode_split" not in probes
    _check(got, _reference(q, k, v, n - sq, mask), dt)


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n,rep,d,split", [(33, 2, 64, 0), (129, 4, 128, 0), (645, 8, 128, 0), (700, 3, 64, 96),
                                           (130, 4, 256, 0)])
def test_int8_decode_rows_match_float64(n, rep, d, split, dt):
    """The codes are exact in the 16-bit tiles and the row scales enter in fp32;
    one key's scale is far from the others'."""
    print("int8 decode rows", n, rep, d, dt, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(n)
    b, hkv = 2, 2
    q = torch.randn(b, hkv * rep, 1, d, generator=gen, device="cuda").to(dt)
    k8, v8 = (torch.randint(-127, 128, (b, hkv, n + 5, d), generator=gen, device="cuda", dtype=torch.int8)
              for _ in range(2))
    ks, vs = (torch.rand(b, hkv, n + 5, 1, generator=gen, device="cuda") * 0.02 + 1e-4 for _ in range(2))
    vs[:, :, 7] = 30.0
    (out, path), probes = _probed(
        lambda: abi.decode_int8(q, k8, v8, ks, vs, n, split_len=split, causal=True, offset=n - 1))
    assert path == _lib.PATH_DECODE
    # 256 channels of codes are the vector kernel's
    assert ("decode_mfma_int8" in probes) == (d < 256) and ("decode_split_int8" in probes) == (d == 256)
    k, v = ((c.double() * s.double())[:, :, :n] for c, s in ((k8, ks), (v8, vs)))
    _check(out, _reference(q, k, v, n - 1, None), dt)


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("d", [64, 128])
def test_probabilities_enter_with_all_their_bits(d, dt):
    """Over values that are one-hot a split's partial rows are its probabilities:
    half of them are odd in their last of 24 bits."""
    b, hkv, rep, n = 4, 2, 4, d
    gen = torch.Generator(device="cuda").manual_seed(d)
    q, k = (torch.randn(b, h, s, d, generator=gen, device="cuda").to(dt) for h, s in ((hkv * rep, 1), (hkv, n)))
    v = torch.eye(n, dtype=dt, device="cuda").expand(b, hkv, n, d).contiguous()
    p = abi.problem(q, k, v)
    lib, out = _lib.load(), torch.empty_like(q)
    nbytes = lib.tsattn_decode_workspace(ctypes.byref(p), n)
    ws = torch.zeros(nbytes // 4, device="cuda")
    _lib.check(lib.tsattn_decode_forward(ctypes.byref(p), abi.view(q), abi.view(k), abi.view(v), abi.view(out), n,
                                         ws.data_ptr(), nbytes, abi.stream()), "decode")
    part = ws[:b * hkv * rep * (d + 2)].view(b, hkv, rep, d + 2)  # one split: acc, max, sum
    bits = part[..., :d].contiguous().view(torch.int32)
    seen = part[..., :d] > part[..., :d].amax(-1, keepdim=True) * 2.0**-15
    assert seen.float().mean() > 0.9
    odd = (bits[seen] & 1).float().mean().item()  # of 2048 and more: 0.5 +- 0.011
    assert 0.45 < odd < 0.55, odd
    total = part[..., :d].double().sum(-1)  # and their sum is the denominator, within its fp32 sums
    assert ((part[..., d + 1].double() - total).abs() / total).max().item() <= 1e-6


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("d,n,int8", [(64, 200, False), (128, 700, False), (256, 90, False), (64, 200, True),
                                      (128, 700, True)])
def test_infinite_values_stay_infinite(d, n, int8, dt):
    """p inf is inf, whatever the parts p is split in; the other channels, splits
    and heads are as they were."""
    print("decode, infinite values", d, n, int8, dt, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(n)
    b, hkv, rep, inf = 2, 2, 4, math.inf
    q = torch.randn(b, hkv * rep, 1, d, generator=gen, device="cuda").to(dt) * 0.5
    if int8:
        k, v = (torch.randint(-127, 128, (b, hkv, n, d), generator=gen, device="cuda", dtype=torch.int8)
                for _ in range(2))
        ks, vs = (torch.full((b, hkv, n, 1), 0.02, device="cuda") for _ in range(2))
        v[:, 0, 7, 3], vs[:, 0, 7] = 0, inf  # (that channel: inf * 0)
        out, _ = abi.decode_int8(q, k, v, ks, vs, n, causal=True, offset=n - 1)
        k, v = k.double() * ks.double(), v.double() * vs.double()
    else:
        k, v = (torch.randn(b, hkv, n, d, generator=gen, device="cuda").to(dt) for _ in range(2))
        v[:, 0, 7, 3], v[:, 0, 75, 4], v[:, 0, 60, 5] = inf, -inf, math.nan
        v[:, 0, 20, 6], v[:, 0, 21, 6] = inf, -inf
        out = abi.decode(q, k, v, causal=True, offset=n - 1)
    want = _reference(q, k, v, n - 1, None)
    assert torch.isinf(want).any() and torch.isnan(want).any() and torch.isfinite(want[:, rep:]).all()
    fine = torch.isfinite(want)
    assert torch.equal(torch.nan_to_num(out[~fine].double(), posinf=1, neginf=-1),
                       torch.nan_to_num(want[~fine], posinf=1, neginf=-1))
    for x, y in ((out.masked_fill(~fine, 0), want.masked_fill(~fine, 0)), (out[:, rep:], want[:, rep:])):
        _check(x, y, dt)


@pytest.mark.parametrize("b,hkv,d,n,int8,kernel", [
    (2, 2, 64, 200, False, "decode_mfma"), (2, 2, 128, 200, False, "decode_mfma"),
    (2, 2, 128, 200, True, "decode_mfma_int8"), (1, 2, 256, 150, False, "decode_split"),
    (16, 8, 128, 200, False, "decode_split"), (16, 8, 128, 4000, False, "decode_mfma"),
    (16, 8, 64, 8300, False, "decode_split"), (16, 8, 128, 4200, True, "decode_split_int8")])
def test_two_rows_take_the_faster_kernel(b, hkv, d, n, int8, kernel):
    """Two rows a KV head on both sides of the rule, and one row on the vector kernel."""
    print("decode, two rows", b, hkv, d, n, int8, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(n)
    q = torch.randn(b, 2 * hkv, 1, d, generator=gen, device="cuda").half()
    if int8:
        k, v = (torch.randint(-127, 128, (b, hkv, n, d), generator=gen, device="cuda", dtype=torch.int8) for _ in range(2))
        ks, vs = (torch.rand(b, hkv, n, 1, generator=gen, device="cuda") * 0.02 + 1e-4 for _ in range(2))
        run = lambda q: abi.decode_int8(q, k, v, ks, vs, n, causal=True, offset=n - 1)[0]
    else:
        k, v = (torch.randn(b, hkv, n, d, generator=gen, device="cuda").half() for _ in range(2))
        run = lambda q: abi.decode(q, k, v, causal=True, offset=n - 1)
    got, probes = _probed(lambda: run(q))
    assert kernel in probes, sorted(probes)
    one, probes = _probed(lambda: run(q[:, :hkv]))
    assert "decode_split_int8" in probes if int8 else "decode_split" in probes
    last = slice(b - 1, b)  # (one sequence against float64)
    kd, vd = (k[last].double() * ks[last].double(), v[last].double() * vs[last].double()) if int8 else (k[last], v[last])
    _check(got[last], _reference(q[last], kd, vd, n - 1, None), q.dtype)
    _check(one[last], _reference(q[last, :hkv], kd, vd, n - 1, None), q.dtype)
