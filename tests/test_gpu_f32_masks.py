"""General masks on the fp32 matrix-core kernels, against the oracle and the
generic kernels.

Boolean and additive masks of any broadcast strides are read one tile ahead of
the products, and a tile the mask forbids whole is skipped.  The cases sit
where that can go wrong: ragged ends in both directions, one row or key more
than a tile, strides that are not the key order, whole tiles and whole rows
masked, grouped heads, and both forms (split and whole) of every mask's kernels,
which their probes name.  Bounds
as for the unmasked fp32 kernels: every product and sum is fp32.
"""

from __future__ import annotations

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():  # pragma: no cover - CPU containers
    pytest.skip("no GPU", allow_module_level=True)

import abi  # noqa: E402
from oracle import attention as A  # noqa: E402
from oracle.inputs import attention_inputs  # noqa: E402
from tensorsmith_hip import _lib  # noqa: E402

TOL = dict(rtol=1e-4, atol=3e-5)
DT = "float32"

CASES = [
    # (B, Hq, Hkv, Sq, Sk, D, causal, offset, mask kind)
    (2, 2, 2, 97, 97, 64, True, 0, "documents"),
    (1, 3, 3, 33, 65, 32, False, 0, "random"),
    (2, 4, 2, 129, 161, 64, True, 32, "random"),       # GQA
    (1, 2, 1, 200, 333, 128, True, 133, "random"),
    (1, 2, 2, 160, 160, 64, False, 0, "transposed"),   # keys not contiguous
    (2, 2, 2, 64, 96, 32, False, 0, "rows"),           # [B,H,Q,1]: zero key stride
    (4, 32, 32, 257, 257, 64, True, 0, "documents"),   # enough blocks for the whole form
    (4, 32, 32, 130, 130, 32, False, 0, "random"),
    (2, 8, 8, 520, 520, 64, True, 0, "add-f32"),
    (2, 8, 4, 513, 530, 32, False, 0, "add-bf16"),
    (2, 8, 8, 600, 600, 128, True, 0, "add-f16"),
    (2, 8, 8, 640, 640, 64, False, 0, "add-lowest"),
    (1, 2, 2, 1, 200, 64, True, 199, "add-f32"),       # fewer rows than a workgroup's
    (2, 3, 3, 33, 97, 32, False, 0, "add-bf16"),
    (1, 2, 1, 96, 96, 64, True, 0, "add-f32"),
    (2, 2, 2, 127, 127, 128, True, 0, "add-f16"),
    # enough row blocks for the whole form (the key blocks of grouped heads: the split one)
    (4, 32, 32, 257, 257, 64, True, 0, "add-f32"),
    (4, 16, 16, 513, 513, 128, True, 0, "add-f32"),
    (4, 32, 8, 300, 290, 32, False, 0, "add-bf16"),
    (8, 16, 16, 300, 300, 64, False, 0, "add-lowest"),
]


def _mask(kind, b, h, sq, sk, rng):
    """(mask as NumPy, mask as the device tensor handed to the kernels)."""
    if kind == "documents":
        ids = np.sort(rng.integers(0, 3, (b, max(sq, sk))), axis=1)
        m = (ids[:, :sq, None] == ids[:, None, :sk])[:, None]
    elif kind == "rows":
        m = rng.random((b, h, sq, 1)) > 0.4
    elif kind.startswith("add"):
        m = (rng.standard_normal((b, 1, sq, sk)) * 1.5).astype(np.float32)
        m[rng.random(m.shape) < 0.2] = -np.inf
        m[..., 7:8, :] = -np.inf  # a row that sees nothing
        m[..., 40:72, 64:] = -np.inf
        if kind == "add-lowest":  # the type's lowest value on a whole row: its softmax is uniform
            m[..., 11, :] = np.finfo(np.float32).min
        dt = {"add-f16": torch.float16, "add-bf16": torch.bfloat16}.get(kind, torch.float32)
        t = torch.from_numpy(m).to(dt).cuda()
        return t.float().cpu().numpy(), t
    else:
        m = rng.random((b, 1, sq, sk)) > 0.4
        m[..., 5, :] = False          # a row that sees nothing
        m[..., : min(sq, 40), 32:64] = False  # whole tiles masked
    t = torch.from_numpy(np.ascontiguousarray(m)).cuda()
    if kind == "transposed":
        t = t.transpose(-1, -2).contiguous().transpose(-1, -2)
    return m, t


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c)))
def test_f32_general_masks(case):
    b, hq, hkv, sq, sk, d, causal, off, kind = case
    print("f32 general mask", case, flush=True)
    rng = np.random.default_rng(sq + sk)
    mask, tm = _mask(kind, b, hq, sq, sk, rng)
    inp = attention_inputs(b, hq, sq, d, DT, heads_kv=hkv, seq_k=sk, seed=29)
    q, k, v, g = (abi.dev_tensor(x, DT) for x in (inp.q, inp.k, inp.v, inp.do))
    kw = dict(causal=causal, offset=off, mask=tm)
    _lib.profile_reset()
    _lib.profile_enable(True)
    out, lse, path = abi.forward(q, k, v, **kw)
    grads = abi.backward(q, k, v, out, g, lse, **kw)
    torch.cuda.synchronize()
    _lib.profile_enable(False)
    probes = _lib.profile_read()
    assert path == _lib.PATH_MFMA and grads[3] == _lib.PATH_MFMA
    for name, blocks in (("fwd_mfma_f32_masked", -(-sq // 128) * hq * b), ("bwd_dq_mfma_f32_masked", -(-sq // 128) * hq * b),
                         ("bwd_dkdv_mfma_f32_masked", -(-sk // 128) * hkv * b)):
        split = d <= 64 and blocks < torch.cuda.get_device_properties(0).multi_processor_count
        assert name + ("_split" if split else "") in probes, (name, split, sorted(probes))
    with abi.generic_only():
        out_g, lse_g, path = abi.forward(q, k, v, **kw)
        grads_g = abi.backward(q, k, v, out_g, g, lse_g, **kw)
    torch.cuda.synchronize()
    assert path == _lib.PATH_GENERIC
    got = [abi.host(x) for x in (out, *grads[:3])]
    want = [abi.host(x) for x in (out_g, *grads_g[:3])]
    names = ("out", "dq", "dk", "dv")
    for x, y, n in zip(got, want, names):
        np.testing.assert_allclose(x, y, **TOL, err_msg=f"{n} against the generic kernels")
    la, lb = abi.host(lse), abi.host(lse_g)
    np.testing.assert_array_equal(np.isneginf(la), np.isneginf(lb))
    live = np.isfinite(lb)
    np.testing.assert_allclose(la[live], lb[live], **TOL)
    if b * hq * sq * sk <= 2_000_000 and kind != "add-lowest":
        ref = A.sdpa(inp.q, inp.k, inp.v, mask, causal, dtype=DT, causal_offset=off,
                     backend="streaming", enable_gqa=hkv != hq)
        for x, y, n in zip(got, (ref.out_cast, *ref.backward(inp.do)), names):
            np.testing.assert_allclose(x, y, **TOL, err_msg=n)


NONFINITE = [
    # (B, Hq, Hkv, S, D, mask): few row blocks (the split form) and enough of them (the whole form)
    (1, 2, 2, 100, 64, "bool"), (1, 2, 1, 131, 32, "add"), (1, 2, 2, 135, 128, "bool"), (1, 2, 2, 135, 128, "add"),
    (16, 16, 16, 97, 64, "bool"), (16, 16, 8, 129, 32, "add"), (16, 16, 16, 129, 64, "add"),
]


@pytest.mark.parametrize("case", NONFINITE, ids=lambda c: "x".join(map(str, c)))
def test_masked_infinities_and_nan_stay_out(case):
    """Infinities and NaN in K and V of masked keys, in Q and dO of rows that see
    nothing, and in V and dO where they are seen: finite and non-finite where the
    generic kernels are, which multiply with P != 0 only."""
    b, hq, hkv, s, d, kind = case
    print("f32 masks, non-finite operands", case, flush=True)
    rng = np.random.default_rng(s + d)
    inp = attention_inputs(b, hq, s, d, DT, heads_kv=hkv, seed=31)
    q, k, v, g = (x.copy() for x in (inp.q, inp.k, inp.v, inp.do))
    inf, nan = np.inf, np.nan
    seen = rng.random((b, 1, s, s)) > 0.3
    seen[..., 40:72, 32:64] = False     # a whole tile masked, and one in part
    seen[:, :, :, [3, 45, 70]] = False  # keys nobody sees, with what a cache's unused rows can hold
    k[:, :, 3], k[:, :, 45, 1], k[:, :, 70, 0] = nan, inf, -inf
    v[:, :, 3], v[:, :, 45, 5], v[:, :, 70, 7] = nan, inf, -inf
    seen[:, :, :, [10, 33]] = False     # keys some rows see, whose infinities and NaN these rows get
    seen[:, :, 7, 10] = seen[:, :, 80, 10] = seen[:, :, 20, 33] = seen[:, :, 80, 33] = True
    v[:, :, 10, [0, 9, 31]] = [inf, -inf, nan]
    v[:, :, 33, [0, 9, 30]] = [inf, inf, -inf]
    seen[:, :, [12, 50]] = False        # rows that see nothing
    q[:, :, 12], q[:, :, 50, 2], g[:, :, 12, 4], g[:, :, 50] = nan, inf, inf, nan
    g[:, :, 66, 6] = inf                # a row that does
    mask = torch.from_numpy(seen).cuda()
    if kind == "add":
        mask = torch.zeros(mask.shape, device="cuda").masked_fill_(~mask, -inf)
        k[:, :, [3, 45, 70]] = inp.k[:, :, [3, 45, 70]]  # (NaN + -inf is NaN: the next test)
        q[:, :, [12, 50]] = inp.q[:, :, [12, 50]]
    t = [abi.dev_tensor(x, DT) for x in (q, k, v, g)]

    def run():
        out, lse, path = abi.forward(*t[:3], mask=mask)
        return path, [abi.host(x) for x in (out, *abi.backward(*t[:3], out, t[3], lse, mask=mask)[:3], lse)]

    path, got = run()
    assert path == _lib.PATH_MFMA
    with abi.generic_only():
        path, want = run()
    assert path == _lib.PATH_GENERIC
    assert np.isinf(want[0]).any() and np.isnan(want[0]).any() and np.isfinite(want[0]).mean() > 0.5
    for x, y, n in zip(got, want, ("out", "dq", "dk", "dv", "lse")):
        fine = np.isfinite(y)
        np.testing.assert_array_equal(np.isfinite(x), fine, err_msg=n)
        np.testing.assert_allclose(x[fine], y[fine], **TOL, err_msg=n)
    for n, i in (("out", 0), ("dv", 3)):  # and the same infinities
        np.testing.assert_array_equal(np.nan_to_num(got[i][~np.isfinite(want[i])], posinf=1, neginf=-1),
                                      np.nan_to_num(want[i][~np.isfinite(want[i])], posinf=1, neginf=-1), err_msg=n)


@pytest.mark.parametrize("what", ["K", "Q", "overflow"])
@pytest.mark.parametrize("b,d", [(1, 64), (16, 64), (16, 128)])
def test_a_tile_of_minus_infinity_is_skipped_only_where_that_is_exact(b, d, what):
    """-inf added to a score that is NaN or overflows is NaN, also where it is -inf
    for the whole tile."""
    print("f32 masks, -inf tiles", b, d, what, flush=True)
    h, s = 16, 130
    inp = attention_inputs(b, h, s, d, DT, seed=37)
    q, k, v, g = (x.copy() for x in (inp.q, inp.k, inp.v, inp.do))
    if what == "K":
        k[:, 0, 40, 3] = np.nan
    elif what == "Q":
        q[:, 0, 33, 3] = np.inf
    else:
        q[:, 0, 5], k[:, 0, 40] = 1e20, 1e20
    mask = torch.zeros(1, 1, s, s, device="cuda")
    mask[..., 32:64] = -np.inf
    t = [abi.dev_tensor(x, DT) for x in (q, k, v, g)]

    def run():
        out, lse, path = abi.forward(*t[:3], mask=mask)
        return [abi.host(x) for x in (out, *abi.backward(*t[:3], out, t[3], lse, mask=mask)[:3])]

    got = run()
    with abi.generic_only():
        want = run()
    assert np.isnan(want[0][:, 0]).any() and np.isfinite(want[0][:, 1:]).all()
    for x, y, n in zip(got, want, ("out", "dq", "dk", "dv")):
        np.testing.assert_array_equal(np.isfinite(x), np.isfinite(y), err_msg=n)
        # (the head's rows are NaN, and their P without a sum to divide by: the others')
        np.testing.assert_allclose(x[:, 1:], y[:, 1:], **TOL, err_msg=n)
