"""General masks on the fp32 matrix-core kernels, against the oracle and the
generic kernels.

Boolean and additive masks of any broadcast strides are read one tile ahead of
the products, and a tile the mask forbids whole is skipped.  The cases sit
where that can go wrong: ragged ends in both directions, one row or key more
than a tile, strides that are not the key order, whole tiles and whole rows
masked, grouped heads, and both forms (split and whole) of the kernels.  Bounds
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
        m[..., 7, :] = -np.inf  # a row that sees nothing
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
    out, lse, path = abi.forward(q, k, v, **kw)
    grads = abi.backward(q, k, v, out, g, lse, **kw)
    torch.cuda.synchronize()
    assert path == _lib.PATH_MFMA and grads[3] == _lib.PATH_MFMA
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
