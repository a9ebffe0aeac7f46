"""Which sizes the layer kernels and the split forward take, on both sides of each
rule's lines: sizes where the library's product, the chain of array operations or
the unsplit forward measured faster are not theirs."""

from __future__ import annotations

import ctypes

import pytest

pytest.importorskip("torch")

from tensorsmith_hip import _lib  # noqa: E402
from tensorsmith_hip.nn import functional as F  # noqa: E402


@pytest.mark.parametrize("tokens,m,n,pays", [
    (4095, 512, 512, False), (4096, 512, 512, True), (131072, 1024, 2048, True),
    (8192, 1400, 1400, True), (4096, 3072, 768, True), (65535, 1536, 1536, True), (65536, 1536, 1536, False),
    (4096, 4096, 1024, False), (32768, 18432, 16, False), (4096, 16, 16384, False), (4096, 16, 8192, True),
    (4096, 128, 16384, True)])
def test_weight_gradients(tokens, m, n, pays):
    assert F._wgrad_pays(tokens, m, n) == pays
    assert F._wgrad_pays(tokens, n, m) == pays


@pytest.mark.parametrize("tokens,stride", [(1, 2**29), (1, 2**25), (4096, 2**18 - 8)])
def test_weight_gradients_refuse_rows_past_their_offsets(tokens, stride):
    """Rows past the last token are addressed and read as zeros: with their 32-bit
    offsets wrapped they would be token 0 again.  (Refused before any launch.)"""
    lib, at = _lib.load(), 1 << 20
    rc = lib.tsattn_linear_wgrad(_lib.F16, _lib.F16, tokens, 64, 64, at, stride, at, stride, at, at,
                                 lib.tsattn_linear_wgrad_workspace(tokens, 64, 64), None)
    assert rc == _lib.ERR_UNSUPPORTED


@pytest.mark.parametrize("rows,k,n,pays", [
    (1, 512, 32000, True), (16, 4096, 11008, True), (17, 4096, 11008, False), (32, 4096, 8192, True),
    (1, 4096, 14336, False), (33, 4096, 8192, True), (33, 512, 8196, False), (1, 8192, 4, True),
    (1, 8200, 4, False), (4, 1048576, 4, False), (1, 12288, 4096, True), (64, 8192, 5120, False)])
def test_few_rows(rows, k, n, pays):
    assert F._rows_pays(rows, k, n) == pays


@pytest.mark.parametrize("rows,dim,pays", [(1, 8, True), (2**16, 8, True), (2**16 + 1, 8, False),
                                           (2**16 + 1, 56, False), (2**20, 64, True), (2**20, 8192, True)])
def test_norms(rows, dim, pays):
    assert F._norm_pays(rows, dim) == pays


@pytest.mark.parametrize("b,h,sq,sk,causal,parts", [
    (1, 32, 16, 8192, True, 16), (1, 32, 500, 8192, True, 4), (1, 8, 16, 704, False, 2), (1, 8, 1024, 1024, False, 2),
    (1, 16, 1024, 1024, False, 1), (1, 32, 1024, 1024, False, 1), (1, 32, 1024, 2048, False, 1),
    (1, 32, 1024, 4096, False, 2), (1, 16, 1024, 2048, False, 4), (1, 16, 2048, 2048, True, 2),
    (1, 8, 4096, 4096, True, 2), (4, 32, 128, 800, False, 1), (4, 32, 128, 3000, False, 4), (1, 33, 1024, 8192, False, 1),
    (1, 16, 800, 1100, False, 1), (1, 16, 1000, 1600, False, 1), (1, 32, 500, 1600, False, 1),
    (1, 32, 1024, 2400, True, 1), (3, 8, 1000, 1600, True, 1), (8, 8, 244, 1254, False, 1)])
def test_split_forwards(b, h, sq, sk, causal, parts):
    p = _lib.Problem()
    p.dtype, p.batch, p.heads_q, p.heads_kv = _lib.BF16, b, h, h
    p.len_q, p.len_kv, p.dim_qk, p.dim_v, p.scale = sq, sk, 128, 128, 0.1
    p.is_causal, p.causal_offset, p.mask_kind = int(causal), sk - sq, _lib.MASK_NONE
    want = parts * b * h * sq * 130 * 4 if parts > 1 else 0
    assert _lib.load().tsattn_sdpa_forward_workspace(ctypes.byref(p)) == want
