"""Tape ops around the attention path, on hip tensors.

Each op is one autograd node with the reference's semantics
(``src/tensorsmith/nn/functional.py`` and ``nn/primitives.py``).  The norms and
the SwiGLU activation run as one HIP kernel a pass (``csrc/layers.hip``) where
their operands allow; the rest of the array math, and operands outside those
kernels, as PyTorch-ROCm library calls on the device tensors (GEMMs in
hipBLASLt).
"""

from __future__ import annotations

import ctypes
import math

from .. import _lib
from ..amp import _autocast, _cast_inputs
from ..device import launch, random_uniform
from ..tensor import Tensor, _sum_to_shape, is_grad_enabled, is_torch, no_grad
from .attention import rotary_embedding, scaled_dot_product_attention

__all__ = [
    "cross_entropy", "dropout", "embedding", "gelu", "layer_norm", "linear", "rms_norm",
    "rotary_embedding", "scaled_dot_product_attention", "silu",
]


def _require_hip(t: Tensor, op: str):
    if not is_torch(t._data):
        raise RuntimeError(f"{op}: tensorsmith_hip computes on hip devices only")


def _code(raw) -> int:
    """The C ABI's code of a dtype the layer kernels take, or -1."""
    import torch

    return {torch.float32: _lib.F32, torch.float16: _lib.F16, torch.bfloat16: _lib.BF16}.get(raw.dtype, -1)


def _flat(raw):
    """``raw`` as the layer kernels read it: contiguous, 16-byte aligned."""
    raw = raw.contiguous()
    return raw if raw.data_ptr() % 16 == 0 else raw.clone()


def _ptr(raw):
    return None if raw is None else ctypes.c_void_p(raw.data_ptr())


def _compute(raw):
    """Half inputs compute in float32 (reference ``primitives.py:16-18``)."""
    import torch

    return raw.float() if raw.dtype in (torch.float16, torch.bfloat16) else raw


def linear(input: Tensor, weight: Tensor, bias: Tensor | None = None) -> Tensor:
    """x @ W^T + b as one node (reference ``functional.py:63-90``), autocast-aware:
    the casts belong to the node, its gradients are rounded as the cast operands'
    would be and returned in the dtypes of the operands given."""
    given = (input, weight) if bias is None else (input, weight, bias)
    casts = bool(_autocast.get())
    if casts:
        with no_grad():
            input, weight, bias = _cast_inputs(input, weight, bias)
    if input.ndim < 1 or weight.ndim != 2 or input.shape[-1] != weight.shape[1]:
        raise ValueError("linear expects [...,in_features] and [out_features,in_features]")
    parents = (input, weight) if bias is None else (input, weight, bias)
    dev = input.device
    if any(p.device is not dev and p.device != dev for p in parents):
        raise ValueError("linear tensors must be on the same device")
    if bias is not None and bias.shape != (weight.shape[0],):
        raise ValueError("linear bias must have shape [out_features]")
    _require_hip(input, "linear")
    w = weight._data
    x = input._data.reshape(-1, weight.shape[1])
    out = _rows_linear(x, w, None if bias is None else bias._data, dev)
    if out is None:
        out = x @ w.t()
        if bias is not None:
            out = out + bias._data.to(out.dtype)
    out = out.reshape(input.shape[:-1] + (weight.shape[0],))

    def backward(g):
        flat = g.reshape(-1, weight.shape[0])
        grads = [(flat @ w).reshape(input.shape).to(input.dtype),
                 _weight_grad(flat, x, dev, weight.dtype, given[1].dtype)]
        if bias is not None:
            grads.append(flat.sum(0).to(bias.dtype))
        return tuple(d.to(t.dtype) for d, t in zip(grads, given)) if casts else tuple(grads)

    return Tensor._from_op(out, given, backward, "linear")


def _wgrad_pays(tokens: int, m: int, n: int) -> bool:
    """Whether the split contraction is the faster one: a long product of an output
    small enough to leave most of the chip idle otherwise.  Library and kernel, us:
    512 x 512 over 8192 tokens 52 and 20, 1400 x 1400 67 and 47; 3072 x 768 over 4096
    41 and 38, 4096 x 1024 48 and 51; at 2048 tokens both take about 19.  Outputs of
    more than half as many 128 x 128 tiles as CUs lose their lead over many tokens
    (1536 x 1536: 65536 tokens 543 and 485, 131072 852 and 1034), thin ones of many
    tiles are mostly padding (16 x 16384 over 4096: 22 and 26)."""
    tiles = -(-m // 128) * -(-n // 128)
    return (tokens >= 4096 and tiles <= (144 if tokens < 65536 else 128)
            and (tiles <= 64 or min(m, n) >= 128))


def _weight_grad(g, x, dev, dtype, store):
    """``g^T x`` over the tokens, rounded to ``dtype`` and given in ``store`` (that
    or float32, into which the kernel widens the rounded sums): one split contraction
    kernel (``tsattn_linear_wgrad``) where that pays, else the library's product."""
    tokens, m = g.shape
    if g.dtype.itemsize != 2 or tokens < 4096:
        return (g.t() @ x).to(dtype)
    import torch

    n = x.shape[1]
    if (g.dtype not in (torch.float16, torch.bfloat16) or x.dtype != g.dtype or not _wgrad_pays(tokens, m, n)
            or m % 8 or n % 8 or m == 0 or n == 0
            or (tokens + 32) * max(g.stride(0), x.stride(0)) * 2 >= 2**31
            or any(t.stride(1) != 1 or t.stride(0) % 8 or t.stride(0) < t.shape[1] or t.data_ptr() % 16
                   for t in (g, x))):
        return (g.t() @ x).to(dtype)
    if store != torch.float32 or dtype != g.dtype:
        store = g.dtype
    lib = _lib.load()
    out = torch.empty((m, n), dtype=store, device=g.device)
    nbytes = lib.tsattn_linear_wgrad_workspace(tokens, m, n)
    try:
        ws = torch.empty(nbytes, dtype=torch.uint8, device=g.device)
    except torch.OutOfMemoryError:  # no room for the partial sums
        return (g.t() @ x).to(dtype)
    _lib.check(launch(dev, lib.tsattn_linear_wgrad, _code(g), _code(out), tokens, m, n, g.data_ptr(), g.stride(0),
                      x.data_ptr(), x.stride(0), out.data_ptr(), ws.data_ptr(), nbytes), "linear weight gradient")
    return out if dtype == g.dtype else out.to(dtype)


def _rows_pays(rows: int, k: int, n: int) -> bool:
    """Whether a few rows' product is the faster call on its own kernel: as long as
    the library's, bound by some 19 us of host time, does not end in the GPU's
    (K 4096, N 4096: 10 us here).  The kernel reads large weights at 4.5 TB/s, the
    library a little faster (N 28672, K 4096, 1 row: 37 us here, 35 there; over 16
    rows N 11008: 20 and 19; over 32 rows each weight is read by two row blocks:
    N 16384, 64 rows: 51 and 32).  And a long contraction of few outputs is one
    workgroup's serial chain (N 256: K 8192 12 and 19 us, 16384 21 and 19, 65536 72
    and 43)."""
    if rows > 32 and n > 8192:
        return False
    return n * k * 2 <= (96 if rows <= 16 else 64) << 20 and (k <= 8192 or n >= 4096)


def _rows_linear(x, w, bias, dev):
    """``x W^T (+ bias)`` of a few 16-bit rows in one kernel
    (``tsattn_rows_linear``), or None outside it.  The kernel's offsets are
    32-bit: rows picked out of a tensor of 2^31 bytes and more are the library's."""
    rows, k = x.shape
    if x.dtype.itemsize != 2 or rows > 64:
        return None
    import torch

    n = w.shape[0]
    if (x.dtype not in (torch.float16, torch.bfloat16) or w.dtype != x.dtype or rows == 0
            or not _rows_pays(rows, k, n) or k % 8 or n % 4 or k == 0 or n == 0 or x.stride(1) != 1
            or x.stride(0) % 8 or (rows * x.stride(0) + k) * 2 >= 2**31
            or not w.is_contiguous() or x.data_ptr() % 16 or w.data_ptr() % 16
            or (bias is not None and (bias.dtype != x.dtype or not bias.is_contiguous()
                                      or bias.data_ptr() % 16))):
        return None
    out = torch.empty((rows, n), dtype=x.dtype, device=x.device)
    _lib.check(launch(dev, _lib.load().tsattn_rows_linear, _code(x), rows, k, n, x.data_ptr(), x.stride(0),
                      w.data_ptr(), None if bias is None else bias.data_ptr(), None, 0, out.data_ptr(), n),
               "few-row linear")
    return out


def gelu(input: Tensor) -> Tensor:
    """Tanh-approximate GELU (reference ``primitives.py:21-49``)."""
    _require_hip(input, "gelu")
    import torch

    x = _compute(input._data)
    factor = math.sqrt(2 / math.pi)
    tangent = torch.tanh(factor * (x + 0.044715 * x**3))
    out = (0.5 * x * (1 + tangent)).to(input.dtype)

    def backward(g):
        d = 0.5 * (1 + tangent) + 0.5 * x * (1 - tangent**2) * factor * (1 + 3 * 0.044715 * x**2)
        return ((g * d).to(input.dtype),)

    return Tensor._from_op(out, (input,), backward, "bias_gelu")


def _norm_pays(rows: int, dim: int) -> bool:
    """Whether the norm kernel, a wave a row, is the faster one: many rows shorter
    than a wave's lanes leave it idle (f32, 2^20 rows of 8, forward and VJP: 742 us
    here, 209 as a chain of array operations; of 64: 1032 and 1646; 2^16 rows of 8: 65 and
    109)."""
    return dim >= 64 or rows <= 2**16


def _norm(input: Tensor, weight: Tensor, bias: Tensor | None, eps: float, rms: bool) -> Tensor:
    """Layer / RMS norm over the trailing ``weight.ndim`` dims (reference
    ``primitives.py:67-136``): half inputs compute in float32, the VJP uses
    the saved normalised values and reciprocal std."""
    if eps <= 0 or not math.isfinite(eps):
        raise ValueError("eps must be positive")
    if input.shape[-weight.ndim:] != weight.shape:
        raise ValueError("normalization weight must match the trailing input dimensions")
    if bias is not None and bias.shape != weight.shape:
        raise ValueError("normalization bias and weight must have equal shapes")
    parents = (input, weight) if bias is None else (input, weight, bias)
    dev = input.device
    if any(p.device is not dev and p.device != dev for p in parents):
        raise ValueError("normalization tensors must be on the same device")
    _require_hip(input, "rms_norm" if rms else "layer_norm")
    dim = math.prod(weight.shape)
    if (0 < dim <= 8192 and dim % 8 == 0 and _code(input._data) >= 0 and _code(weight._data) >= 0
            and input.size > 0 and (bias is None or bias.dtype == weight.dtype)
            and _norm_pays(input.size // dim, dim)):
        return _norm_kernel(input, weight, bias, eps, rms, dim, parents)
    axes = tuple(range(input.ndim - weight.ndim, input.ndim))
    x = _compute(input._data)
    w = weight._data.to(x.dtype)
    centered = x if rms else x - x.mean(dim=axes, keepdim=True)
    rstd = 1 / (centered.square().mean(dim=axes, keepdim=True) + eps).sqrt()
    normalized = centered * rstd
    out = normalized * w
    if bias is not None:
        out = out + bias._data.to(x.dtype)
    out = out.to(input.dtype)

    def backward(g):
        g = g.to(x.dtype)
        weighted = g * w
        dx = rstd * (weighted - normalized * (weighted * normalized).mean(dim=axes, keepdim=True))
        if not rms:
            dx = dx - rstd * weighted.mean(dim=axes, keepdim=True)
        grads = [dx.to(input.dtype), _sum_to_shape(g * normalized, weight.shape).to(weight.dtype)]
        if bias is not None:
            grads.append(_sum_to_shape(g, bias.shape).to(bias.dtype))
        return tuple(grads)

    return Tensor._from_op(out, parents, backward, "rms_norm" if rms else "layer_norm")


def _norm_kernel(input, weight, bias, eps, rms, dim, parents) -> Tensor:
    """``_norm`` in one kernel, and its VJP (``tsattn_norm_forward`` / ``_backward``)."""
    import torch

    lib = _lib.load()
    x, w = _flat(input._data), _flat(weight._data)
    b = None if bias is None else _flat(bias._data)
    code, w_code, rows = _code(x), _code(w), x.numel() // dim
    out = torch.empty(x.shape, dtype=x.dtype, device=x.device)
    mean = rstd = None
    if is_grad_enabled() and any(p.requires_grad for p in parents):
        rstd = torch.empty(rows, dtype=torch.float32, device=x.device)
        mean = None if rms else torch.empty(rows, dtype=torch.float32, device=x.device)
    _lib.check(launch(input.device, lib.tsattn_norm_forward, code, w_code, rows, dim, rms, _ptr(x), _ptr(w),
                      _ptr(b), _ptr(out), _ptr(mean), _ptr(rstd), eps), "norm")

    def backward(g):
        g = _flat(g.to(x.dtype))
        dx = torch.empty(x.shape, dtype=x.dtype, device=x.device)
        dw = torch.empty(w.shape, dtype=w.dtype, device=x.device)
        db = None if b is None else torch.empty(b.shape, dtype=b.dtype, device=x.device)
        nbytes = lib.tsattn_norm_backward_workspace(rows, dim, rms)
        ws = torch.empty(nbytes, dtype=torch.uint8, device=x.device)
        _lib.check(launch(input.device, lib.tsattn_norm_backward, code, w_code, rows, dim, rms, _ptr(x),
                          _ptr(w), _ptr(g), _ptr(mean), _ptr(rstd), _ptr(dx), _ptr(dw), _ptr(db),
                          _ptr(ws), nbytes), "norm backward")
        return (dx, dw) if b is None else (dx, dw, db)

    return Tensor._from_op(out, parents, backward, "rms_norm" if rms else "layer_norm")


def layer_norm(input: Tensor, weight: Tensor, bias: Tensor | None = None, eps: float = 1e-5) -> Tensor:
    """Layer norm (reference ``primitives.py:134-135``)."""
    return _norm(input, weight, bias, eps, False)


def rms_norm(input: Tensor, weight: Tensor, eps: float = 1e-6) -> Tensor:
    """RMS norm, ``x / sqrt(mean(x^2) + eps) * weight`` (reference ``primitives.py:138-139``)."""
    return _norm(input, weight, None, eps, True)


def silu(input: Tensor) -> Tensor:
    """``x * sigmoid(x)`` in float32 for half inputs (reference ``primitives.py:52-64``)."""
    _require_hip(input, "silu")
    import torch

    x = _compute(input._data)
    sig = torch.sigmoid(x)
    out = (x * sig).to(input.dtype)

    def backward(g):
        return ((g.to(x.dtype) * (sig + x * sig * (1 - sig))).to(input.dtype),)

    return Tensor._from_op(out, (input,), backward, "silu")


def _silu_mul(gate: Tensor, up: Tensor) -> Tensor:
    """``silu(gate) * up``, the SwiGLU activation (reference
    ``transformer.py:190-205``): one kernel forward and one backward, rounding
    where the two ops would."""
    a, b = gate._data, up._data
    if (not is_torch(a) or not is_torch(b) or a.dtype != b.dtype or a.shape != b.shape
            or gate.device != up.device or _code(a) < 0 or a.numel() == 0 or a.numel() % 8):
        return silu(gate) * up
    import torch

    lib, code = _lib.load(), _code(a)
    a, b = _flat(a), _flat(b)
    out = torch.empty(a.shape, dtype=a.dtype, device=a.device)
    _lib.check(launch(gate.device, lib.tsattn_silu_mul, code, a.numel(), _ptr(a), _ptr(b), _ptr(out)), "SwiGLU")

    def backward(g):
        g = _flat(g.to(a.dtype))
        da, db = torch.empty_like(a), torch.empty_like(b)
        _lib.check(launch(gate.device, lib.tsattn_silu_mul_backward, code, a.numel(), _ptr(a), _ptr(b),
                          _ptr(g), _ptr(da), _ptr(db)), "SwiGLU backward")
        return da, db

    return Tensor._from_op(out, (gate, up), backward, "silu_mul")


def embedding(indices: Tensor, weight: Tensor) -> Tensor:
    """Row gather with scatter-add VJP (reference ``functional.py:130-142``)."""
    if indices.requires_grad:
        raise ValueError("embedding indices cannot require gradients")
    if indices.device != weight.device:
        raise ValueError("indices and embedding weight must be on the same device")
    _require_hip(weight, "embedding")
    idx = indices._data.long()
    out = weight._data[idx]

    def backward(g):
        import torch

        grad = torch.zeros_like(weight._data)
        grad.index_add_(0, idx.reshape(-1), g.reshape(-1, weight.shape[-1]).to(grad.dtype))
        return (grad,)

    return Tensor._from_op(out, (weight,), backward, "embedding")


def dropout(input: Tensor, p: float = 0.5, training: bool = True) -> Tensor:
    """Inverted dropout (reference ``functional.py:121-127``); identity when off."""
    if not 0 <= p < 1:
        raise ValueError("dropout probability must be in [0, 1)")
    if not training or p == 0:
        return input
    _require_hip(input, "dropout")
    mask = (random_uniform(input.shape, input.device) >= p).to(input.dtype) / (1 - p)
    return Tensor._from_op(input._data * mask, (input,), lambda g: (g * mask,), "dropout")


def cross_entropy(input: Tensor, target: Tensor, reduction: str = "mean", *, axis: int = 1,
                  ignore_index: int = -100, label_smoothing: float = 0.0) -> Tensor:
    """Indexed cross-entropy (reference ``functional.py:397-472``)."""
    if input.ndim < 2:
        raise ValueError("cross_entropy expects logits with at least two dimensions")
    if input.device != target.device or "float" not in str(input.dtype):
        raise ValueError("cross_entropy needs floating logits and targets on the same device")
    if not 0 <= label_smoothing <= 1:
        raise ValueError("label_smoothing must be in [0, 1]")
    if reduction not in {"mean", "sum", "none"}:
        raise ValueError("reduction must be 'none', 'mean', or 'sum'")
    if target.requires_grad:
        raise ValueError("class targets cannot require gradients")
    if "int" not in str(target.dtype):
        raise TypeError("class targets must have an integer dtype")
    if not -input.ndim <= axis < input.ndim:
        raise ValueError("class axis is out of range")
    _require_hip(input, "cross_entropy")
    import torch

    axis %= input.ndim
    classes = input.shape[axis]
    expected = input.shape[:axis] + input.shape[axis + 1:]
    labels = target._data
    if tuple(labels.shape) != expected:
        raise ValueError(f"target shape {tuple(labels.shape)} does not match logits shape {input.shape}")
    valid = labels != ignore_index
    if bool((((labels < 0) | (labels >= classes)) & valid).any()):
        raise ValueError("target class index is out of range")
    perm = tuple(i for i in range(input.ndim) if i != axis) + (axis,)
    inverse = tuple(perm.index(i) for i in range(input.ndim))
    logits = _compute(input._data.permute(*perm).reshape(-1, classes))
    index = torch.where(valid, labels, torch.zeros_like(labels)).reshape(-1).long()
    active = valid.reshape(-1)
    log_probs = torch.log_softmax(logits, dim=-1)
    losses = -(1 - label_smoothing) * log_probs.gather(1, index[:, None])[:, 0]
    if label_smoothing:
        losses = losses - label_smoothing * log_probs.mean(dim=-1)
    losses = torch.where(active, losses, torch.zeros_like(losses))
    count = max(int(valid.sum()), 1)
    out = losses.reshape(expected) if reduction == "none" else losses.sum() / (
        count if reduction == "mean" else 1)

    def backward(g):
        grad = log_probs.exp() - label_smoothing / classes
        grad.scatter_add_(1, index[:, None], torch.full_like(grad[:, :1], -(1 - label_smoothing)))
        grad = torch.where(active[:, None], grad, torch.zeros_like(grad))
        grad = grad * (g.reshape(-1, 1) if reduction == "none"
                       else g / (count if reduction == "mean" else 1))
        return (grad.reshape(expected + (classes,)).permute(*inverse).to(input.dtype),)

    return Tensor._from_op(out, (input,), backward, "cross_entropy")
