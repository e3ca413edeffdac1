"""The GPT-2 block kernels (include/tfgfa_gpt2.h) on torch tensors, for model_inference.

The functions launch on the current stream and return new tensors (except where said).  They
take what :func:`takes` accepts and leave everything else to the caller's torch operators.
"""
from __future__ import annotations

import torch
from torch.autograd import forward_ad

from . import _C, _launch_on

MAX_NORM_DIM = _C.GPT2_MAX_NORM_DIM
MAX_ROWS = _C.GPT2_MAX_ROWS
MAX_NORM_ROWS = _C.GPT2_MAX_NORM_ROWS
MAX_VALUES = _C.GPT2_MAX_VALUES
_NORM_LDS_FLOATS = 15360  # rows * (width + 4) of a projection with a norm before it
_TYPES = (torch.Tensor, torch.nn.Parameter)


def _has(obj, path: str) -> bool:
    for name in path.split("."):
        obj = getattr(obj, name, None)
    return obj is not None


# What eager() asks torch; a torch without one of them has the modules run its operators.
_ANSWERS = _has(forward_ad, "_current_level") and all(_has(torch, n) for n in (
    "compiler.is_compiling", "_C._get_tracing_state", "_C._len_torch_dispatch_stack",
    "_C._len_torch_function_stack", "_C._functorch.peek_interpreter_stack"))


def eager() -> bool:
    """No tracing, compilation, function transform, forward-mode level or torch mode is active, so
    a kernel launched on raw pointers is what the torch operators would have been."""
    C = torch._C
    return not (torch.compiler.is_compiling() or C._get_tracing_state() is not None
                or C._len_torch_dispatch_stack() or C._len_torch_function_stack()
                or C._functorch.peek_interpreter_stack() is not None
                or forward_ad._current_level >= 0)


if not _ANSWERS:
    def eager() -> bool:
        return False


def takes(x: torch.Tensor, *params, dtypes=(torch.float32,)) -> bool:
    """``x`` (of one of ``dtypes``) and the float32 ``params`` (None allowed) are plain, contiguous,
    16-byte aligned tensors on one GPU and need no gradient."""
    if not (type(x) in _TYPES and x.is_cuda and x.dtype in dtypes and x.is_contiguous()
            and x.data_ptr() % 16 == 0):
        return False
    dev, grad = x.device, torch.is_grad_enabled()
    if grad and x.requires_grad:
        return False
    for p in params:
        if p is not None and not (type(p) in _TYPES and p.dtype == torch.float32 and p.device == dev
                                  and p.is_contiguous() and p.data_ptr() % 16 == 0
                                  and not (grad and p.requires_grad)):
            return False
    return True


def _ptr(t) -> int:
    return 0 if t is None else t.data_ptr()


def _planes(rows: int, width: int, dev):
    return torch.empty((3, rows, width), dtype=torch.bfloat16, device=dev)


def layernorm(x, scale, shift, eps: float, dtype=torch.float32, delta=None, planes: bool = False):
    """LayerNorm over the last dimension, in ``dtype`` (float32 or bfloat16), or as the three bf16
    planes (3, rows, width) that :func:`linear_planes` takes.  With ``delta`` (bf16, like x): the norm
    of x + delta, returned as (x + delta, norm)."""
    d = x.shape[-1]
    rows = x.numel() // d
    y = _planes(rows, d, x.device) if planes else torch.empty(x.shape, dtype=dtype, device=x.device)
    s = None if delta is None else torch.empty_like(x)
    kind = _C.GPT2_PLANES if planes else _C.GPT2_BF16 if dtype == torch.bfloat16 else _C.GPT2_F32
    _launch_on(x.get_device(), _C.gpt2_layernorm, x.data_ptr(), _ptr(delta), _ptr(s), scale.data_ptr(),
               shift.data_ptr(), y.data_ptr(), kind, rows, d, eps)
    return y if delta is None else (s, y)


def planes_splits(rows: int, w) -> int:
    """Splits of the contraction :func:`linear_planes` would use, 0 where it does not take the sizes."""
    return _C.gpt2_linear_planes_splits(rows, *w.shape)


def linear_planes(x, w, bias, splits: int, gelu: bool = False, residual=None):
    """x w^T + bias for ``x`` as (3, rows, K) planes and float32 ``w`` (N, K): + ``residual`` (float32, any
    shape of rows x N, the result's too), or with ``gelu`` its GELU as planes (3, rows, N)."""
    rows, (N, K), dev = x.shape[1], w.shape, x.device
    part = None
    if gelu:
        y = _planes(rows, N, dev)
    else:
        y = torch.empty((rows, N) if residual is None else residual.shape, dtype=torch.float32, device=dev)
    if splits > 1:
        part = torch.empty((splits, rows, N), dtype=torch.float32, device=dev)
    _launch_on(x.get_device(), _C.gpt2_linear_planes, x.data_ptr(), w.data_ptr(), _ptr(bias), gelu,
               _ptr(residual), y.data_ptr(), _ptr(part), splits, rows, N, K)
    return y


def gelu(x):
    """0.5 x (1 + tanh(sqrt(2/pi) (x + 0.044715 x^3)))"""
    y = torch.empty_like(x)
    _launch_on(x.get_device(), _C.gpt2_gelu, x.data_ptr(), y.data_ptr(), x.numel())
    return y


def cast_bf16(pairs) -> None:
    """dst.copy_(src) for each (src float32, dst bf16) pair of equal, multiple-of-4 sizes."""
    _launch_on(pairs[0][0].get_device(), _C.gpt2_cast_bf16,
               [(s.data_ptr(), d.data_ptr(), s.numel()) for s, d in pairs])


def rows_fit(rows: int, width: int, norm: bool) -> bool:
    """Whether :func:`linear_rows` takes ``rows`` rows of ``width`` values, and gives as many."""
    return (1 <= rows <= MAX_ROWS and width % 4 == 0 and 4 <= width <= _C.GPT2_MAX_OUTPUTS
            and (not norm or (width <= MAX_NORM_DIM and rows * (width + 4) <= _NORM_LDS_FLOATS)))


def linear_rows(x, parts, dtype, norm=None, gelu=False, residual=None):
    """y = f(xhat w^T + bias) (+ residual) for each (w, bias) of ``parts`` (at most 3, equal shapes),
    as a list of tensors of ``dtype``.  ``x``: (..., K) float32 or bf16, few rows (:func:`rows_fit`);
    ``norm`` = (scale, shift, eps): xhat is x's LayerNorm (x float32); with a norm ``gelu`` makes f the
    GELU, or ``dtype`` may be bf16."""
    N, K = parts[0][0].shape
    ys = [torch.empty(x.shape[:-1] + (N,), dtype=dtype, device=x.device) for _ in parts]
    scale, shift, eps = norm if norm is not None else (None, None, 0.0)
    _launch_on(x.get_device(), _C.gpt2_linear_rows, x.data_ptr(), x.dtype == torch.bfloat16, _ptr(scale),
               _ptr(shift), eps, [(w.data_ptr(), _ptr(b), y.data_ptr()) for (w, b), y in zip(parts, ys)],
               gelu, _ptr(residual), dtype == torch.bfloat16, x.numel() // K, N, K)
    return ys
