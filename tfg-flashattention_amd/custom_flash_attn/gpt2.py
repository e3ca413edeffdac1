"""The GPT-2 block kernels (include/tfgfa_gpt2.h) on torch tensors, for model_inference.

The functions launch on the current stream and return new tensors (except where said).  They
take what :func:`takes` accepts and leave everything else to the caller's torch operators.
"""
from __future__ import annotations

import torch
from torch.autograd import forward_ad

from . import _C

MAX_NORM_DIM = _C.GPT2_MAX_NORM_DIM
_TYPES = (torch.Tensor, torch.nn.Parameter)


def eager() -> bool:
    """No tracing, compilation, function transform, forward-mode level or torch mode is active, so
    a kernel launched on raw pointers is what the torch operators would have been."""
    C = torch._C
    return not (torch.compiler.is_compiling() or C._get_tracing_state() is not None
                or C._len_torch_dispatch_stack() or C._len_torch_function_stack()
                or C._functorch.peek_interpreter_stack() is not None
                or forward_ad._current_level >= 0)


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


def _stream(dev) -> int:
    return torch.cuda.current_stream(dev).cuda_stream


def layernorm(x, scale, shift, eps: float, dtype=torch.float32, delta=None):
    """LayerNorm over the last dimension, in ``dtype`` (float32 or bfloat16).  With ``delta`` (bf16,
    like x): the norm of x + delta, returned as (x + delta, norm)."""
    d = x.shape[-1]
    y = torch.empty(x.shape, dtype=dtype, device=x.device)
    s = None if delta is None else torch.empty_like(x)
    with torch.cuda.device(x.device):
        _C.gpt2_layernorm(x.data_ptr(), _ptr(delta), _ptr(s), scale.data_ptr(), shift.data_ptr(),
                          y.data_ptr(), dtype == torch.bfloat16, x.numel() // d, d, eps,
                          _stream(x.device))
    return y if delta is None else (s, y)


def gelu(x):
    """0.5 x (1 + tanh(sqrt(2/pi) (x + 0.044715 x^3)))"""
    y = torch.empty_like(x)
    with torch.cuda.device(x.device):
        _C.gpt2_gelu(x.data_ptr(), y.data_ptr(), x.numel(), _stream(x.device))
    return y
