"""Device kernels for the dense steps around the codec.

Each function is an expression of ``components/layers.py`` or
``components/ops.py`` as one or two launches of ``csrc/layers.hip``, or the
product of ``operations.A_compBT`` as one of ``csrc/linear.hip``, for the
tensors that ``native`` accepts; the callers keep ATen's expression for the
others (host tensors, other types, strided views, and wherever autograd,
tracing or a transform has to see the operations).
"""
from __future__ import annotations

import torch
from torch import Tensor
from torch.autograd import forward_ad

from . import hip

_PLAIN = (Tensor, torch.nn.Parameter)
_MAX_COLUMNS = 4096
# The entry points' limits, larger tensors being ATen's: a launch has fewer than
# 2^32 threads (lct_relu_square: 8 elements each; lct_rms_norm: 64 per row).
_MAX_ELEMENTS = 1 << 33
_MAX_NORM_ROWS = (1 << 26) - 4
# Row groups of the partial sums: the most that lct_column_sum and
# lct_rms_norm_backward make.
_COLUMN_GROUPS = 128
_NORM_GROUPS = 512
_MIN_SUM_ROWS = 1024


def native(*tensors: Tensor) -> bool:
    """Whether the kernels may read ``tensors`` directly: plain non-empty
    contiguous device tensors of the current device, with no autograd graph,
    forward-mode level, transform, dispatch mode, autocast or tracing that
    would have to see the operations."""
    if (torch.compiler.is_compiling() or torch._C._get_tracing_state() is not None
            or torch._C._len_torch_dispatch_stack() or forward_ad._current_level >= 0
            or torch.is_autocast_enabled("cuda")):
        return False
    grad = torch.is_grad_enabled()
    for t in tensors:
        if (type(t) not in _PLAIN or not t.is_cuda or t.get_device() != torch._C._cuda_getDevice()
                or not t.is_contiguous() or t.numel() == 0
                or (grad and t.requires_grad) or torch._C._functorch.is_functorch_wrapped_tensor(t)
                or t.data_ptr() & 15 or t.is_conj() or t.is_neg()):
            return False
    return True


def _stream(tensor: Tensor) -> int:
    return torch._C._cuda_getCurrentRawStream(tensor.get_device())


def relu_square(z: Tensor):
    """``(relu(z), relu(z)^2)``, or None."""
    if z.dtype != torch.bfloat16 or z.numel() > _MAX_ELEMENTS or not native(z):
        return None
    relu, square = torch.empty_like(z), torch.empty_like(z)
    hip.call("lct_relu_square", z.data_ptr(), relu.data_ptr(), square.data_ptr(), z.numel(),
             _stream(z))
    return relu, square


def relu_square_backward(grad: Tensor, relu: Tensor):
    """``grad`` becomes the gradient of ``relu(z)^2`` from its own, in place;
    returns ``relu^2``, or None (``grad`` is then as it was)."""
    if (grad.dtype != torch.bfloat16 or relu.dtype != torch.bfloat16 or grad.shape != relu.shape
            or relu.numel() > _MAX_ELEMENTS or not native(grad, relu)):
        return None
    square = torch.empty_like(relu)
    hip.call("lct_relu_square_backward", relu.data_ptr(), grad.data_ptr(), square.data_ptr(),
             relu.numel(), _stream(relu))
    return square


# Where a kernel is faster than the expression it replaces, from host time per
# call and kernel time together (us per call of calls in a row, the kernel's
# against ATen's).


def column_sum_pays(g: Tensor, dtype: torch.dtype) -> bool:
    """:func:`column_sum`, about 13 us up to 8192 x 4096, against ``g.sum(0)`` and,
    unless ``dtype`` is ``g``'s, its cast.  With the cast: 12.7 | 11.9 at 1024 x
    64, 12.8 | 14.3 at 1536 x 64, 13.0 | 15.4 at 1024 x 128, 12.7 | 23.5 at 8192 x
    768.  Without: 13.1 | 12.4 at 1536 x 768, 13.0 | 13.5 at 2048 x 768, 13.0 |
    11.6 at 4096 x 128, 13.0 | 16.0 at 4096 x 256, 12.9 | 20.9 at 8192 x 768."""
    numel = g.numel()
    if g.shape[0] < _MIN_SUM_ROWS:
        return False
    if dtype != g.dtype:
        return numel > 1 << 16
    return numel >= 3 << 19 or (numel >= 1 << 20 and g.shape[0] >= 4096 and g.shape[1] >= 256)


MIN_NORM_ELEMENTS = 1 << 20   # below, norm_pays is False for a gain of x's dtype


def norm_pays(x: Tensor, gain: Tensor) -> bool:
    """:func:`rms_norm`, 11.7 us up to 8192 x 1024.  With a gain that ATen has to
    have cast: 12.0 | 13.5 at any smaller size, 12.4 | 14.9 at 8192 x 1024, 29.6 |
    31.6 at 8192 x 4096.  Without: 11.7 | 7.3 at 1024 x 768, 11.9 | 11.3 at 8192 x
    768, 11.8 to 13.9 | 12.4 at 8192 x 1024, 13.5 | 13.0 at 16384 x 64, 11.8 | 13.8
    at 16384 x 256, 11.8 | 10.4 at 4096 x 2048, 13.5 | 13.5 at 4096 x 3072, 16.0 |
    16.5 at 4096 x 4096, 13.2 | 17.4 at 8192 x 2048: ATen's time follows the
    elements and, as 1024 more of them, the rows."""
    if gain.dtype != x.dtype:
        return True
    numel = x.numel()
    return (numel >= MIN_NORM_ELEMENTS
            and numel + 1024 * (numel // x.shape[-1]) >= 18 << 20)


def norm_backward_pays(x: Tensor) -> bool:
    """:func:`rms_norm_backward` without ``rebuild``, 17.3 us up to 8192 x 1024,
    for a gain of ``x``'s dtype: 17.4 | 10.1 at 16 x 768, 17.3 | 15.0 at 2048 x
    768, 17.2 | 22.0 at 4096 x 768, 17.4 | 14.8 at 4096 x 64, 17.3 | 20.4 at 8192 x
    64, 17.3 | 16.5 at 1024 x 2048, 17.2 | 23.8 at 2048 x 2048, 18.7 | 18.6 at 512 x
    3072, 18.6 | 17.8 at 256 x 4096, 19.1 | 21.7 at 512 x 4096, 74 | 144 at 8192 x
    4096.  (With ``rebuild``: 19.2 | 35 at 16 x 768 and more apart from there.)"""
    numel = x.numel()
    if numel < 1 << 18:
        return False
    cols = x.shape[-1]
    return numel + 512 * (numel // cols) > (2 << 20 if cols > 2048 else 3 << 20)


def column_sum(g: Tensor, dtype: torch.dtype):
    """``g.sum(0).to(dtype)`` of a matrix, or None."""
    if (g.dtype != torch.bfloat16 or dtype not in (torch.bfloat16, torch.float32) or g.ndim != 2
            or g.shape[0] < _MIN_SUM_ROWS or g.shape[1] % 8 or not 0 < g.shape[1] <= 1 << 20
            or g.numel() > _MAX_ELEMENTS or not native(g)):
        return None
    rows, cols = g.shape
    partials = torch.empty(_COLUMN_GROUPS * cols, dtype=torch.float32, device=g.device)
    out = torch.empty(cols, dtype=dtype, device=g.device)
    hip.call("lct_column_sum", g.data_ptr(), rows, cols, partials.data_ptr(), partials.numel(),
             out.data_ptr(), int(dtype == torch.bfloat16), _stream(g))
    return out


def _norm_takes(x: Tensor, gain: Tensor) -> bool:
    return (x.dtype == torch.bfloat16 and gain.dtype in (torch.bfloat16, torch.float32)
            and x.ndim > 0 and gain.shape == x.shape[-1:] and x.shape[-1] % 4 == 0
            and x.shape[-1] <= _MAX_COLUMNS and x.numel() <= _MAX_ELEMENTS)


# lct_skinny_linear's range of A's rows, and of W's.
MAX_SKINNY_TOKENS = 16
_MAX_SKINNY_ROWS = (1 << 29) - 64


def skinny_linear(a: Tensor, w: Tensor):
    """``a @ w.T`` of at most 16 rows, or None (from there on the library's
    product is faster: 21 us against 28 at 17 to 32 rows of 11008 x 4096; below,
    the times of 1 to 16 rows stand at csrc/linear.hip)."""
    if (a.dtype != torch.bfloat16 or w.dtype != torch.bfloat16 or a.ndim != 2
            or w.ndim != 2 or w.shape[1] != a.shape[1]
            or a.shape[0] > MAX_SKINNY_TOKENS or a.shape[1] % 8
            or w.shape[0] > _MAX_SKINNY_ROWS or w.shape[1] > 1 << 30 or not native(a, w)):
        return None
    tokens, cols = a.shape
    rows = w.shape[0]
    out = torch.empty((tokens, rows), dtype=torch.bfloat16, device=a.device)
    hip.call("lct_skinny_linear", a.data_ptr(), w.data_ptr(), out.data_ptr(), tokens, rows, cols,
             _stream(a))
    return out


def rms_norm(x: Tensor, gain: Tensor):
    """``(bf16(x * rstd * bf16(gain)), rstd)`` over the last dimension, or None."""
    if (not _norm_takes(x, gain) or x.numel() > _MAX_NORM_ROWS * x.shape[-1]
            or not native(x, gain)):
        return None
    cols = x.shape[-1]
    y = torch.empty_like(x)
    rstd = torch.empty((*x.shape[:-1], 1), dtype=torch.float32, device=x.device)
    hip.call("lct_rms_norm", x.data_ptr(), gain.data_ptr(), int(gain.dtype == torch.bfloat16),
             y.data_ptr(), rstd.data_ptr(), x.numel() // cols, cols, _stream(x))
    return y, rstd


def rms_norm_backward(grad: Tensor, x: Tensor, rstd: Tensor, gain: Tensor, dtype: torch.dtype,
                      rebuild: bool):
    """``(grad_x, grad_gain, normalized)``: the gradients of :func:`rms_norm`
    (the gain's rounded to BF16, in ``dtype``) and, with ``rebuild``, its
    output again as a matrix (else None); or None."""
    if (not _norm_takes(x, gain) or grad.dtype != torch.bfloat16 or grad.shape != x.shape
            or rstd.dtype != torch.float32 or rstd.numel() * x.shape[-1] != x.numel()
            or dtype not in (torch.bfloat16, torch.float32)
            or not native(grad, x, gain, rstd)):
        return None
    cols = x.shape[-1]
    grad_x = torch.empty_like(x)
    normalized = torch.empty_like(x) if rebuild else None
    grad_gain = torch.empty(cols, dtype=dtype, device=x.device)
    partials = torch.empty(_NORM_GROUPS * cols, dtype=torch.float32, device=x.device)
    hip.call("lct_rms_norm_backward", grad.data_ptr(), x.data_ptr(), rstd.data_ptr(),
             gain.data_ptr(), int(gain.dtype == torch.bfloat16), grad_x.data_ptr(),
             None if normalized is None else normalized.data_ptr(), partials.data_ptr(),
             partials.numel(), grad_gain.data_ptr(), int(dtype == torch.bfloat16),
             x.numel() // cols, cols, _stream(x))
    return grad_x, grad_gain, None if normalized is None else normalized.view(-1, cols)
