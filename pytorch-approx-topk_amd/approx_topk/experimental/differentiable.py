"""``approx_topk.topk`` with a gradient.

The reference registers no autograd formula for its operator
(approx_topk/priority_queue.py:14: ``mutates_args=()`` and nothing else), and
neither does ``approx_topk.topk`` here: an autograd kernel on the operator
costs every call about 3 us of host time, gradient or not.  This wrapper is the
opt-in: same arguments, same results, and the values' gradient flows back to
the input.  The values are a gather of the input at the returned indices, so
their gradient scatters to those positions and every other position gets zero;
the indices are distinct along ``dim``, so a plain scatter is exact.

Along the last dim one kernel writes the gradient (``csrc/topk_grad.hip``); zeros
and a scatter are left to derivatives of the gradient and to the dims the operator takes only
when every bucket is kept whole.
"""
from __future__ import annotations

import torch
from torch import Tensor, is_grad_enabled
from torch._C import _AutoDispatchBelowAutograd, _is_torch_function_mode_enabled
from torch._C._functorch import peek_interpreter_stack
from torch.autograd import forward_ad
from torch.compiler import is_compiling

from .. import _native
from ..priority_queue import topk as _topk, topk_grad as _topk_grad


_PLAIN = (Tensor, torch.nn.Parameter)


def _autograd_has_work(grad_values: Tensor) -> bool:
    """Whether the gradient may itself be differentiated or traced: reverse mode, forward mode (both kinds enter
    a level), a functorch transform, or ``torch.compile``, which does not look into dispatcher guards."""
    return ((is_grad_enabled() and grad_values.requires_grad) or forward_ad._current_level >= 0
            or peek_interpreter_stack() is not None or is_compiling())


def _gradient(grad_values: Tensor | None, indices: Tensor, shape: torch.Size, dtype: torch.dtype, dim: int, k0: int,
              j: int, interleaved: bool) -> Tensor:
    """The gradient with respect to an input of `shape` and `dtype`, given that of the values."""
    if grad_values is None:  # (not materialized: that would fill an int64 gradient of the indices as well)
        return indices.new_zeros(shape, dtype=dtype)
    if len(shape) and dim == len(shape) - 1 and indices.numel() and shape[-1] <= _native.MAX_GRAD_ROW:
        if _autograd_has_work(grad_values):
            return _topk_grad(grad_values, indices, shape[-1], k0, j, interleaved)
        # the operator's autograd kernel would find nothing to do, in 6 us of host time
        with _AutoDispatchBelowAutograd():
            return _topk_grad(grad_values, indices, shape[-1], k0, j, interleaved)
    if len(shape) == 0:
        return grad_values.reshape(()) if indices.numel() else grad_values.new_zeros(())
    return grad_values.new_zeros(shape).scatter(dim, indices, grad_values)


if _native.host is not None:
    _native.host.set_gradient(_gradient)


class _TopkWithGradient(torch.autograd.Function):
    @staticmethod
    def forward(ctx, xs, k, dim, j, k_mult, interleaved, multithread_buckets):
        values, indices = _topk(xs, k, dim, j, k_mult, interleaved, multithread_buckets)
        ctx.dim = dim if dim >= 0 else dim + xs.ndim
        ctx.shape, ctx.dtype = xs.shape, xs.dtype
        ctx.buckets = (k * k_mult, j, interleaved)
        ctx.set_materialize_grads(False)
        ctx.save_for_backward(indices)
        ctx.mark_non_differentiable(indices)
        return values, indices

    @staticmethod
    def backward(ctx, grad_values, _grad_indices):
        (indices,) = ctx.saved_tensors
        grad_xs = _gradient(grad_values, indices, ctx.shape, ctx.dtype, ctx.dim, *ctx.buckets)
        return grad_xs, None, None, None, None, None, None


def topk(
    xs: Tensor,
    k: int,
    dim: int,
    j: int = 1,
    k_mult: int = 1,
    interleaved: bool = True,
    multithread_buckets: bool | None = False,
) -> tuple[Tensor, Tensor]:
    """``approx_topk.topk`` whose values carry a gradient with respect to ``xs``."""
    # Plain GPU tensors outside of every transform and mode that would see the operator's call: the same node in
    # native code (csrc/host_binding.cpp), whose backward leaves all but a plain gradient to `_gradient`.
    if (not is_compiling() and _native.host is not None and type(xs) in _PLAIN and xs.is_cuda
            and peek_interpreter_stack() is None and forward_ad._current_level < 0
            and not _is_torch_function_mode_enabled()):
        out = _native.host.differentiable_topk(xs, k, dim, j, k_mult, interleaved, multithread_buckets)
        if out is not None:
            return out
    return _TopkWithGradient.apply(xs, k, dim, j, k_mult, interleaved, multithread_buckets)
