"""``mamtorch_kernel_v4::fullyconnected`` wrapper (mamtorch/kernel/v4/fullyconnected.py:6-64).

The reference's v4 kernel is approximate (index packed into the low mantissa bits,
mamtorch/kernel/v4/csrc/cuda/fullyconnected_kernel.cu:133-137); here the same operator name is
served by the exact kernel, so its error against the oracle is zero.

``fullyconnected_wt`` is an addition: it takes the module's ``weight`` (out, in) as stored, so no
transposed copy of the weight is made per call, adds the bias inside the kernel, and returns the
weight gradient in (out, in) layout.  With ``hand_over`` the raw operator returns a fourth tensor of
shape (4, N, out): the selected weights w[argmax], w[argmin] and the selected inputs x[argmax],
x[argmin].  The index resolution has them in hand, and the backward then needs no random reads of
the weight matrix or of the input.
"""
import torch
from torch import Tensor

from .._registration import register_exact_forward

__all__ = ["fullyconnected", "fullyconnected_wt", "fullyconnected_wt_output"]

library_name = "mamtorch_kernel_v4"
K = torch.ops.mamtorch_kernel_v4


def fullyconnected(a: Tensor, b: Tensor) -> list[Tensor]:
    return K.fullyconnected.default(a, b)


def fullyconnected_wt(a: Tensor, weight: Tensor, bias=None) -> list[Tensor]:
    """a (N, in), weight (out, in), bias (out) or None -> [C, argmax, argmin]."""
    # the selected operands are only worth writing when a backward will read them
    hand_over = torch.is_grad_enabled() and (a.requires_grad or weight.requires_grad)
    return K.fullyconnected_wt.default(a, weight, bias, hand_over)[:3]


def fullyconnected_wt_output(a: Tensor, weight: Tensor, bias=None) -> Tensor:
    """C of ``fullyconnected_wt``, for callers that need the indices in the backward only: they go there as one word for both."""
    if weight.size(1) <= 65535 and torch.is_grad_enabled() and (a.requires_grad or weight.requires_grad):
        return K.fullyconnected_wt_picks.default(a, weight, bias)[0]
    return fullyconnected_wt(a, weight, bias)[0]


register_exact_forward(library_name)


@torch.library.register_fake(f"{library_name}::fullyconnected_wt_picks")
def _(a, weight, bias):
    torch._check(a.dim() == 2 and weight.dim() == 2)
    torch._check(a.size(1) == weight.size(1))
    torch._check(a.dtype == torch.float)
    torch._check(weight.dtype == torch.float)
    torch._check(a.device == weight.device)
    shape = (a.size(0), weight.size(0))
    return [torch.empty(shape, dtype=torch.float, device=a.device),
            torch.empty(shape, dtype=torch.int, device=a.device),
            torch.empty((4,) + shape, dtype=torch.float, device=a.device)]


@torch.library.register_fake(f"{library_name}::fullyconnected_wt_picks_backward")
def _(a, weight, grad, picks, sel, with_bias):
    torch._check(a.size(1) == weight.size(1))
    torch._check(grad.size(0) == a.size(0))
    torch._check(grad.size(1) == weight.size(0))
    torch._check(grad.shape == picks.shape)
    torch._check(picks.dtype == torch.int)
    grads = [torch.empty((a.size(0), a.size(1)), dtype=torch.float, device=a.device),
             torch.empty((weight.size(0), weight.size(1)), dtype=torch.float, device=a.device)]
    return grads + [torch.empty((weight.size(0),), dtype=torch.float, device=a.device)] if with_bias else grads


@torch.library.register_fake(f"{library_name}::fullyconnected_wt")
def _(a, weight, bias, hand_over):
    torch._check(a.dim() == 2 and weight.dim() == 2)
    torch._check(a.size(1) == weight.size(1))
    torch._check(a.dtype == torch.float)
    torch._check(weight.dtype == torch.float)
    torch._check(a.device == weight.device)
    shape = (a.size(0), weight.size(0))
    return [torch.empty(shape, dtype=torch.float, device=a.device),
            torch.empty(shape, dtype=torch.int, device=a.device),
            torch.empty(shape, dtype=torch.int, device=a.device),
            torch.empty((4 if hand_over else 0,) + shape, dtype=torch.float, device=a.device)]


@torch.library.register_fake(f"{library_name}::fullyconnected_wt_backward")
def _(a, weight, grad, argmax, argmin, sel):
    torch._check(a.size(1) == weight.size(1))
    torch._check(grad.size(0) == a.size(0))
    torch._check(grad.size(1) == weight.size(0))
    torch._check(grad.shape == argmax.shape)
    torch._check(grad.shape == argmin.shape)
    torch._check(argmax.dtype == torch.int)
    torch._check(argmin.dtype == torch.int)
    return [torch.empty((a.size(0), a.size(1)), dtype=torch.float, device=a.device),
            torch.empty((weight.size(0), weight.size(1)), dtype=torch.float, device=a.device)]


@torch.library.register_fake(f"{library_name}::fullyconnected_wt_backward_bias")
def _(a, weight, grad, argmax, argmin, sel):
    torch._check(a.size(1) == weight.size(1))
    torch._check(grad.size(0) == a.size(0))
    torch._check(grad.size(1) == weight.size(0))
    torch._check(grad.shape == argmax.shape)
    torch._check(grad.shape == argmin.shape)
    torch._check(argmax.dtype == torch.int)
    torch._check(argmin.dtype == torch.int)
    return [torch.empty((a.size(0), a.size(1)), dtype=torch.float, device=a.device),
            torch.empty((weight.size(0), weight.size(1)), dtype=torch.float, device=a.device),
            torch.empty((weight.size(0),), dtype=torch.float, device=a.device)]
