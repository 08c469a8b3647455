"""Fake (meta) kernels shared by the operator namespaces (mamtorch/kernel/v4/fullyconnected.py:12-28,
mamtorch/kernel/v1/fullyconnected.py:12-28).  The autograd formulas are registered in csrc/torch_autograd.cpp.
"""
import torch


def _check_forward(a, b):
    torch._check(a.dim() == 2 and b.dim() == 2)
    torch._check(a.size(1) == b.size(0))
    torch._check(a.dtype == torch.float)
    torch._check(b.dtype == torch.float)
    torch._check(a.device == b.device)


def register_exact_forward(ns):
    """ns::fullyconnected(a, b) -> [C, argmax, argmin] and ns::fullyconnected_backward."""
    @torch.library.register_fake(f"{ns}::fullyconnected")
    def _(a, b):
        _check_forward(a, b)
        shape = (a.size(0), b.size(1))
        return [torch.empty(shape, dtype=torch.float, device=a.device),
                torch.empty(shape, dtype=torch.int, device=a.device),
                torch.empty(shape, dtype=torch.int, device=a.device)]

    @torch.library.register_fake(f"{ns}::fullyconnected_backward")
    def _(a, b, grad, argmax, argmin):
        _check_forward(a, b)
        torch._check(grad.size(0) == a.size(0))
        torch._check(grad.size(1) == b.size(1))
        torch._check(grad.shape == argmax.shape)
        torch._check(grad.shape == argmin.shape)
        torch._check(grad.dtype == torch.float)
        torch._check(argmax.dtype == torch.int)
        torch._check(argmin.dtype == torch.int)
        torch._check(argmax.is_contiguous())
        torch._check(argmin.is_contiguous())
        return [torch.empty((a.size(0), a.size(1)), dtype=torch.float, device=a.device),
                torch.empty((b.size(0), b.size(1)), dtype=torch.float, device=a.device)]
