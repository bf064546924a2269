"""SwiGLU block for MI355X: fused-activation autograd function and the nn.Module.

Keeps the surface of the reference's megagemm/swiglu.py:86-172:
`MegaGemmFunction.apply(w12_out, hidden_dim)` maps [..., 2*hidden] = [gate | up] to
[..., hidden] = silu(gate) * up, and `MegaGemmTriton(d_model, multiple_of=256,
hidden_multiple=5/3)` owns `w12` (d_model -> 2*hidden) and `w3` (hidden -> d_model), both
bias-free nn.Linear layers.  In 16 bits the whole block runs on the package's own matrix products
(ops.swiglu_mlp; a decoding step of a few rows with nothing to differentiate in ops.swiglu_block);
calls those do not take go through the projections on torch.matmul and the activation.  The class
keeps its historical name for drop-in use; nothing here uses Triton -- products, activation and
backward are HIP kernels reached through mgrrmsnorm_amd.ops.
"""
from __future__ import annotations

import torch
import torch.nn as nn
import torch.nn.functional as F
from torch.nn.modules import linear as _linear, module as _module
from torch.autograd.function import once_differentiable

from . import ops


class MegaGemmFunction(torch.autograd.Function):
    """silu(gate) * up on a fused [..., 2*hidden_dim] tensor, reading both halves in place."""

    @staticmethod
    def forward(ctx, w12_out: torch.Tensor, hidden_dim: int):
        if w12_out.size(-1) != 2 * hidden_dim:
            raise RuntimeError(
                f"last dimension must be 2*hidden_dim = {2 * hidden_dim}, got {w12_out.size(-1)}")
        fused = w12_out.contiguous()
        ctx.save_for_backward(fused)
        ctx.hidden_dim = hidden_dim
        out = ops.swiglu_forward(fused.view(-1, 2 * hidden_dim), hidden_dim)
        return out.view(*fused.shape[:-1], hidden_dim)

    @staticmethod
    @once_differentiable
    def backward(ctx, grad_output: torch.Tensor):
        (fused,) = ctx.saved_tensors
        hidden_dim = ctx.hidden_dim
        dh = grad_output.contiguous().view(-1, hidden_dim)
        if dh.dtype != fused.dtype:
            dh = dh.to(fused.dtype)
        grad = ops.swiglu_backward(dh, fused.view(-1, 2 * hidden_dim), hidden_dim)
        return grad.view(fused.shape), None


def _defined_in(module, function):
    """`function` if it is `module`'s own, else None: replaced before this package was imported."""
    code = getattr(function, "__code__", None)
    return function if code is not None and code.co_filename == module.__file__ else None


# What a projection's call consists of, to notice when any part of it has been replaced.
_Linear = nn.Linear
_LINEAR_FORWARD = _defined_in(_linear, nn.Linear.forward)
_MODULE_CALL = _defined_in(_module, nn.Module.__call__)
_CALL_IMPL = _defined_in(_module, nn.Module._call_impl)
_SWIGLU = _defined_in(ops, ops.swiglu)
_SET_ON_AN_INSTANCE = frozenset(("forward", "weight", "bias", "_compiled_call_impl", "_call_impl", "_wrapped_call_impl"))


def _calls_replaced():
    """nn.Linear, the calling of modules, the linear operator or the activation is not the original:
    its replacement has to be called in a decoding step as everywhere else."""
    return (_Linear.forward is not _LINEAR_FORWARD or _Linear.__call__ is not _MODULE_CALL
            or _Linear._call_impl is not _CALL_IMPL or F.linear is not torch._C._nn.linear or ops.swiglu is not _SWIGLU)


def _plain_weight(linear):
    """The weight of a projection that is exactly `x @ weight.T`: a bias-free nn.Linear that nobody
    has hooked, replaced, parametrised, compiled or wrapped; else None."""
    if (type(linear) is not _Linear or linear._forward_hooks or linear._forward_pre_hooks or linear._backward_hooks
            or linear._backward_pre_hooks or not _SET_ON_AN_INSTANCE.isdisjoint(linear.__dict__)):
        return None
    parameters = linear._parameters
    weight = parameters.get("weight")
    return weight if type(weight) is nn.Parameter and parameters.get("bias") is None else None


def _calls_observed():
    """Something wants to see the projections as torch operations: a trace, autocast, a dispatch or function
    mode, or a global module hook."""
    return (torch.jit.is_tracing() or torch.is_autocast_enabled()
            or torch._C._len_torch_dispatch_stack() > 0 or torch._C._len_torch_function_stack() > 0
            or _module._global_forward_hooks or _module._global_forward_pre_hooks or _module._global_backward_hooks
            or _module._global_backward_pre_hooks)


class MegaGemmTriton(nn.Module):
    """SwiGLU feed-forward block: w3(silu(w1 x) * (w2 x)) with w1 and w2 fused into w12.

    Args:
        d_model: input and output width.
        multiple_of: the hidden width is rounded up to a multiple of this (default 256).
        hidden_multiple: expansion factor before rounding (default 5/3).

    Rows [0, hidden) of `w12.weight` are the gate projection and rows [hidden, 2*hidden)
    the up projection, as in the reference (benchmark_swiglu.py:87-88).
    """

    def __init__(self, d_model: int, multiple_of: int = 256, hidden_multiple: float = 5 / 3):
        super().__init__()
        raw = int(d_model * hidden_multiple)
        self.hidden = multiple_of * ((raw + multiple_of - 1) // multiple_of)
        self.w12 = nn.Linear(d_model, 2 * self.hidden, bias=False)
        self.w3 = nn.Linear(self.hidden, d_model, bias=False)

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        # The whole block at once, while the projections are the plain ones this module made: a decoding step in
        # two kernels that read the weights once, everything else on the package's own matrix products.  The compiler is
        # asked about first, because it cannot trace the other questions; then the size, which other calls end at.
        if not torch.compiler.is_compiling() and type(x) is torch.Tensor:
            decoding = ops.swiglu_block_fits(x, self.hidden)
            if ((decoding or ops.swiglu_mlp_fits(x, self.hidden)) and not _calls_observed() and not _calls_replaced()):
                w12, w3 = _plain_weight(self.w12), _plain_weight(self.w3)
                if w12 is not None and w3 is not None and w3.dim() == 2 and w3.size(1) == self.hidden:
                    out = ops.swiglu_block(x, w12, w3) if decoding else None
                    if out is None:
                        out = ops.swiglu_mlp(x, w12, w3)
                    if out is not None:
                        return out
        # the activation's autograd node lives in the compiled extension when that is built
        # (else MegaGemmFunction); with nothing to differentiate it is the bare kernel
        return self.w3(ops.swiglu(self.w12(x), self.hidden))

    def extra_repr(self) -> str:
        return f"d_model={self.w12.in_features}, hidden={self.hidden} (Triton Accelerated)"
