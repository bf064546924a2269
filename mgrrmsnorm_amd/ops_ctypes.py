"""Tensor-level operators on top of the C ABI, bound with ctypes: checks, output allocation,
launch.  This is the binding that needs no C++ compiler; `mgrrmsnorm_amd.ops` prefers the
compiled extension (csrc/torch_binding.cpp) over the same C ABI when it has been built and
falls back to this module otherwise.  Both call the same library: there is one kernel path.

`rmsnorm_forward` / `rmsnorm_backward` keep the call signatures and return values of the
reference's extension module (pytorch_binding/binding.cpp:16,73-78,136-139):

    rmsnorm_forward(input[R,C], weight[C], epsilon) -> [output, inv_rms(fp32,[R])]
    rmsnorm_backward(grad_output, input, weight, inv_rms) -> [grad_input, grad_weight]

`swiglu_forward` / `swiglu_backward` are the tensor-level form of the two Triton launches
(megagemm/swiglu.py:89-131).  All four run on torch's current stream of the tensors'
device and never synchronise.
"""
from __future__ import annotations

import ctypes

import torch
from torch.autograd.function import once_differentiable

from . import _lib


def _require_gpu(t: torch.Tensor, name: str) -> None:
    # binding.cpp:9 CHECK_CUDA
    if not t.is_cuda:
        raise RuntimeError(f"{name} must be a CUDA tensor")


def _require_contiguous(t: torch.Tensor, name: str) -> None:
    # binding.cpp:10 CHECK_CONTIGUOUS
    if not t.is_contiguous():
        raise RuntimeError(f"{name} must be contiguous")


def _check_pair(input: torch.Tensor, weight: torch.Tensor) -> None:
    if input.dim() != 2:
        raise RuntimeError("Input must be 2D")
    if weight.dim() != 1 or weight.size(0) != input.size(1):
        raise RuntimeError("Weight size must match hidden size")
    if weight.dtype != input.dtype:
        raise RuntimeError(
            f"weight dtype ({weight.dtype}) must equal input dtype ({input.dtype}); "
            "cast the module, e.g. model.half() or model.to(torch.bfloat16)")
    if weight.device != input.device:
        raise RuntimeError("input and weight must be on the same device")


def rmsnorm_forward(input: torch.Tensor, weight: torch.Tensor, epsilon: float):
    """y = x * rsqrt(mean(x^2) + eps) * w.  Returns [output, inv_rms]."""
    return _rmsnorm_forward(input, weight, epsilon, True)


def rmsnorm_output(input: torch.Tensor, weight: torch.Tensor, epsilon: float):
    """The output of rmsnorm_forward alone, where no backward pass follows."""
    return _rmsnorm_forward(input, weight, epsilon, False)[0]


def _rmsnorm_forward(input, weight, epsilon, backward_follows):
    if not (input.is_cuda and weight.is_cuda and input.is_contiguous() and weight.is_contiguous()):
        for t, n in ((input, "input"), (weight, "weight")):
            _require_gpu(t, n)
            _require_contiguous(t, n)
    if input.dim() != 2 or weight.dim() != 1 or weight.size(0) != input.size(1) \
            or weight.dtype != input.dtype or weight.device != input.device:
        _check_pair(input, weight)
    code = _lib.dtype_code(input.dtype)
    rows, cols = input.shape
    if cols < 1:
        raise RuntimeError("hidden size must be >= 1")
    lib = _lib.load()
    dev = input.device
    with _lib.device_of(dev):
        output = torch.empty_like(input)
        inv_rms = torch.empty((rows,), dtype=torch.float32, device=dev) if backward_follows else None
        rc = lib.mg_rmsnorm_fwd(output.data_ptr(), None if inv_rms is None else inv_rms.data_ptr(), input.data_ptr(),
                                weight.data_ptr(), rows, cols, epsilon, code, _lib.stream_ptr(dev))
    if rc != 0:
        _lib.check(rc, "RMSNorm forward")
    return [output, inv_rms]


# (device index, rows, cols, dtype code) -> (num_partials, ld); the answer depends on nothing else
# but the tuning options, so the table is dropped whenever the library's count of option changes
# has moved (through _lib.set_option or a direct mg_set_option alike)
_workspace_shapes: dict = {}
_workspace_generation = -1


def _bwd_workspace(lib, dev, rows, cols, code):
    global _workspace_generation
    generation = lib.mg_option_generation()
    if generation != _workspace_generation:
        _workspace_shapes.clear()
        _workspace_generation = generation
    key = (dev.index, rows, cols, code)
    hit = _workspace_shapes.get(key)
    if hit is None:
        n_part, ld = ctypes.c_int64(0), ctypes.c_int64(0)
        _lib.check(lib.mg_rmsnorm_bwd_workspace(rows, cols, code, ctypes.byref(n_part), ctypes.byref(ld)),
                   "RMSNorm backward (workspace query)")
        hit = (n_part.value, ld.value)
        if len(_workspace_shapes) < 4096:
            _workspace_shapes[key] = hit
    return hit


def rmsnorm_backward_f32(grad_output: torch.Tensor, input: torch.Tensor, weight: torch.Tensor,
                         inv_rms: torch.Tensor, need_weight_grad: bool = True):
    """Backward with dW kept in fp32: returns (grad_input, grad_weight_f32, grad_weight_cast)
    where grad_weight_cast has the weight's dtype (it is grad_weight_f32 itself for fp32).
    With need_weight_grad=False the dW reduction is not launched and both are None."""
    if not (grad_output.is_cuda and input.is_cuda and weight.is_cuda and inv_rms.is_cuda
            and grad_output.is_contiguous() and input.is_contiguous() and weight.is_contiguous()
            and inv_rms.is_contiguous()):
        for t, n in ((grad_output, "grad_output"), (input, "input"), (weight, "weight"), (inv_rms, "inv_rms")):
            _require_gpu(t, n)
            _require_contiguous(t, n)
    if input.dim() != 2 or weight.dim() != 1 or weight.size(0) != input.size(1) \
            or weight.dtype != input.dtype or weight.device != input.device:
        _check_pair(input, weight)
    if grad_output.shape != input.shape or grad_output.dtype != input.dtype:
        raise RuntimeError("grad_output must have the shape and dtype of input")
    if inv_rms.dtype != torch.float32 or inv_rms.dim() != 1 or inv_rms.size(0) != input.size(0):
        raise RuntimeError("inv_rms must be a float32 vector with one entry per row")
    code = _lib.dtype_code(input.dtype)
    rows, cols = input.shape
    lib = _lib.load()
    dev = input.device
    with _lib.device_of(dev):
        stream = _lib.stream_ptr(dev)
        grad_input = torch.empty_like(input)
        dw_f32 = dw_cast = None
        if need_weight_grad:
            dw_f32 = torch.empty((cols,), dtype=torch.float32, device=dev)
            dw_cast = dw_f32 if code == _lib.MG_F32 else torch.empty_like(weight)
        if lib.mg_rmsnorm_bwd_small_fits(rows, cols, code):    # few rows: one launch, no workspace
            rc = lib.mg_rmsnorm_bwd_small(grad_input.data_ptr(), None if dw_f32 is None else dw_f32.data_ptr(),
                                          None if dw_cast is dw_f32 else dw_cast.data_ptr(), grad_output.data_ptr(),
                                          input.data_ptr(), weight.data_ptr(), inv_rms.data_ptr(), rows, cols, code, stream)
            if rc != 0:
                _lib.check(rc, "RMSNorm backward")
            return grad_input, dw_f32, dw_cast
        n_part, ld = _bwd_workspace(lib, dev, rows, cols, code)
        partial = torch.empty((n_part, ld), dtype=torch.float32, device=dev)
        rc = lib.mg_rmsnorm_bwd(grad_input.data_ptr(), partial.data_ptr(), grad_output.data_ptr(),
                                input.data_ptr(), weight.data_ptr(), inv_rms.data_ptr(), rows, cols, code,
                                n_part, ld, stream)
        if rc != 0:
            _lib.check(rc, "RMSNorm backward")
        if need_weight_grad:
            rc = lib.mg_rmsnorm_dw_reduce(dw_f32.data_ptr(), None if dw_cast is dw_f32 else dw_cast.data_ptr(),
                                          code, partial.data_ptr(), n_part, ld, cols, stream)
            if rc != 0:
                _lib.check(rc, "RMSNorm backward (dW reduction)")
    return grad_input, dw_f32, dw_cast


def rmsnorm_backward(grad_output: torch.Tensor, input: torch.Tensor, weight: torch.Tensor,
                     inv_rms: torch.Tensor):
    """Returns [grad_input, grad_weight]; grad_weight has the weight's dtype
    (binding.cpp:90), rounded once from the fp32 column sums."""
    grad_input, _, dw_cast = rmsnorm_backward_f32(grad_output, input, weight, inv_rms)
    return [grad_input, dw_cast]


def swiglu_forward(gate_up: torch.Tensor, hidden_dim: int) -> torch.Tensor:
    """gate_up: [M, 2*hidden_dim] = [gate | up] per row -> [M, hidden_dim]."""
    return _swiglu_forward(gate_up, hidden_dim, True)


def swiglu_output(gate_up: torch.Tensor, hidden_dim: int) -> torch.Tensor:
    """swiglu_forward where no backward pass follows."""
    return _swiglu_forward(gate_up, hidden_dim, False)


def _swiglu_forward(gate_up, hidden_dim, backward_follows):
    _require_gpu(gate_up, "w12_out")
    _require_contiguous(gate_up, "w12_out")
    if gate_up.dim() != 2 or gate_up.size(1) != 2 * hidden_dim:
        raise RuntimeError(f"expected a [M, {2 * hidden_dim}] matrix, got {tuple(gate_up.shape)}")
    code = _lib.dtype_code(gate_up.dtype)
    M = gate_up.size(0)
    lib = _lib.load()
    with _lib.device_of(gate_up.device):
        out = torch.empty((M, hidden_dim), dtype=gate_up.dtype, device=gate_up.device)
        forward = lib.mg_swiglu_fwd if backward_follows else lib.mg_swiglu_fwd_only
        rc = forward(out.data_ptr(), gate_up.data_ptr(), M, hidden_dim, code, _lib.stream_ptr(gate_up.device))
    _lib.check(rc, "SwiGLU forward")
    return out


def swiglu_backward(grad_out: torch.Tensor, gate_up: torch.Tensor, hidden_dim: int) -> torch.Tensor:
    """grad_out: [M, hidden_dim], gate_up: [M, 2*hidden_dim] -> [M, 2*hidden_dim] = [d_gate | d_up]."""
    for t, n in ((grad_out, "grad_output"), (gate_up, "w12_out")):
        _require_gpu(t, n)
        _require_contiguous(t, n)
    if gate_up.dim() != 2 or gate_up.size(1) != 2 * hidden_dim:
        raise RuntimeError(f"expected a [M, {2 * hidden_dim}] matrix, got {tuple(gate_up.shape)}")
    if grad_out.shape != (gate_up.size(0), hidden_dim) or grad_out.dtype != gate_up.dtype:
        raise RuntimeError("grad_output must be [M, hidden_dim] with the dtype of the forward input")
    code = _lib.dtype_code(gate_up.dtype)
    M = gate_up.size(0)
    lib = _lib.load()
    with _lib.device_of(gate_up.device):
        grad_in = torch.empty_like(gate_up)
        rc = lib.mg_swiglu_bwd(grad_in.data_ptr(), grad_out.data_ptr(), gate_up.data_ptr(), M, hidden_dim, code,
                               _lib.stream_ptr(gate_up.device))
    _lib.check(rc, "SwiGLU backward")
    return grad_in


# ---- the whole SwiGLU block on the library's own products (megagemm_hip_mlp.h) ----

_MLP_CODES = {torch.float16: 1, torch.bfloat16: 2}


_MLP_ALL, _MLP_FORWARD_ONLY, _MLP_X_LEARNS = range(3)


def _preferred(x, hidden, call):
    d_model = x.size(-1)
    return _lib.load().mg_mlp_preferred(x.numel() // d_model, d_model, hidden, _MLP_CODES[x.dtype], call) == 1


def swiglu_mlp_fits(x: torch.Tensor, hidden_dim: int) -> bool:
    if x.dtype not in _MLP_CODES or not x.is_cuda or x.dim() < 1 or x.size(-1) < 1:
        return False
    return _preferred(x, hidden_dim, _MLP_ALL if torch.is_grad_enabled() else _MLP_FORWARD_ONLY)


def _plain_dense(t: torch.Tensor) -> bool:
    """A dense tensor of a GPU that nothing else wants to see the operations of."""
    return (type(t) in (torch.Tensor, torch.nn.Parameter) and t.layout is torch.strided and t.is_cuda and not t.is_nested
            and not t.is_conj() and not t.is_neg() and not t._is_zerotensor()
            and not torch._C._functorch.is_functorch_wrapped_tensor(t)
            and torch.autograd.forward_ad.unpack_dual(t).tangent is None)


def _plain_backward(grad) -> bool:
    """Whether a backward pass is for the kernels: one gradient, of which the same holds as of the operands (a batch of
    them is no such tensor), and no dispatch mode that looks on."""
    return (grad is not None and _plain_dense(grad) and not torch._C._functorch.is_legacy_batchedtensor(grad)
            and torch._C._len_torch_dispatch_stack() == 0)


def _pointer(t) -> int | None:
    return None if t is None else t.data_ptr()


def _mlp_workspace(x, tokens, d_model, hidden, wanted):
    """(tensor or None, its bytes) that a pass needs besides its tensors; wanted: nothing for the forward pass,
    else the gradients of x, w12 and w3 that are."""
    need = ctypes.c_int64(0)
    mask = sum(1 << i for i, w in enumerate(wanted) if w)
    _lib.check(_lib.load().mg_mlp_workspace(tokens, d_model, hidden, _MLP_CODES[x.dtype], mask, ctypes.byref(need)),
               "SwiGLU block (workspace query)")
    return (torch.empty(need.value, dtype=torch.uint8, device=x.device) if need.value else None), need.value


def _mlp_forward(x, w12, w3, keep_gate_up):
    d_model, hidden = w3.shape
    tokens = x.numel() // d_model
    with _lib.device_of(x.device):
        gate_up = x.new_empty(tokens, 2 * hidden) if keep_gate_up else None
        h = x.new_empty(*x.shape[:-1], hidden)
        out = torch.empty_like(x)
        work, size = _mlp_workspace(x, tokens, d_model, hidden, ())
        rc = _lib.load().mg_mlp_fwd(out.data_ptr(), h.data_ptr(), _pointer(gate_up), x.data_ptr(), w12.data_ptr(), w3.data_ptr(),
                                    _pointer(work), size, tokens, d_model, hidden, _MLP_CODES[x.dtype], _lib.stream_ptr(x.device))
    _lib.check(rc, "SwiGLU block forward")
    return out, gate_up, h


class _MlpFunction(torch.autograd.Function):
    """(out, h or None): h is an output where w3 learns, as a graph recorded over the gradient of w3 gets through it to x and
    w12.  What linear layers keep is kept: x (contiguous here) for the gradient of w12, w12 for that of x, w3, h for that of w3."""

    @staticmethod
    def forward(ctx, x, w12, w3):
        for_x, for_12, for_3 = ctx.needs_input_grad
        # aliases, for the kernels: they keep the data they were made of when a caller gives an operand other data before
        # the backward pass; the operands themselves are for one that records its own graph
        xd, ad, bd = x.detach(), w12.detach(), w3.detach()
        out, gate_up, h = _mlp_forward(xd, ad, bd, True)
        if not for_3:
            h = None
        ctx.save_for_backward(xd if for_12 else None, ad if for_x else None, bd, gate_up, h,
                              x if for_12 else None, w12 if for_x else None, w3)
        ctx.set_materialize_grads(False)
        return out, h

    @staticmethod
    def backward(ctx, grad_output, grad_h):
        saved, want, records = ctx.saved_tensors, ctx.needs_input_grad, torch.is_grad_enabled()
        if not records and grad_h is None and _plain_backward(grad_output):
            return _mlp_backward(grad_output, want, *saved[:5])
        want = [w and _asked_for(node) for w, (node, _) in zip(want, ctx.next_functions)]
        return _mlp_backward_in_operations(grad_output, grad_h, want, *(saved[5:] if records else saved[:3]), *saved[3:5])


def _mlp_backward(grad_output, want, x, w12, w3, gate_up, h):
    d_model, hidden = w3.shape
    tokens = gate_up.size(0)
    dy = grad_output.contiguous().to(gate_up.dtype)
    if dy.data_ptr() % 16 != 0:
        dy = dy.clone()
    with _lib.device_of(dy.device):
        shapes = (dy.shape, (2 * hidden, d_model), (d_model, hidden))
        grads = [dy.new_empty(s) if w else None for s, w in zip(shapes, want)]
        d_gate_up = torch.empty_like(gate_up) if want[0] or want[1] else None
        work, size = _mlp_workspace(dy, tokens, d_model, hidden, want[:3])
        rc = _lib.load().mg_mlp_bwd(*map(_pointer, grads), _pointer(d_gate_up), dy.data_ptr(), _pointer(x), _pointer(w12), w3.data_ptr(),
                                    gate_up.data_ptr(), _pointer(h), _pointer(work), size, tokens, d_model, hidden, _MLP_CODES[dy.dtype],
                                    _lib.stream_ptr(dy.device))
    _lib.check(rc, "SwiGLU block backward")
    return tuple(grads)


def _asked_for(node) -> bool:
    """Whether the backward pass under way goes on to `node`: with w3 alone asked for, the activation is not to be reached, which
    does not take every gradient that a product takes."""
    try:
        return torch._C._will_engine_execute_node(node)
    except RuntimeError:      # a leaf whose gradient torch.autograd.grad returns
        return True


@once_differentiable
def _activation_backward(gate_up, dh):
    return swiglu_backward(dh.to(gate_up.dtype).contiguous(), gate_up, dh.size(1)), None


def _mlp_backward_in_operations(grad_output, dh, want, x, w12, w3, gate_up, h):
    """What the projections' and the activation's backward passes do, as operations that record a graph where one is
    wanted, take the gradients those take and refuse what those refuse."""
    d_model, hidden = w3.shape
    out = [None, None, None]
    if grad_output is None and dh is None:
        return tuple(out)
    lead = (grad_output if dh is None else dh).shape[:-1]
    if dh is not None:
        dh = dh.reshape(-1, hidden)
    if grad_output is not None:
        dy = grad_output.to(gate_up.dtype).reshape(-1, d_model)
        if want[2]:
            out[2] = dy.t().mm(h.reshape(-1, hidden))
        if want[0] or want[1]:
            dh = dy.mm(w3) if dh is None else dh + dy.mm(w3)
    if dh is None or not (want[0] or want[1]):
        return tuple(out)
    d_gate_up, _ = _activation_backward(gate_up, dh)
    if want[0]:
        out[0] = d_gate_up.mm(w12).reshape(*lead, d_model)
    if want[1]:
        out[1] = d_gate_up.t().mm(x.reshape(-1, d_model))
    return tuple(out)


def swiglu_mlp(x: torch.Tensor, w12: torch.Tensor, w3: torch.Tensor):
    """ops.swiglu_mlp; the same calls are taken as in csrc/torch_binding.cpp."""
    if x.dtype not in _MLP_CODES or x.dim() < 1 or w12.dim() != 2 or w3.dim() != 2 or not all(map(_plain_dense, (x, w12, w3))):
        return None
    if torch._C._autograd._top_saved_tensors_default_hooks(False) is not None or torch._C._functorch.peek_interpreter_stack() is not None:
        return None
    d_model, hidden = w3.shape
    if d_model < 1 or x.size(-1) != d_model or w12.shape != (2 * hidden, d_model):
        return None
    if any(w.dtype != x.dtype or w.device != x.device or not w.is_contiguous() or w.data_ptr() % 16 != 0 for w in (w12, w3)):
        return None
    weights_learn = w12.requires_grad or w3.requires_grad
    learns = torch.is_grad_enabled() and (x.requires_grad or weights_learn)
    call = _MLP_FORWARD_ONLY if not learns else _MLP_ALL if weights_learn else _MLP_X_LEARNS
    if not _preferred(x, hidden, call) or (x.is_contiguous() and x.data_ptr() % 16 != 0):
        return None
    if learns:
        return _MlpFunction.apply(x.contiguous(), w12, w3)[0] if x.requires_grad or w12.requires_grad else None
    return _mlp_forward(x.contiguous(), w12, w3, False)[0]
