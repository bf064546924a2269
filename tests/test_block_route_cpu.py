"""Which calls MegaGemmTriton may hand to the decoding step's kernels as a whole: only those whose
projections are what this package made of them.  Everything that looks at, replaces or wraps a
projection has to be reached in a decoding step too.  The kernels themselves are stubbed here."""
import pytest
import torch
import torch.nn as nn
import torch.nn.functional as F

from mgrrmsnorm_amd import MegaGemmTriton, ops


@pytest.fixture
def handed_over(monkeypatch):
    """Calls the module and returns the (w12, w3) it handed to ops.swiglu_block, or None if it went
    through the projections."""
    calls = []
    monkeypatch.setattr(ops, "swiglu_block_fits", lambda x, hidden: True, raising=False)
    monkeypatch.setattr(ops, "swiglu_block", lambda x, w12, w3: calls.append((w12, w3)))

    def call(module, x=None):
        calls.clear()
        try:
            with torch.no_grad():
                module(torch.zeros(2, 16) if x is None else x)
        except RuntimeError:       # past the hand-over: no GPU, or a stand-in of another shape
            pass
        return calls[0] if calls else None
    return call


def _module():
    return MegaGemmTriton(16, multiple_of=8)


def test_a_module_as_made_is_handed_over_with_its_weights(handed_over):
    m = _module()
    w12, w3 = handed_over(m)
    assert w12 is m.w12.weight and w3 is m.w3.weight


class _Sub(nn.Linear):
    pass


def _shadow(name, value):
    return lambda m: m.w3.__dict__.__setitem__(name, value)


CHANGES = {
    "forward hook": lambda m: m.w12.register_forward_hook(lambda *a: None),
    "forward pre-hook": lambda m: m.w3.register_forward_pre_hook(lambda *a: None),
    "full backward hook": lambda m: m.w12.register_full_backward_hook(lambda *a: None),
    "forward of the instance": lambda m: setattr(m.w12, "forward", lambda x: x),
    "weight set over the parameter": _shadow("weight", torch.ones(16, 32)),
    "bias set over the parameter": _shadow("bias", torch.ones(16)),
    "compiled projection": lambda m: m.w12.compile(backend="eager"),
    "another kind of projection": lambda m: setattr(m, "w12", _Sub(16, 2 * m.hidden, bias=False)),
    "a projection with bias": lambda m: setattr(m, "w3", nn.Linear(m.hidden, 16)),
    "parametrised weight": lambda m: nn.utils.parametrize.register_parametrization(m.w3, "weight", nn.Identity()),
    "wrapped projection": lambda m: setattr(m, "w12", nn.Sequential(m.w12)),
}


@pytest.mark.parametrize("change", CHANGES)
def test_a_changed_projection_is_called(handed_over, change):
    m = _module()
    assert handed_over(m) is not None
    CHANGES[change](m)
    assert handed_over(m) is None


REPLACED = {
    "nn.Linear.forward": (nn.Linear, "forward", lambda self, x: x),
    "nn.Linear.__call__": (nn.Linear, "__call__", lambda self, x: nn.Module.__call__(self, x)),
    "functional.linear": (F, "linear", lambda x, w, b=None: x @ w.t()),
    "the activation": (ops, "swiglu", lambda x, hidden: x[..., :hidden]),
}


@pytest.mark.parametrize("what", REPLACED)
def test_a_replaced_function_is_called(handed_over, monkeypatch, what):
    m = _module()
    owner, name, value = REPLACED[what]
    monkeypatch.setattr(owner, name, value)
    assert handed_over(m) is None


def test_modes_and_global_hooks_see_the_projections(handed_over):
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    class Functions(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    m = _module()
    for mode in (Functions(), Dispatch()):
        with mode:
            assert handed_over(m, torch.zeros(2, 16)) is None
    for register in (nn.modules.module.register_module_forward_hook, nn.modules.module.register_module_forward_pre_hook):
        handle = register(lambda *a: None)
        try:
            assert handed_over(m) is None
        finally:
            handle.remove()
    assert handed_over(m) is not None


def test_projections_are_taken_through_their_attributes(handed_over):
    m = _module()
    other = nn.Linear(16, 2 * m.hidden, bias=False)
    m.__dict__["w12"] = other                           # set over the registered module
    assert handed_over(m)[0] is other.weight

    class Tied(MegaGemmTriton):
        def __getattr__(self, name):
            return other if name == "w12" else super().__getattr__(name)

    assert handed_over(Tied(16, multiple_of=8))[0] is not None
    tied = Tied(16, multiple_of=8)
    del tied._modules["w12"]
    assert handed_over(tied)[0] is other.weight


def test_parameters_swapped_for_one_call(handed_over):
    m = _module()
    values = {name: p.detach() * 2 for name, p in m.named_parameters()}
    seen = handed_over(lambda x: torch.func.functional_call(m, values, (x,)))
    assert seen is None


def test_the_block_compiles_as_one_graph(monkeypatch):
    """With an activation that can be traced, the module is one graph: the question whether a
    compiler is looking comes before anything that the compiler itself cannot trace."""
    monkeypatch.setattr(ops, "swiglu", lambda x, hidden: F.silu(x[..., :hidden]) * x[..., hidden:])
    m = _module()
    x = torch.randn(2, 16)
    torch._dynamo.reset()
    with torch.no_grad():
        compiled = torch.compile(m, backend="eager", fullgraph=True)
        assert torch.equal(compiled(x), m(x))


def test_calls_of_other_sizes_end_at_the_size(monkeypatch):
    """A call that is not for the two kernels is not held up by questions about modes and projections."""
    from mgrrmsnorm_amd import swiglu

    asked = []
    monkeypatch.setattr(swiglu, "_calls_observed", lambda: asked.append(1))
    with pytest.raises(RuntimeError):           # a tensor of the CPU
        _module()(torch.zeros(65, 16))
    assert not asked


def test_a_trace_records_the_projections(handed_over):
    m = _module()
    assert handed_over(lambda x: torch.jit.trace(m, x, check_trace=False)) is None
    assert handed_over(m) is not None
