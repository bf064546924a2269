"""The SwiGLU block on the package's own matrix products (megagemm_hip_mlp.h): every output against the same
formula in float64 at the edges of the tiles, and what the module does around it."""
import ctypes

import pytest
import torch

import gpu_util as U
from mgrrmsnorm_amd import MegaGemmTriton, ops
from test_block_gpu import _case, _within

pytestmark = pytest.mark.gpu

# largest relative error of rounding to p significant bits, 2^-p: bf16 has 8 of them, fp16 11
ROUNDING = {"bf16": 2.0 ** -8, "fp16": 2.0 ** -11}


def _call(name, tensors, sizes, dtype):
    need = ctypes.c_int64(0)
    wanted = sum(1 << i for i, t in enumerate(tensors[:3]) if t is not None) if name == "mg_mlp_bwd" else 0
    U.check(U.lib().mg_mlp_workspace(*sizes, U.CODES[dtype], wanted, ctypes.byref(need)))
    size = need.value
    work = torch.full((size + 1024,), 0xFF, device="cuda", dtype=torch.uint8)       # NaN where nothing is written
    U.check(getattr(U.lib(), name)(*[t if t is None else t.data_ptr() for t in tensors], work.data_ptr() if size else None, size,
                                   *sizes, U.CODES[dtype], U.stream()))
    assert (work[size:] == 0xFF).all()


def _guarded(shape, dtype):
    """An output between two canaries."""
    n = shape[0] * shape[1]
    flat = torch.full((n + 512,), 7.0, device="cuda", dtype=dtype)
    return flat[256:256 + n].view(shape), flat


def _intact(*flats):
    for f in flats:
        assert (f[:256] == 7).all() and (f[-256:] == 7).all()


def _bounded(got, ref, terms, count, dtype, extra=0.0):
    """One rounding of the result and an fp32 sum of `count` products whose absolute values add up to `terms`."""
    u, tiny = ROUNDING[dtype], 2.0 ** -25 if dtype == "fp16" else 0.0
    bound = ((count + 8) * 2.0 ** -24 * terms + extra) * (1 + u) + u * ref.abs() + tiny
    worst = ((got.double() - ref).abs() - bound).max().item()
    assert worst <= 0.0, f"beyond the error bound by {worst}"


# every product on every tile, k whole and in parts: tests/test_mlp_cpu.py asks the planner
SIZES = [
    (1, 64, 64), (17, 1024, 1792), (64, 2048, 5504), (65, 64, 192), (127, 192, 64), (128, 128, 128), (129, 128, 256), (257, 320, 448), (300, 704, 1088),
    (1000, 512, 1344), (1024, 2048, 3584), (513, 1536, 4096), (2047, 1024, 2816), (96, 4096, 6912), (640, 3136, 8384),
    (127, 1024, 11008), (130, 3136, 8000), (70, 8192, 1088), (200, 704, 2752),   # k in 2 to 8 parts, of 43.5 and 9.5 steps
    (2048, 512, 512), (4099, 512, 1024), (4096, 2048, 3584), (10601, 64, 4416),  # weight gradients in parts, k ragged in two of them
    (603, 3456, 9216), (1322, 3200, 5376), (1499, 2944, 5120), (18342, 6592, 192),   # second projection and gradient of x on the large tiles
]


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("tokens,d_model,hidden", SIZES)
def test_products_against_float64(tokens, d_model, hidden, dtype):
    x, w12, w3 = _case(tokens, d_model, hidden, dtype)
    dy = torch.randn(tokens, d_model, device="cuda", generator=torch.Generator("cuda").manual_seed(5)).to(x.dtype)
    sizes, dt = (tokens, d_model, hidden), x.dtype

    def run():
        (out, c0), (h, c1), (gu, c2) = (_guarded(s, dt) for s in ((tokens, d_model), (tokens, hidden), (tokens, 2 * hidden)))
        _call("mg_mlp_fwd", (out, h, gu, x, w12, w3), sizes, dtype)
        (dx, c3), (da, c4), (db, c5), (dgu, c6) = (_guarded(s, dt) for s in (
            (tokens, d_model), (2 * hidden, d_model), (d_model, hidden), (tokens, 2 * hidden)))
        _call("mg_mlp_bwd", (dx, da, db, dgu, dy, x, w12, w3, gu, h), sizes, dtype)
        _intact(c0, c1, c2, c3, c4, c5, c6)
        return out, h, gu, dx, da, db, dgu

    out, h, gu, dx, da, db, dgu = first = run()
    assert all(torch.equal(a, b) for a, b in zip(first, run()))          # fixed summation order
    _within(out, x, w12, w3, dtype)
    xd, ad, bd, yd, hd, gd = (t.double() for t in (x, w12, w3, dy, h, gu))
    _bounded(gu, xd @ ad.t(), xd.abs() @ ad.abs().t(), d_model, dtype)
    _bounded(out, hd @ bd.t(), hd.abs() @ bd.abs().t(), hidden, dtype)
    _bounded(db, yd.t() @ hd, yd.abs().t() @ hd.abs(), tokens, dtype)
    # the activation's backward from the stored gate and up, and the error of the sum it starts from
    gate, up = gd.chunk(2, -1)
    dh, terms = yd @ bd, yd.abs() @ bd.abs()
    s = torch.sigmoid(gate)
    slope = s * (1 + gate * (1 - s))
    wiggle = 24 * 2.0 ** -24 * dh.abs()                                  # of the activation's own arithmetic
    parts = (1 + gate.abs()) * s
    for got, factor, size in ((dgu[:, :hidden], up * slope, up.abs() * parts), (dgu[:, hidden:], gate * s, gate.abs() * s)):
        _bounded(got, dh * factor, terms * size, d_model, dtype, wiggle * size)
    dd = dgu.double()
    _bounded(dx, dd @ ad, dd.abs() @ ad.abs(), 2 * hidden, dtype)
    _bounded(da, dd.t() @ xd, dd.abs().t() @ xd.abs(), tokens, dtype)
    # each gradient alone, and no [gate | up] kept
    again = torch.empty_like(out)
    _call("mg_mlp_fwd", (again, torch.empty_like(h), None, x, w12, w3), sizes, dtype)
    assert torch.equal(again, out)
    work = torch.empty_like(dgu)
    for i, (want, a, b, count) in enumerate(((dx, dd, ad, 2 * hidden), (da, dd.t(), xd, tokens), (db, yd.t(), hd, tokens))):
        alone = [None, None, None]                       # in a launch to itself the sums may go another way
        alone[i] = torch.empty_like(want)
        _call("mg_mlp_bwd", (*alone, None if i == 2 else work, dy, x, w12, w3, gu, h), sizes, dtype)
        dw = work.double() if i < 2 else None
        a = (dw if i == 0 else dw.t()) if i < 2 else a
        _bounded(alone[i], a @ b, a.abs() @ b.abs(), count, dtype)


@pytest.mark.parametrize("tokens,d_model,hidden", [(1198371, 64, 448), (5, 65536, 8128)])
def test_tensors_just_below_2_gib(tokens, d_model, hidden):
    """On whole numbers, whose sums are exact: every result is the one in float64 rounded once."""
    dt, sizes, g = torch.bfloat16, (tokens, d_model, hidden), torch.Generator("cuda").manual_seed(0)
    ints = lambda *s: torch.randint(-1, 2, s, device="cuda", generator=g, dtype=torch.int8).to(dt)
    x, w12, w3, dy, h2 = ints(tokens, d_model), ints(2 * hidden, d_model), ints(d_model, hidden), ints(tokens, d_model), ints(tokens, hidden)

    def same(got, a, b, scale=1.0):
        b = b.double()
        for i in range(0, a.size(0), 1 << 16):
            assert torch.equal(got[i:i + (1 << 16)], (a[i:i + (1 << 16)].double() @ b * scale).to(dt))

    def same_over_tokens(got, a, b):
        total = sum(a[i:i + (1 << 16)].double().t() @ b[i:i + (1 << 16)].double() for i in range(0, tokens, 1 << 16))
        assert torch.equal(got, total.to(dt))

    (out, c0), (h, c1), (gu, c2) = (_guarded(s, dt) for s in ((tokens, d_model), (tokens, hidden), (tokens, 2 * hidden)))
    _call("mg_mlp_fwd", (out, h, gu, x, w12, w3), sizes, "bf16")
    _intact(c0, c1, c2)
    same(gu, x, w12.t())
    for i in range(0, tokens, 1 << 16):
        hd, bd = h[i:i + (1 << 16)].double(), w3.double()
        _bounded(out[i:i + (1 << 16)], hd @ bd.t(), hd.abs() @ bd.abs().t(), hidden, "bf16")
    del out, h, c0, c1
    gu[:, :hidden], gu[:, hidden:] = 64, 1                   # where silu(g) is g and its slope 1
    (dx, c3), (da, c4), (db, c5), (dgu, c6) = (_guarded(s, dt) for s in (
        (tokens, d_model), (2 * hidden, d_model), (d_model, hidden), (tokens, 2 * hidden)))
    _call("mg_mlp_bwd", (dx, da, db, dgu, dy, x, w12, w3, gu, h2), sizes, "bf16")
    _intact(c2, c3, c4, c5, c6)
    same(dgu[:, :hidden], dy, w3)
    same(dgu[:, hidden:], dy, w3, 64.0)
    same(dx, dgu, w12)
    same_over_tokens(da, dgu, x)
    same_over_tokens(db, dy, h2)


def test_a_workspace_that_is_missing_or_too_small_is_refused():
    """By the host, before anything is launched."""
    sizes = t, d, h = 127, 1024, 11008
    x, w12, w3 = _case(t, d, h, "bf16")
    out, hid, gu = torch.zeros_like(x), x.new_empty(t, h), x.new_empty(t, 2 * h)
    grads = [torch.zeros_like(v) for v in (x, w12, w3)]
    for name, wanted, tensors in (("mg_mlp_fwd", 0, (out, hid, gu, x, w12, w3)), ("mg_mlp_bwd", 7, (*grads, torch.empty_like(gu), out, x, w12, w3, gu, hid))):
        need = ctypes.c_int64(0)
        U.check(U.lib().mg_mlp_workspace(*sizes, 2, wanted, ctypes.byref(need)))
        assert need.value > 0
        work = torch.empty(need.value, device="cuda", dtype=torch.uint8)
        for p, n in ((None, 0), (None, need.value), (work.data_ptr(), need.value - 1), (work.data_ptr(), 0)):
            assert getattr(U.lib(), name)(*(v.data_ptr() for v in tensors), p, n, *sizes, 2, U.stream()) == -1
            assert "workspace must hold" in U.lib().mg_last_error().decode()
    torch.cuda.synchronize()
    assert not out.any() and not any(v.any() for v in grads)


def test_what_is_not_finite_stays_in_its_row_and_column():
    x, w12, w3 = _case(200, 256, 512, "bf16")
    dy = torch.randn_like(x)
    sizes = (200, 256, 512)

    def run(x):
        out, h, gu = torch.empty_like(x), x.new_empty(200, 512), x.new_empty(200, 1024)
        _call("mg_mlp_fwd", (out, h, gu, x, w12, w3), sizes, "bf16")
        dx, dgu = torch.empty_like(x), torch.empty_like(gu)
        _call("mg_mlp_bwd", (dx, None, None, dgu, dy, x, w12, w3, gu, h), sizes, "bf16")
        return out, dx

    want = run(x)
    bad = x.clone()
    bad[77] = float("nan")
    bad[199, 3] = float("inf")
    keep = [i for i in range(200) if i not in (77, 199)]
    for a, b in zip(run(bad), want):
        assert torch.isnan(a[77]).all() and not torch.isfinite(a[199]).any() and torch.equal(a[keep], b[keep])


def _module(d_model=512, hidden=1024, dtype=torch.bfloat16, seed=0):
    torch.manual_seed(seed)
    module = MegaGemmTriton(d_model, multiple_of=64, hidden_multiple=hidden / d_model).cuda().to(dtype)
    assert module.hidden == hidden
    return module


def _grads(module, x, dy, call=None):
    for p in module.parameters():
        p.grad = None
    x = x.detach().clone().requires_grad_()
    y = (call or module)(x)
    y.backward(dy)
    return [y.detach(), x.grad, module.w12.weight.grad, module.w3.weight.grad]


def _through_projections(module):
    return lambda x: module.w3(ops.swiglu(module.w12(x), module.hidden))


def _close(got, want):
    for a, b in zip(got, want):      # [gate | up] and the gradient of h rounded on one way and not on the other
        assert a.shape == b.shape and a.dtype == b.dtype
        assert (a.float() - b.float()).norm() <= 2.0 ** -6 * b.float().norm()


def _takes(module, x):
    return ops.swiglu_mlp(x, module.w12.weight, module.w3.weight) is not None


@pytest.mark.parametrize("binding", ["extension", "ctypes"])
@pytest.mark.parametrize("shape", [(300, 512), (3, 100, 512), (2, 5, 33, 512)])
def test_module_takes_it(shape, binding, monkeypatch):
    if binding == "ctypes":
        monkeypatch.setattr(ops, "_binding", None)
        monkeypatch.setattr(ops, "_resolved", True)
    module = _module()
    x, dy = (torch.randn(shape, device="cuda", dtype=torch.bfloat16) for _ in range(2))
    got = _grads(module, x, dy)
    _close(got, _grads(module, x, dy, _through_projections(module)))
    with torch.no_grad():
        assert torch.equal(module(x), got[0]) and torch.equal(ops.swiglu_mlp(x, module.w12.weight, module.w3.weight), got[0])
    with torch.inference_mode():
        assert torch.equal(module(x.clone()), got[0]) and module(x[0, ..., :]).shape == x[0].shape
    # operands and gradients of other layouts
    xt = x.transpose(0, 1).contiguous().transpose(0, 1)
    assert all(torch.equal(a, b) for a, b in zip(_grads(module, x, dy), _grads(module, x, dy.transpose(0, 1).contiguous().transpose(0, 1))))
    assert torch.equal(module(xt), got[0])
    # the same in place: y is not a view of anything saved
    xa = x.clone().requires_grad_()
    y = module(xa)
    y.mul_(2).backward(dy / 2)
    assert torch.equal(xa.grad, got[1])
    # parts of the gradients, a second backward pass, other data under the operands in between
    xa = x.clone().requires_grad_()
    y = module(xa)
    xa.data = torch.zeros_like(x)
    w = module.w3.weight
    keep, w.data = w.data, torch.zeros_like(w.data)
    assert all(torch.equal(a, b) for a, b in zip(torch.autograd.grad(y, (xa, module.w12.weight, w), dy, retain_graph=True), got[1:]))
    for t, want in ((xa, got[1]), (module.w12.weight, got[2]), (w, got[3])):
        _close(torch.autograd.grad(y, t, dy, retain_graph=True), [want])
    w.data = keep
    for name in ("w12", "w3"):
        frozen = getattr(module, name).weight.requires_grad_(False)
        part = _grads(module, x, dy)
        frozen.requires_grad_()
        assert [g is None for g in part] == [False, False, name == "w12", name == "w3"]
        assert torch.equal(part[0], got[0])
        _close([g for g in part if g is not None], [want for g, want in zip(part, got) if g is not None])
    xa = x.clone().requires_grad_()
    y = module(xa)
    with torch.no_grad():
        xa.add_(1)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.backward(dy)


@pytest.mark.parametrize("binding", ["extension", "ctypes"])
def test_what_goes_through_the_projections(binding, monkeypatch):
    if binding == "ctypes":
        monkeypatch.setattr(ops, "_binding", None)
        monkeypatch.setattr(ops, "_resolved", True)
    module = _module()
    w12, w3 = module.w12.weight, module.w3.weight
    x = torch.randn(300, 512, device="cuda", dtype=torch.bfloat16)
    assert _takes(module, x) and _takes(module, x[:1])
    with torch.no_grad():
        assert _takes(module, x[:65]) and not _takes(module, x[:64])
    for y in (x.float(), x[:, :511], torch.randn(300 * 512 + 1, device="cuda", dtype=torch.bfloat16)[1:].view(300, 512)):
        assert ops.swiglu_mlp(y, w12, w3) is None
    assert ops.swiglu_mlp(x, w12.t().contiguous().t(), w3) is None and ops.swiglu_mlp(x, w12.half(), w3) is None
    assert ops.swiglu_mlp(x.to_sparse(), w12, w3) is None and ops.swiglu_mlp(x.cpu(), w12, w3) is None
    assert ops.swiglu_mlp(x, w12.detach()[:, :448].contiguous(), w3.detach()[:448].contiguous()) is None
    odd = torch.zeros(2 * 1000, 512, device="cuda", dtype=torch.bfloat16)
    assert ops.swiglu_mlp(x, odd, torch.zeros(512, 1000, device="cuda", dtype=torch.bfloat16)) is None
    # who looks at saved tensors, tangents or transforms sees the projections' ones
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t):
        assert not _takes(module, x)
    with torch.autograd.forward_ad.dual_level():
        assert not _takes(module, torch.autograd.forward_ad.make_dual(x, torch.ones_like(x)))
    seen = []
    torch.func.vmap(lambda t: (seen.append(_takes(module, t)), t)[1])(x.expand(2, 300, 512))
    torch.func.grad(lambda t: (seen.append(_takes(module, t)), t.sum())[1])(x)
    assert seen == [False, False]
    w12.requires_grad_(False)
    assert not _takes(module, x) and _takes(module, x.clone().requires_grad_())   # only w3 learns
    w12.requires_grad_()
    # frozen weights and more tokens than the gradient of x alone is taken for
    wide = _module(1024, 1792).requires_grad_(False)
    many = torch.randn(9000, 1024, device="cuda", dtype=torch.bfloat16)
    assert not _takes(wide, many.requires_grad_()) and _takes(wide, many[:8000])
    wide.w12.requires_grad_()
    assert _takes(wide, many)
    # a checkpointed block, and a gradient of a gradient, which the activation refuses
    dy = torch.randn_like(x)
    got = _grads(module, x, dy, lambda t: torch.utils.checkpoint.checkpoint(module, t, use_reentrant=False))
    _close(got, _grads(module, x, dy))
    xa = x.clone().requires_grad_()
    with pytest.raises(RuntimeError):
        torch.autograd.grad(module(xa).sum(), xa, create_graph=True)[0].sum().backward()
    for call in (module, _through_projections(module)):       # past the activation it can be had
        g = torch.autograd.grad(call(x), w3, dy, create_graph=True)[0]
        second = torch.autograd.grad(g.float().square().sum(), w12)[0]
        assert torch.isfinite(second).all() and second.abs().max() > 0


def test_the_block_under_graph_capture_and_on_other_streams():
    import threading

    module = _module()
    module.requires_grad_(False)
    xs = [torch.randn(300, 512, device="cuda", dtype=torch.bfloat16) for _ in range(4)]
    dy = torch.randn_like(xs[0])

    def step(x):
        x.requires_grad_()
        y = module(x)
        return y.detach(), torch.autograd.grad(y, x, dy)[0]

    want = [step(x.clone()) for x in xs]
    static, graph = xs[0].clone(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        out = step(static)
    for x, y in zip(xs, want):
        with torch.no_grad():
            static.copy_(x)
        torch.zeros(1024, device="cuda").add_(1)       # eager work between replays
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(out, y))
    got = [None] * 4

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(10):
                got[i] = step(xs[i].clone())
            torch.cuda.current_stream().synchronize()

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert all(torch.equal(a, b) for g, w in zip(got, want) for a, b in zip(g, w))


@pytest.fixture(params=["extension", "ctypes"])
def binding(request, monkeypatch):
    if request.param == "ctypes":
        monkeypatch.setattr(ops, "_binding", None)
        monkeypatch.setattr(ops, "_resolved", True)
    return request.param


def _batch(*shape, seed=0):
    return torch.randn(shape, device="cuda", generator=torch.Generator("cuda").manual_seed(seed)).to(torch.bfloat16)


def test_a_recorded_backward_pass_runs_hooks_once(binding):
    module = _module()
    module.w3.requires_grad_(False)          # with w3 learning the activation refuses to be recorded
    w12, x, dy = module.w12.weight, _batch(300, 512).requires_grad_(), _batch(300, 512, seed=1)
    want = torch.autograd.grad(module(x), (x, w12), dy)
    calls = []
    x.register_hook(lambda g: calls.append("x"))
    w12.register_hook(lambda g: calls.append("w12"))
    got = torch.autograd.grad(module(x), (x, w12), dy, create_graph=True)
    assert sorted(calls) == ["w12", "x"]
    _close(got, want)


def test_second_derivatives(binding):
    """Of the gradient of w3, through the activation to x and w12: as through the projections."""
    module = _module()
    w12, w3, dy = module.w12.weight, module.w3.weight, _batch(300, 512, seed=1)

    def second(call):
        x = _batch(300, 512).requires_grad_()
        g = torch.autograd.grad(call(x), w3, dy, create_graph=True)[0]
        return g.detach(), *torch.autograd.grad(g.float().square().sum() / 2, (x, w12))

    _close(second(module), second(_through_projections(module)))


def test_gradients_that_are_no_plain_tensors(binding):
    """A batch of them (is_grads_batched), lazily negated ones, and a dispatch mode that looks on."""
    module = _module()
    w3, x, dy = module.w3.weight, _batch(300, 512), _batch(3, 300, 512, seed=1)
    y = module(x)
    _close(torch.autograd.grad(y, w3, dy, is_grads_batched=True, retain_graph=True),
           [torch.stack([torch.autograd.grad(y, w3, d, retain_graph=True)[0] for d in dy])])
    with pytest.raises(RuntimeError):        # the activation's kernel takes no batch, as ever
        torch.autograd.grad(y, module.w12.weight, dy, is_grads_batched=True, retain_graph=True)
    _close(_grads(module, x, torch._neg_view(dy[0]))[1:], _grads(module, x, -dy[0])[1:])

    class Seen(torch.utils._python_dispatch.TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))

    class Nothing(torch.autograd.Function):
        @staticmethod
        def forward(ctx, t):
            return t.sum()

        @staticmethod
        def backward(ctx, g):
            return None

    assert torch.autograd.grad(Nothing.apply(y), (module.w12.weight, w3), retain_graph=True, allow_unused=True) == (None, None)
    seen = []
    with Seen():
        got = torch.autograd.grad(y, (module.w12.weight, w3), dy[0], retain_graph=True)
    assert torch.ops.aten.mm.default in seen
    _close(got, torch.autograd.grad(y, (module.w12.weight, w3), dy[0]))


@pytest.mark.parametrize("learning", ["x", "w12", "x w3", "w12 w3", "x w12", "x w12 w3"])
def test_nothing_is_kept_that_no_gradient_needs(learning, binding):
    """x is kept for the gradient of w12, w12 for that of x, h for that of w3, as by the projections: the others
    may be changed between the passes, and the memory of activations is free."""
    module = _module()
    w12, w3 = module.w12.weight.requires_grad_("w12" in learning), module.w3.weight.requires_grad_("w3" in learning)
    x0, dy = _batch(100, 512).requires_grad_("x" in learning.split()), _batch(100, 512, seed=1)   # tensors below 1 MiB: allocated to size
    wanted = [t for t in (x0, w12, w3) if t.requires_grad]
    want = torch.autograd.grad(module(x0), wanted, dy)
    mib = lambda: torch.cuda.memory_allocated()
    before = mib()
    y = module(x0 * 1)
    elements = 512 + 2 * 1024 + (1024 if "w3" in learning else 0) + (512 if "w12" in learning else 0)
    assert mib() - before == 100 * elements * 2       # y, [gate | up], h, x
    x = x0 * 1
    y = module(x)
    with torch.no_grad():
        if "w12" not in learning:
            x.add_(y)
        if "x" not in learning.split():
            w12.mul_(2)
    assert all(torch.equal(a, b) for a, b in zip(torch.autograd.grad(y, wanted, dy, retain_graph=True), want))
    for t in [w3] + [x] * ("w12" in learning) + [w12] * ("x" in learning.split()):
        y = module(x)
        with torch.no_grad():
            t.add_(1)
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            torch.autograd.grad(y, wanted, dy)
    # a graph over the gradient of w3 reaches whatever learns
    if "w3" in learning:
        def second(call):
            y = call(x0)
            g = torch.autograd.grad(y, w3, dy, create_graph=True)[0]
            return torch.autograd.grad(g.float().square().sum() / 2, wanted[:-1])

        _close(second(module), second(_through_projections(module)))


def test_x_that_is_not_contiguous_is_kept_once(binding):
    module, x0 = _module(), _batch(5, 20, 512).requires_grad_()
    before = torch.cuda.memory_allocated()
    y = module((x0 * 1).transpose(0, 1))
    assert torch.cuda.memory_allocated() - before == 100 * (512 + 2 * 1024 + 1024 + 512) * 2 and y.shape == (20, 5, 512)


def test_inputs_that_no_wanted_gradient_reads_may_be_null():
    x, w12, w3 = _case(300, 512, 1024, "bf16")
    dy, sizes = _batch(300, 512), (300, 512, 1024)
    out, h, gu = torch.empty_like(x), x.new_empty(300, 1024), x.new_empty(300, 2048)
    _call("mg_mlp_fwd", (out, h, gu, x, w12, w3), sizes, "bf16")
    for wanted, unread in ((0, (5, 9)), (1, (6, 9)), (2, (5, 6, 7, 8))):       # dx, dw12, dw3
        results = []
        for drop in ((), unread):
            grads = [torch.empty_like(t) if i == wanted else None for i, t in enumerate((x, w12, w3))]
            work = None if wanted == 2 else torch.empty_like(gu)
            tensors = [*grads, work, dy, x, w12, w3, gu, h]
            _call("mg_mlp_bwd", [None if i in drop else t for i, t in enumerate(tensors)], sizes, "bf16")
            results.append(grads[wanted])
        assert torch.equal(*results)
        for needed in {4, 5, 6, 7, 8, 9} - set(unread):
            with pytest.raises(Exception, match="must not be NULL"):
                _call("mg_mlp_bwd", [None if i == needed else t for i, t in enumerate(tensors)], sizes, "bf16")
