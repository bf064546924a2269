"""The SwiGLU block as one operator (megagemm_hip_fused.h): a decoding step through MegaGemmTriton
against the same formula in float64, at the sizes where the split over workgroups, waves and
16-row tiles has edges, and the calls that have to keep going through the projections."""
import pytest
import torch

import gpu_util as U
from mgrrmsnorm_amd import MegaGemmTriton, ops

pytestmark = pytest.mark.gpu

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
HALF_ULP = {"bf16": 2.0 ** -9, "fp16": 2.0 ** -12}   # largest relative error of one rounding (bf16: 8 bits, fp16: 11)


def _case(tokens, d_model, hidden, dtype, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    n = lambda *s: torch.randn(s, generator=g, device="cuda")
    dt = DTYPES[dtype]
    return n(tokens, d_model).to(dt), (n(2 * hidden, d_model) * d_model ** -0.5).to(dt), (n(d_model, hidden) * hidden ** -0.5).to(dt)


def _within(out, x, w12, w3, dtype):
    """Every element within what one rounding of h, one of the result and two fp32 sums can do."""
    xd, ad, bd = x.double(), w12.double(), w3.double()
    gate, up = (xd @ ad.t()).chunk(2, -1)
    h = torch.nn.functional.silu(gate) * up
    ref = h @ bd.t()
    u, e = HALF_ULP[dtype], 2.0 ** -24
    tiny = 2.0 ** -25 if dtype == "fp16" else 0.0                       # half a subnormal step of fp16
    # error of gate and up from an fp32 sum of d_model products, carried through silu'(g) <= 1.1
    ag, au = (xd.abs() @ ad.abs().t()).chunk(2, -1)
    k = (x.size(-1) + 8) * e
    dh = k * (1.1 * ag * up.abs() + au * gate.abs()) + 8 * e * h.abs() + u * h.abs() + tiny
    bound = (dh + (w3.size(1) + 8) * e * h.abs()) @ bd.abs().t() * (1 + u) + u * ref.abs() + tiny
    worst = ((out.double() - ref).abs() - bound).max().item()
    assert worst <= 0.0, f"beyond the error bound by {worst}"


def _two_kernels(x, w12, w3, dtype):
    """The block through the C entry points, which take up to 64 tokens of any size."""
    tokens, d_model, hidden = x.size(0), x.size(1), w3.size(1)
    h, out = torch.empty(tokens, hidden, device="cuda", dtype=x.dtype), torch.empty_like(x)
    U.check(U.lib().mg_block_gate_up(h.data_ptr(), x.data_ptr(), w12.data_ptr(), tokens, d_model, hidden, U.CODES[dtype], U.stream()))
    U.check(U.lib().mg_block_down(out.data_ptr(), h.data_ptr(), w3.data_ptr(), tokens, d_model, hidden, U.CODES[dtype], U.stream()))
    return out


def _taken(tokens, d_model, hidden):
    """The operator's rule: tokens, MiB of weights, and how far the two widths lie apart."""
    mib, apart = 6 * d_model * hidden / 2 ** 20, max(d_model, hidden) / min(d_model, hidden)
    return tokens <= 16 or (tokens <= 32 and mib <= 42 and apart <= 4) or (tokens <= 64 and mib <= 9 and apart <= 3)


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("tokens,d_model,hidden", [
    (1, 8, 8), (3, 40, 24), (16, 64, 72), (15, 72, 1000), (2, 520, 264), (16, 1152, 3072),
    (8, 4096, 6912),      # three and a half tiles of columns per workgroup, one of the second projection
    (5, 64, 9000),        # more columns per workgroup than four tiles hold
    (7, 17000, 128),      # the same in the second projection
    (9, 8192, 2048),      # two tiles of the second projection per workgroup
    (17, 40, 24), (24, 4096, 6912), (32, 1152, 3072), (33, 264, 9000), (48, 520, 264), (49, 9000, 72), (64, 1024, 3072),   # tiles of tokens
])
def test_decode_block_against_float64(tokens, d_model, hidden, dtype):
    x, w12, w3 = _case(tokens, d_model, hidden, dtype)
    out = _two_kernels(x, w12, w3, dtype)
    _within(out, x, w12, w3, dtype)
    assert torch.equal(out, _two_kernels(x, w12, w3, dtype))   # fixed summation order
    block = ops.swiglu_block(x, w12, w3)
    assert (block is not None) == _taken(tokens, d_model, hidden)
    if block is not None:
        assert block.shape == x.shape and block.dtype == x.dtype and torch.equal(block, out)


@pytest.mark.parametrize("tokens,d_model,hidden,taken", [
    (16, 8192, 14336, True), (17, 2048, 3584, True), (17, 2048, 3592, False), (32, 2048, 3584, True),
    (24, 4096, 6912, False), (17, 1024, 4096, True), (17, 1024, 4104, False), (17, 4104, 1024, False),
    (33, 768, 2048, True), (33, 768, 2056, False), (64, 768, 2048, True), (64, 1024, 3072, False),
    (33, 512, 1536, True), (33, 512, 1544, False), (64, 1544, 512, False),
])
def test_where_the_block_takes_the_two_kernels(tokens, d_model, hidden, taken):
    """Beyond these lines the library's products are at least as fast on the GPU (see block_in_two_kernels)."""
    assert _taken(tokens, d_model, hidden) == taken
    x, w12, w3 = (torch.zeros(s, device="cuda", dtype=torch.bfloat16) for s in ((tokens, d_model), (2 * hidden, d_model), (d_model, hidden)))
    assert (ops.swiglu_block(x, w12, w3) is not None) == taken


def test_rows_do_not_depend_on_each_other():
    x, w12, w3 = _case(16, 256, 512, "bf16")
    out = ops.swiglu_block(x, w12, w3)
    for t in (1, 5):
        assert torch.equal(ops.swiglu_block(x[:t].contiguous(), w12, w3), out[:t])
    x[3] = float("nan")
    bad = ops.swiglu_block(x, w12, w3)
    keep = [t for t in range(16) if t != 3]
    assert torch.isnan(bad[3]).all() and torch.equal(bad[keep], out[keep])


def test_module_takes_it_and_steps_aside():
    module = MegaGemmTriton(256).cuda().to(torch.bfloat16)
    x = torch.randn(2, 3, 256, device="cuda", dtype=torch.bfloat16)
    w12, w3 = module.w12.weight, module.w3.weight
    with torch.no_grad():
        fused = module(x)
        assert torch.equal(fused, ops.swiglu_block(x, w12, w3)) and fused.shape == x.shape
        seen = []
        handle = module.w12.register_forward_hook(lambda m, i, o: seen.append(o.shape))
        hooked = module(x)
        handle.remove()
        assert seen == [(2, 3, 2 * module.hidden)]
        assert (hooked - fused).abs().max() <= 2.0 ** -6 * fused.abs().max()   # h and [gate | up] rounded on the way
        with torch.autocast("cuda", dtype=torch.float16):
            assert module(x).dtype == torch.float16
    y = module(x)                                       # gradients wanted: the differentiable path
    assert y.requires_grad
    y.sum().backward()
    assert w12.grad is not None and w3.grad is not None


@pytest.mark.parametrize("change", ["tokens", "size", "dtype", "width", "alignment", "layout"])
def test_calls_it_does_not_take(change):
    x, w12, w3 = _case(4, 64, 64, "bf16")
    if change == "tokens":
        x = x.repeat(17, 1)
    elif change == "size":
        x, w12, w3 = _case(25, 4096, 6912, "bf16")   # the library is as fast from here on
    elif change == "dtype":
        x, w12, w3 = x.float(), w12.float(), w3.float()
    elif change == "width":
        x, w12, w3 = _case(4, 60, 64, "bf16")
    elif change == "alignment":
        w3 = torch.empty(64 * 64 + 1, device="cuda", dtype=torch.bfloat16)[1:].view(64, 64).copy_(w3)
    else:
        w12 = w12.t().contiguous().t()
    assert ops.swiglu_block(x, w12, w3) is None


@pytest.mark.parametrize("operand", [0, 1, 2])
def test_sparse_operands(operand):
    """Coordinate tensors are left to the projections; compressed ones raise here.  Neither is taken on
    to torch's products: those of 16-bit compressed weights end the process instead of raising."""
    operands = list(_case(4, 64, 64, "bf16"))
    dense = operands[operand]
    operands[operand] = dense.to_sparse()
    assert ops.swiglu_block(*operands) is None
    operands[operand] = dense.to_sparse_csr()
    with pytest.raises(RuntimeError, match="contiguous"):
        ops.swiglu_block(*operands)


def test_the_block_under_graph_capture_and_on_other_streams():
    """A decoding step captured into a graph, and issued from four threads on streams of their own."""
    import threading

    module = MegaGemmTriton(512).cuda().to(torch.bfloat16)
    xs = [torch.randn(8, 512, device="cuda", dtype=torch.bfloat16) for _ in range(4)]
    with torch.no_grad():
        want = [module(x) for x in xs]
        assert torch.equal(want[0], ops.swiglu_block(xs[0], module.w12.weight, module.w3.weight))
        static, graph = xs[0].clone(), torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        with torch.cuda.graph(graph):
            out = module(static)
        for x, y in zip(xs, want):
            static.copy_(x)
            torch.zeros(1024, device="cuda").add_(1)       # eager work between replays
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, y)
    got = [None] * 4

    def work(i):
        with torch.no_grad(), torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(20):
                got[i] = module(xs[i])
            torch.cuda.current_stream().synchronize()

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert all(torch.equal(a, b) for a, b in zip(got, want))
