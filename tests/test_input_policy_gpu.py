"""Most forward kernels read inputs of up to 128 MiB with another cache policy than larger ones, which
are other instances of the kernel: the same rows give the same bits on both sides of that line."""
import pytest
import torch

pytestmark = pytest.mark.gpu

LINE = 128 << 20
F16, BF16, F32 = torch.float16, torch.bfloat16, torch.float32


def _copies(block, rows):
    return block.repeat((rows + block.size(0) - 1) // block.size(0), 1)[:rows].contiguous()


# by family of forward kernels, with shapes on different numbers of lanes
FOLLOW_THE_LINE = [
    (4096, BF16), (8191, F16), (1032, BF16), (2048, F32), (16384, BF16),     # a row over 64 ... 1024 threads
    (1024, F16), (512, BF16), (256, F16),                                    # several vectors per lane, 32, 16 and 8 lanes
    (80, BF16), (64, F32), (264, BF16), (24, F16), (8, BF16),                # row groups, 16, 16, 64, 4 and 1 lanes
]
# ... and those that read every input alike, where only the rows' independence of their number is tested
READ_ALIKE = [(100, BF16), (129, F16), (70000, BF16)]                        # ragged groups and lanes; rows read twice


@pytest.mark.parametrize("cols,dtype", FOLLOW_THE_LINE + READ_ALIKE)
def test_rmsnorm_forward_on_both_sides_of_the_line(cols, dtype):
    from mgrrmsnorm_amd import ops

    size = torch.empty((), dtype=dtype).element_size()
    at = LINE // (cols * size)          # the most rows that still count as small
    g = torch.Generator(device="cuda").manual_seed(cols)
    block = torch.randn(min(at, 37), cols, generator=g, device="cuda", dtype=dtype)
    w = 1 + 0.1 * torch.randn(cols, generator=g, device="cuda", dtype=dtype)
    y, s = ops.rmsnorm_forward(block, w, 1e-6)
    for rows in (at, at + 1):
        yy, ss = ops.rmsnorm_forward(_copies(block, rows), w, 1e-6)
        assert torch.equal(yy, _copies(y, rows)) and torch.equal(ss, _copies(s[:, None], rows)[:, 0])


# aligned half rows follow the line; ragged ones (2731) are read alike
@pytest.mark.parametrize("hidden,dtype", [(4096, BF16), (1000, F32), (2731, F16)])
def test_swiglu_forward_on_both_sides_of_the_line(hidden, dtype):
    from mgrrmsnorm_amd import ops

    at = LINE // (2 * hidden * torch.empty((), dtype=dtype).element_size())
    g = torch.Generator(device="cuda").manual_seed(hidden)
    block = torch.randn(37, 2 * hidden, generator=g, device="cuda", dtype=dtype)
    h = ops.swiglu_forward(block, hidden)
    for rows in (at, at + 1):
        assert torch.equal(ops.swiglu_forward(_copies(block, rows), hidden), _copies(h, rows))


def _kernels(fn):
    """Names of this library's forward kernels that `fn` launches."""
    from torch.profiler import ProfilerActivity, profile

    fn()
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as p:
        fn()
        torch.cuda.synchronize()
    return [e.name for e in p.events() if "rmsnorm_fwd" in e.name or "swiglu_fwd" in e.name]


@pytest.mark.parametrize("backend", ["extension", "ctypes"])
@pytest.mark.parametrize("path", ["rmsnorm", "swiglu"])
def test_inputs_are_kept_only_for_a_backward_pass(monkeypatch, backend, path):
    """Without a gradient to compute, an input of any size is read as a large one is."""
    import mgrrmsnorm_amd
    from mgrrmsnorm_amd import ops

    assert ops.backend() == "extension"
    if backend == "ctypes":
        monkeypatch.setattr(ops, "_binding", None)
    cols = 1024
    norm = mgrrmsnorm_amd.RMSNorm(cols).cuda().to(BF16)
    call = norm if path == "rmsnorm" else lambda x: ops.swiglu(x, cols // 2)
    small, large = (torch.zeros(rows, cols, device="cuda", dtype=BF16) for rows in (512, LINE // (cols * 2) + 1))

    def name(x, grad):
        with torch.set_grad_enabled(grad):
            got = _kernels(lambda: call(x.requires_grad_(grad)))
        assert len(got) == 1, got
        return got[0]

    streamed = name(large, True)
    assert name(small, True) != streamed
    assert name(small, False) == streamed and name(large, False) == streamed
