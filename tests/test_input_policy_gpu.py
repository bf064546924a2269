"""The forward kernels read inputs of up to 128 MiB with another cache policy than larger ones:
the same rows give the same bits on both sides of that line."""
import pytest
import torch

pytestmark = pytest.mark.gpu

LINE = 128 << 20
F16, BF16, F32 = torch.float16, torch.bfloat16, torch.float32


def _copies(block, rows):
    return block.repeat((rows + block.size(0) - 1) // block.size(0), 1)[:rows].contiguous()


# one shape of each family of forward kernels: rows, several vectors per lane, row groups, two reads
@pytest.mark.parametrize("cols,dtype", [(4096, BF16), (8191, F16), (1024, F16), (80, BF16), (64, F32), (100, BF16), (70000, BF16)])
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


@pytest.mark.parametrize("hidden,dtype", [(4096, BF16), (1000, F32), (2731, F16)])
def test_swiglu_forward_on_both_sides_of_the_line(hidden, dtype):
    from mgrrmsnorm_amd import ops

    at = LINE // (2 * hidden * torch.empty((), dtype=dtype).element_size())
    g = torch.Generator(device="cuda").manual_seed(hidden)
    block = torch.randn(37, 2 * hidden, generator=g, device="cuda", dtype=dtype)
    h = ops.swiglu_forward(block, hidden)
    for rows in (at, at + 1):
        assert torch.equal(ops.swiglu_forward(_copies(block, rows), hidden), _copies(h, rows))
