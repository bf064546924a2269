"""RMSNorm backward in one launch (mg_rmsnorm_bwd_small) against the oracle: rows around the 8, 128
and 512 that a wave, a pass and an unrolled pass of the column sums cover, widths around a
128-byte line, a wave of vectors, a workgroup of vectors and two vectors per lane, odd widths (rows ending in
half a dword) and bases off alignment, with canaries around dx and both dW."""
import numpy as np
import pytest
import torch

import gpu_util as U

pytestmark = pytest.mark.gpu

EPS = 1e-6
PAD = 64
SHAPES = [(1, 1), (1, 64), (7, 65), (8, 8191), (9, 3), (127, 512), (128, 513), (129, 63), (512, 1000), (513, 4100),
          (1024, 33), (30, 8192), (17, 8193), (12, 16384), (33, 16383), (5, 12000)]


def _padded(n, td, off, src=None):
    buf = torch.full((PAD + off + n + PAD,), 7.0, dtype=td, device="cuda")
    view = buf[PAD + off:PAD + off + n]
    if src is not None:
        view.copy_(src.reshape(-1))
    return buf, view


@pytest.mark.parametrize("dtype", ["bf16", "fp16", "fp32"])
@pytest.mark.parametrize("rows,cols", SHAPES)
def test_one_launch_backward_against_the_oracle(rows, cols, dtype):
    es = 4 if dtype == "fp32" else 2
    L, td, code = U.lib(), U.DTYPES[dtype], U.CODES[dtype]
    x, dy, w = U.rmsnorm_inputs(rows, cols, dtype, seed=rows * 131 + cols)
    y_ref, s_ref, dx_ref, dw_ref, floor = U.rmsnorm_reference(x, dy, w, EPS, dtype)
    s = torch.from_numpy(s_ref.astype(np.float32)).cuda()
    if cols * es > 32768:
        assert not L.mg_rmsnorm_bwd_small_fits(rows, cols, code)
        p = s.data_ptr()
        assert L.mg_rmsnorm_bwd_small(p, p, None, p, p, p, p, rows, cols, code, U.stream()) == -2
        return
    for off in (0, 1, 4):
        print(f"bwd_small {rows}x{cols} {dtype} offset {off}", flush=True)
        _, xd = _padded(rows * cols, td, off, x)
        _, gd = _padded(rows * cols, td, off, dy)
        _, wd = _padded(cols, td, off, w)
        dxb, dx = _padded(rows * cols, td, off)
        f32b, f32 = _padded(cols, torch.float32, off)
        castb, cast = _padded(cols, td, off)
        U.check(L.mg_rmsnorm_bwd_small(dx.data_ptr(), f32.data_ptr(), cast.data_ptr(), gd.data_ptr(), xd.data_ptr(),
                                       wd.data_ptr(), s.data_ptr(), rows, cols, code, U.stream()))
        torch.cuda.synchronize()
        for buf, n in ((dxb, rows * cols), (f32b, cols), (castb, cols)):
            assert bool((buf[:PAD + off] == 7).all() and (buf[PAD + off + n:] == 7).all()), "store outside an output"
        U.assert_matches(dx.view(rows, cols).contiguous(), dx_ref, dtype, "dx, one launch", floor=floor)
        U.assert_dw(f32.contiguous(), dw_ref, f"dW {rows}x{cols}")
        assert torch.equal(cast, f32.to(td))
        only = torch.empty_like(cast)      # one dW alone, and none: same dx, same bits
        dx2 = torch.empty_like(dx)
        U.check(L.mg_rmsnorm_bwd_small(dx2.data_ptr(), None, only.data_ptr(), gd.data_ptr(), xd.data_ptr(), wd.data_ptr(),
                                       s.data_ptr(), rows, cols, code, U.stream()))
        assert torch.equal(only, cast) and torch.equal(dx2, dx)
        dx2.zero_()
        U.check(L.mg_rmsnorm_bwd_small(dx2.data_ptr(), None, None, gd.data_ptr(), xd.data_ptr(), wd.data_ptr(), s.data_ptr(),
                                       rows, cols, code, U.stream()))
        assert torch.equal(dx2, dx)


def test_which_shapes_take_it():
    fits = U.lib().mg_rmsnorm_bwd_small_fits
    assert fits(1, 1, 2) and fits(1024, 16384, 2) and fits(512, 8192, 0) and fits(1024, 2048, 0)
    assert not fits(0, 64, 2) and not fits(1025, 64, 2) and not fits(1, 16385, 2) and not fits(513, 8192, 0)
    assert not fits(4, 64, 7)


@pytest.mark.parametrize("option", [("force_generic", 1, 0), ("bwd_partials", 7, 0)])
def test_overrides_reach_few_rows_through_both_bindings(option):
    """With an override set, backward of few rows through the bindings is what the two C calls give."""
    from mgrrmsnorm_amd import ops, ops_ctypes

    rows, cols, dtype = 200, 1000, "bf16"
    x, dy, w = U.rmsnorm_inputs(rows, cols, dtype, seed=3)
    xd, gd, wd = x.cuda(), dy.cuda(), w.cuda()
    key, value, default = option
    y, s = ops.rmsnorm_forward(xd, wd, EPS)
    alone = ops.rmsnorm_backward_f32(gd, xd, wd, s)[1]
    try:
        U.check(U.lib().mg_set_option(key.encode(), value))
        dx, dw, cast, _ = U.rmsnorm_bwd(gd, xd, wd, s, dtype)
        for module in (ops, ops_ctypes):
            got = module.rmsnorm_backward_f32(gd, xd, wd, s)
            assert torch.equal(got[0], dx) and torch.equal(got[1], dw) and torch.equal(got[2], cast)
    finally:
        U.check(U.lib().mg_set_option(key.encode(), default))
    assert not torch.equal(dw, alone)          # another summation order: the override did reach the sums
    assert torch.equal(ops.rmsnorm_backward_f32(gd, xd, wd, s)[1], alone)
