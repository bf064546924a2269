"""What of the block's own products can be checked without a GPU: the sizes and arguments the C entry points take,
and the calls MegaGemmTriton hands to them."""
import random
import re
import shutil
import subprocess
from pathlib import Path

import pytest
import torch

from mgrrmsnorm_amd import _lib, ops
from test_block_route_cpu import CHANGES, REPLACED, _module


@pytest.fixture(scope="module")
def lib():
    return _lib.load()


def test_header_compiles_and_declares_what_the_library_exports(lib, tmp_path):
    header = Path(__file__).resolve().parent.parent / "include" / "megagemm_hip_mlp.h"
    text = re.sub(r"/\*.*?\*/", "", header.read_text(), flags=re.S)
    assert sorted(re.findall(r"\b(mg_[a-z0-9_]+)\s*\(", text)) == sorted(_lib.MLP_SIGNATURES)
    assert all(hasattr(lib, name) for name in _lib.MLP_SIGNATURES)
    source = tmp_path / "t.c"
    source.write_text('#include "megagemm_hip_mlp.h"\nint main(void){return MG_MLP_ALL + MG_MLP_FORWARD;}\n')
    for compiler in (["gcc", "-std=c99"], ["g++", "-x", "c++"]):
        subprocess.run([*compiler, "-Wall", "-Werror", f"-I{header.parent}", "-c", str(source), "-o", str(tmp_path / "t.o")], check=True)


@pytest.mark.parametrize("tokens,d_model,hidden,dtype,fits", [
    (1, 64, 64, 1, 1), (0, 64, 64, 1, 0), (1, 64, 64, 0, 0), (5, 96, 64, 2, 0), (5, 64, 96, 2, 0), (5, 65536, 8128, 2, 1), (5, 65536, 8192, 2, 0),
    (5, 65600, 64, 2, 0), (5, 16384, 32704, 2, 1), (5, 16384, 32768, 2, 0), (1 << 24, 64, 64, 2, 0), (8191, 64, 65536, 2, 1), (8192, 64, 65536, 2, 0),
])
def test_sizes(lib, tokens, d_model, hidden, dtype, fits):
    assert lib.mg_mlp_fits(tokens, d_model, hidden, dtype) == fits
    assert all(lib.mg_mlp_preferred(tokens, d_model, hidden, dtype, only) <= fits for only in (0, 1))


@pytest.mark.parametrize("tokens,d_model,hidden,training,alone", [
    (1, 64, 64, 1, 0), (16, 1024, 1792, 1, 0), (64, 1024, 1792, 1, 0), (65, 1024, 1792, 1, 1), (1, 1024, 2816, 1, 1),
    (2048, 4096, 6912, 1, 0), (2049, 4096, 6912, 0, 0), (8192, 4096, 5440, 1, 0),
    # forward alone: faster and slower than the library's products, by the times beside the rule
    (65536, 512, 1024, 1, 1), (1024, 2048, 3584, 1, 1), (8192, 2048, 3584, 1, 0), (256, 4096, 11008, 1, 1), (320, 4096, 11008, 1, 0),
    (384, 4096, 11008, 1, 0), (448, 4096, 11008, 1, 1), (256, 4096, 6912, 1, 1), (640, 4096, 6912, 1, 0), (65536, 4096, 5440, 1, 0),
    (64, 8192, 2048, 1, 0), (64, 4096, 6912, 1, 1),
])
def test_where_they_are_taken(lib, tokens, d_model, hidden, training, alone):
    assert [lib.mg_mlp_preferred(tokens, d_model, hidden, 2, only) for only in (0, 1)] == [training, alone]


@pytest.mark.parametrize("tokens,d_model,hidden,taken", [
    (1, 512, 1024, 1), (65536, 512, 1024, 1), (8192, 1024, 2816, 1), (8193, 1024, 1792, 0), (900, 4096, 6912, 1), (1300, 4096, 6912, 0), (4096, 2048, 3584, 1),
    (8192, 2048, 3584, 0), (1024, 4096, 4096, 1), (1100, 4096, 4096, 0), (2500, 4096, 2048, 0), (3000, 4096, 6912, 0),
])
def test_where_they_are_taken_if_only_x_learns(lib, tokens, d_model, hidden, taken):
    assert lib.mg_mlp_preferred(tokens, d_model, hidden, 1, 2) == taken
    assert lib.mg_mlp_preferred(tokens, d_model, hidden, 1, 0) >= taken


def test_bad_arguments_are_refused(lib):
    t, d, h = 100, 64, 128
    error = lambda: lib.mg_last_error().decode()
    p = {n: 0x10000000 * (i + 1) for i, n in enumerate(("out", "h", "gu", "x", "w12", "w3", "dx", "dw12", "dw3", "dgu", "dy"))}

    def fwd(sizes=(t, d, h), dtype=2, **other):
        q = {**p, **other}
        return lib.mg_mlp_fwd(*(q[n] for n in ("out", "h", "gu", "x", "w12", "w3")), None, 0, *sizes, dtype, None)

    def bwd(**other):
        q = {**p, **other}
        return lib.mg_mlp_bwd(*(q[n] for n in ("dx", "dw12", "dw3", "dgu", "dy", "x", "w12", "w3", "gu", "h")), None, 0, t, d, h, 2, None)

    assert fwd((t, d, 96)) == -2 and fwd(dtype=0) == -2 and fwd((0, d, h)) == -2
    for name in ("out", "h", "x", "w12", "w3"):
        assert fwd(**{name: None}) == -1 and "NULL" in error()
    for name in ("dy", "x", "w12", "w3", "gu", "h", "dgu"):
        assert bwd(**{name: None}) == -1
    for call, name in ((fwd, "x"), (fwd, "gu"), (bwd, "dw3"), (bwd, "h")):
        assert call(**{name: p[name] + 8}) == -1 and "aligned" in error()
    for call, a, b in ((fwd, "out", "x"), (fwd, "h", "gu"), (fwd, "gu", "w12"), (bwd, "dgu", "gu"), (bwd, "dx", "dy"), (bwd, "dw3", "dw12")):
        assert call(**{a: p[b]}) == -1 and "overlaps" in error()


@pytest.fixture
def handed_over(monkeypatch):
    """Calls the module and returns the (w12, w3) it handed to ops.swiglu_mlp, or None."""
    calls = []
    monkeypatch.setattr(ops, "swiglu_block_fits", lambda x, hidden: False)
    monkeypatch.setattr(ops, "swiglu_mlp_fits", lambda x, hidden: True)
    monkeypatch.setattr(ops, "swiglu_mlp", lambda x, w12, w3: calls.append((w12, w3)))

    def call(module):
        calls.clear()
        try:
            module(torch.zeros(2, 16))
        except RuntimeError:       # past the hand-over: no GPU, or a stand-in of another shape
            pass
        return calls[0] if calls else None
    return call


def test_a_module_as_made_is_handed_over(handed_over):
    m = _module()
    w12, w3 = handed_over(m)
    assert w12 is m.w12.weight and w3 is m.w3.weight


@pytest.mark.parametrize("change", CHANGES)
def test_a_changed_projection_is_called(handed_over, change):
    m = _module()
    CHANGES[change](m)
    assert handed_over(m) is None


@pytest.mark.parametrize("what", REPLACED)
def test_a_replaced_function_is_called(handed_over, monkeypatch, what):
    owner, name, value = REPLACED[what]
    monkeypatch.setattr(owner, name, value)
    assert handed_over(_module()) is None


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs a C++ compiler")
def test_every_planned_kernel_is_run_against_float64(lib, tmp_path):
    """What the planner makes of the sizes the C entry points take, against the sizes of test_mlp_gpu.py."""
    from test_mlp_gpu import SIZES

    program = tmp_path / "mlp_plans"
    subprocess.run(["g++", "-std=c++17", "-O2", str(Path(__file__).parent / "standalone" / "mlp_plans.cpp"), "-o", str(program)], check=True)

    def plans(sizes):
        text = "\n".join("%d %d %d" % s for s in sizes)
        return set(subprocess.run([str(program)], input=text, text=True, capture_output=True, check=True).stdout.split())

    rng = random.Random(0)
    spread = lambda low, high: round(low * (high / low) ** rng.random())
    sizes = [(spread(1, 1 << 20), 64 * spread(1, 1024), 64 * spread(1, 1024)) for _ in range(40000)]
    sizes = [s for s in sizes if lib.mg_mlp_fits(*s, 2)]
    assert len(sizes) > 20000
    missing = plans(sizes) - plans(SIZES)
    assert not missing
