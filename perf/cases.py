"""The workloads this package is timed on: RMSNorm, the SwiGLU activation and the SwiGLU block,
through the entry points a program uses (`megagemm.RMSNorm`, `mgrrmsnorm_amd.ops.swiglu`,
`megagemm.MegaGemmTriton`).

A case is a dict: "path" (norm, act, block), "train" (forward + backward, else forward under
`torch.no_grad()`), "dtype" and the sizes -- "rows" x "cols" for norm, "rows" x 2*"hidden" for
act, "tokens" x "d_model" with "hidden" for block -- and for norm "outliers" (1 % of the
entries of x and dy a hundred times larger).
"""
import torch

import megagemm
from mgrrmsnorm_amd import ops

DTYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}
BYTES = {"fp32": 4, "fp16": 2, "bf16": 2}
EPS = 1e-6

# Largest listed norm (65536 x 16384), and what the largest block pass below may multiply-add.
MOST_ELEMENTS = 65536 * 16384
MOST_BLOCK_FLOPS = 5e11


def norm(name, rows, cols, dtype, train, outliers=False):
    return {"name": name, "path": "norm", "rows": rows, "cols": cols, "dtype": dtype, "train": train, "outliers": outliers}


def act(name, rows, hidden, dtype, train):
    return {"name": name, "path": "act", "rows": rows, "hidden": hidden, "dtype": dtype, "train": train}


def block(name, tokens, d_model, hidden, dtype, train):
    return {"name": name, "path": "block", "tokens": tokens, "d_model": d_model, "hidden": hidden, "dtype": dtype, "train": train}


def listed():
    return [
        # one decoding step of a small batch: a norm in front of every projection, nothing but latency
        norm("norm_decode_8x4096_bf16", 8, 4096, "bf16", False),
        # prompt processing, 32 x 128 tokens: the benchmark configuration of the fp16 forward
        norm("norm_prefill_4096x4096_fp16", 4096, 4096, "fp16", False),
        # fine-tuning of a small network in full precision: a training step that is mostly launches
        norm("norm_train_512x768_fp32", 512, 768, "fp32", True),
        # the headline workload
        norm("norm_train_4096x4096_bf16", 4096, 4096, "bf16", True),
        # per-head query/key norm, head dimension 80: rows narrower than a wavefront
        norm("norm_train_262144x80_bf16", 262144, 80, "bf16", True),
        # 8 x 2048 tokens of a wide network
        norm("norm_train_16384x8192_bf16", 16384, 8192, "bf16", True),
        # ragged width (row pitch 8200 bytes), with outliers that stress the accumulation
        norm("norm_train_65536x4100_fp16", 65536, 4100, "fp16", True, True),
        # the largest: 2 GiB per tensor
        norm("norm_train_65536x16384_bf16", 65536, 16384, "bf16", True, True),
        # activation of a feed-forward block, 8 x 1024 tokens
        act("act_train_8192x11008_bf16", 8192, 11008, "bf16", True),
        # hidden width left at 8/3 of 1024 without rounding: half rows of 5460 bytes
        act("act_train_4096x2730_fp16", 4096, 2730, "fp16", True),
        # one decoding step of a small batch through the whole block
        block("block_decode_8x4096_bf16", 8, 4096, 6912, "bf16", False),
        # a training step of the block at the smallest shape of the comparison benchmark, 8 x 128 tokens
        block("block_train_1024x2048_fp16", 1024, 2048, 3584, "fp16", True),
    ]


def spread(rng, low, high):
    """An integer of [low, high], spread over its logarithm."""
    return max(low, min(high, int(round(low * (high / low) ** rng.random()))))


def width(rng, low, high):
    """A row width: three in five a multiple of 64, the others any number."""
    cols = spread(rng, low, high)
    return max(64, (cols + 32) // 64 * 64) if rng.random() < 0.6 else cols


def draw(rng):
    dtype = rng.choice(("bf16", "bf16", "bf16", "fp16", "fp16", "fp32"))
    kind = rng.random()
    if kind < 0.5:  # norm, from a few rows to the largest listed
        train = rng.random() < 0.6
        cols = width(rng, 64, 16384)
        elements = spread(rng, 1 << 12, MOST_ELEMENTS // BYTES[dtype] // 2)
        c = norm("", max(1, min(1 << 20, elements // cols)), cols, dtype, train, rng.random() < 0.25)
    elif kind < 0.8:  # activation
        train = rng.random() < 0.6
        hidden = width(rng, 256, 16384)
        elements = spread(rng, 1 << 12, (1 << 28) // BYTES[dtype])
        c = act("", max(1, min(1 << 17, elements // hidden)), hidden, dtype, train)
    else:  # block: decoding steps of up to 64 tokens, training steps of 128 and more
        train = rng.random() < 0.4
        dtype = "bf16" if dtype == "fp32" else dtype
        d_model = spread(rng, 4, 32) * 128
        hidden = (d_model * rng.choice((5, 8)) // 3 + 255) // 256 * 256
        tokens = spread(rng, 128, 2048) if train else spread(rng, 1, 64)
        most = int(MOST_BLOCK_FLOPS // (18 * d_model * hidden))
        c = block("", min(tokens, most) if train else tokens, d_model, hidden, dtype, train)
    del c["name"]
    return c


def normal(shape, dtype, gen, outliers=False):
    t = torch.randn(shape, generator=gen, device="cuda", dtype=dtype)
    if outliers:
        step = 1 << 26
        flat = t.view(-1)
        for i in range(0, flat.numel(), step):  # in pieces: no second tensor of the size
            piece = flat[i:i + step]
            piece.mul_(1.0 + 99.0 * (torch.rand(piece.shape, generator=gen, device="cuda") < 0.01).to(dtype))
    return t


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype, train = DTYPES[case["dtype"]], case["train"]
    state = {"train": train}
    if case["path"] == "norm":
        with torch.device("cuda"):
            module = megagemm.RMSNorm(case["cols"], EPS).to(dtype)
        with torch.no_grad():
            module.weight.copy_(1.0 + 0.02 * normal((case["cols"],), torch.float32, gen))
        shape, out = (case["rows"], case["cols"]), (case["rows"], case["cols"])
        state.update(call=module, params=[module.weight])
    elif case["path"] == "act":
        hidden = case["hidden"]
        shape, out = (case["rows"], 2 * hidden), (case["rows"], hidden)
        state.update(call=lambda x: ops.swiglu(x, hidden), params=[])
    else:
        d_model, hidden = case["d_model"], case["hidden"]
        with torch.device("meta"):
            module = megagemm.MegaGemmTriton(d_model, multiple_of=1, hidden_multiple=hidden / d_model)
            if module.hidden != hidden:  # the quotient rounded down: the next number gives it
                module = megagemm.MegaGemmTriton(d_model, multiple_of=1, hidden_multiple=(hidden + 0.5) / d_model)
        module = module.to(dtype).to_empty(device="cuda")
        with torch.no_grad():
            for p in module.parameters():
                p.copy_(0.02 * normal(p.shape, dtype, gen))
        shape = out = (case["tokens"], d_model)
        state.update(call=module, params=list(module.parameters()))
    outliers = case.get("outliers", False)
    state["x"] = normal(shape, dtype, gen, outliers)
    if train:
        state["dy"] = normal(out, dtype, gen, outliers)
        state["x"].requires_grad_()
    return state


def run(state):
    x = state["x"]
    if not state["train"]:
        with torch.no_grad():
            return state["call"](x)
    x.grad = None
    for p in state["params"]:
        p.grad = None
    # the switch the package offers for loops of short layers: backward without a thread hand-over
    with megagemm.backward_on_calling_thread():
        y = state["call"](x)
        y.backward(state["dy"])
    return [y, x.grad, *[p.grad for p in state["params"]]]


def work(case):
    """Every input read once, every output written once: x is counted once although forward and
    backward of a training step each read it."""
    size, train = BYTES[case["dtype"]], case["train"]
    if case["path"] == "norm":
        n, c = case["rows"] * case["cols"], case["cols"]
        return {"bytes": (4 * n + 2 * c if train else 2 * n + c) * size, "flops": (12 if train else 4) * n}
    if case["path"] == "act":
        n = case["rows"] * case["hidden"]
        return {"bytes": (6 if train else 3) * n * size, "flops": (16 if train else 5) * n}
    t, d, h = case["tokens"], case["d_model"], case["hidden"]
    weights, io = 3 * d * h, 2 * t * d
    return {"bytes": (2 * (weights + io) if train else weights + io) * size, "flops": (18 if train else 6) * t * d * h}


def tolerance(case):
    # About four times what these paths measure against the same formula in float64 (worst output):
    # one rounding of a result is 1.7e-3 in all and 3.9e-3 at most (bf16), 2.1e-4 and 4.9e-4 (fp16),
    # 1.4e-7 and 3.5e-7 (fp32, column sums included); the block rounds between its stages as well,
    # 3.5e-3 and 1.3e-2 (bf16), 4.4e-4 and 2.5e-3 (fp16).
    if case["path"] == "block":
        return {"bf16": {"rel": 1.4e-2, "max": 5.2e-2}, "fp16": {"rel": 1.8e-3, "max": 1e-2}}[case["dtype"]]
    return {"bf16": {"rel": 7e-3, "max": 1.6e-2}, "fp16": {"rel": 9e-4, "max": 2e-3},
            "fp32": {"rel": 1e-6, "max": 4e-6}}[case["dtype"]]
