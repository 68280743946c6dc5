"""The workloads that the framework's performance is measured on, through its public entry points.

A case is a dict of plain values. Its "kind" says which call a pass makes:

- "conv":   causal convolution with a prepared filter spectrum (`torch.ops.sffft.conv`), the
            forward pass of an inference or evaluation step, at every length the plans cover
            (L = 128..16384 in one launch, 32768..131072 in several);
- "train":  a training step of a long-convolution layer (`LongConv`): the filter is made from
            its parameters, the layer runs, and the gradients of the input and of the filter
            parameters come back;
- "fft":    a batched complex transform (`sffft_amd.fft`), either direction;
- "conv2d": a 2-D circular convolution of images (`sffft_amd.circconv2d`).

`draw` gives further cases of the same ranges: batches 1 to 16, even and odd, channel counts that
are no multiple of anything, both I/O types.
"""
import math

import torch

import sffft_amd as sf
from sffft_amd import torch_ops


def listed():
    return [
        # one short sequence at a time: an interactive caller, bound by launch and latency
        {"name": "conv_one_128", "kind": "conv", "io": "fp32", "B": 1, "H": 256, "L": 128},
        # the benchmark batch (8 sequences of 768 channels) at the length the benchmark is quoted on
        {"name": "conv_1024_fp32", "kind": "conv", "io": "fp32", "B": 8, "H": 768, "L": 1024},
        # the same batch at the longest two-stage length, 16-bit activations
        {"name": "conv_2048_bf16", "kind": "conv", "io": "bf16", "B": 8, "H": 768, "L": 2048},
        # an odd batch and a ragged channel count: the last batch of an evaluation
        {"name": "conv_4096_odd", "kind": "conv", "io": "fp32", "B": 3, "H": 859, "L": 4096},
        {"name": "conv_8192_fp32", "kind": "conv", "io": "fp32", "B": 8, "H": 768, "L": 8192},
        # the long-filter configuration of the benchmark
        {"name": "conv_16384_bf16", "kind": "conv", "io": "bf16", "B": 4, "H": 1536, "L": 16384},
        # long context, beyond what one compute unit holds
        {"name": "conv_65536_bf16", "kind": "conv", "io": "bf16", "B": 2, "H": 768, "L": 65536},
        # training steps: the benchmark batch, a ragged 16-bit one, an odd batch of long sequences
        {"name": "train_1024_fp32", "kind": "train", "io": "fp32", "B": 8, "H": 768, "L": 1024},
        {"name": "train_4096_bf16", "kind": "train", "io": "bf16", "B": 6, "H": 513, "L": 4096},
        {"name": "train_8192_odd", "kind": "train", "io": "fp32", "B": 5, "H": 320, "L": 8192},
        # standalone transforms: long sequences in one pass, and images through the 2-D convolution
        {"name": "fft_16384", "kind": "fft", "batch": 768, "N": 16384, "inverse": True},
        {"name": "conv2d_256", "kind": "conv2d", "B": 8, "H": 16, "N0": 256, "N1": 256},
    ]


# The largest batch of each kind, in samples (B * H * L, or points): that of its listed cases.
MOST = {"conv": 4 * 1536 * 16384, "train": 6 * 513 * 4096, "fft": 768 * 16384, "conv2d": 8 * 16 * 256 * 256}


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["conv"] * 6 + ["train"] * 4 + ["fft", "conv2d"])
    if kind in ("conv", "train"):
        while True:
            io, B, H = rng.choice(["fp32", "bf16"]), rng.randint(1, 16), _log_int(rng, 24, 1536)
            L = 1 << rng.randint(7, 16 if kind == "conv" else 14)
            if L > 16384:
                B += B % 2  # lengths beyond 16384 take pairs of sequences
            if MOST[kind] // 4000 <= B * H * L <= MOST[kind]:
                return {"kind": kind, "io": io, "B": B, "H": H, "L": L}
    if kind == "fft":
        while True:
            batch, N = _log_int(rng, 1, 4096), 1 << rng.randint(6, 20)
            if MOST[kind] // 1000 <= batch * N <= MOST[kind]:
                return {"kind": kind, "batch": batch, "N": N, "inverse": rng.choice([False, True])}
    while True:
        B, H = rng.randint(1, 9), rng.randint(1, 24)
        N0, N1 = 1 << rng.randint(5, 9), 1 << rng.randint(5, 9)
        if MOST[kind] // 100 <= B * H * N0 * N1 <= MOST[kind]:
            return {"kind": kind, "B": B, "H": H, "N0": N0, "N1": N1}


def _inputs(case, seed):
    """The case's tensors, from the seed alone."""
    g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape, dtype=torch.float32):
        return torch.randn(*shape, device="cuda", dtype=dtype, generator=g)

    if case["kind"] == "fft":
        return {"x": normal(case["batch"], case["N"], dtype=torch.complex64)}
    if case["kind"] == "conv2d":
        P = case["N0"] * case["N1"]
        return {"u": normal(case["B"], case["H"], case["N0"], case["N1"]),
                "k": normal(case["H"], case["N0"], case["N1"]) / math.sqrt(P)}
    B, H, L = case["B"], case["H"], case["L"]
    io = torch.bfloat16 if case["io"] == "bf16" else torch.float32
    n = torch.arange(L, device="cuda", dtype=torch.float32)
    # activations of unit variance; filters that decay over 1/32 to 1/2 of the sequence, channel
    # by channel, as a filter network's modulation window makes them
    tau = L * torch.logspace(-5, -1, H, base=2.0, device="cuda")
    d = {"u": normal(B, H, L).to(io), "window": torch.exp(-n[None, :] / tau[:, None]), "w": normal(H, L) / math.sqrt(L)}
    if case["kind"] == "train":
        d["dy"] = normal(B, H, L).to(io)
    return d


def prepare(case, seed):
    s = dict(_inputs(case, seed), case=case)
    if case["kind"] == "conv":
        plan = sf.default_plan(case["L"], case["io"], case["B"])
        s["plan"] = torch_ops.plan_fields(plan)
        s["kf"] = torch.ops.sffft.spectrum(s.pop("w") * s.pop("window"), s["plan"])
    elif case["kind"] == "train":
        s["layer"] = torch_ops.LongConv()
        s["u"].requires_grad_()
        s["w"].requires_grad_()
    return s


def run(state):
    kind = state["case"]["kind"]
    if kind == "conv":
        return torch.ops.sffft.conv(state["u"], state["kf"], state["plan"])
    if kind == "train":
        k = state["w"] * state["window"]  # the filter of this step, from its parameters
        y = state["layer"](state["u"], k)
        du, dw = torch.autograd.grad(y, (state["u"], state["w"]), state["dy"])
        return {"y": y.detach(), "du": du, "dw": dw}
    if kind == "fft":
        N = state["case"]["N"]
        inverse = state["case"]["inverse"]
        return sf.fft(state["x"], inverse=inverse, scale=1.0 / N if inverse else 1.0)
    return sf.circconv2d(state["u"], state["k"])


def work(case):
    if case["kind"] == "fft":
        n = case["batch"] * case["N"]
        return {"bytes": 16 * n, "flops": 5 * n * math.log2(case["N"])}
    if case["kind"] == "conv2d":
        P = case["N0"] * case["N1"]
        img = case["B"] * case["H"]
        # real transforms of the images both ways and of the filters one way, and the product
        return {"bytes": 4 * P * (2 * img + case["H"]),
                "flops": 2.5 * P * math.log2(P) * (2 * img + case["H"]) + 3 * P * img}
    B, H, L = case["B"], case["H"], case["L"]
    s = 2 if case["io"] == "bf16" else 4
    rows, N = B * H, 2 * L
    fft = 2.5 * N * math.log2(N)  # a real transform of the zero-padded row
    if case["kind"] == "conv":
        # u and y once, the non-redundant half of the complex64 spectrum once
        return {"bytes": 2 * rows * L * s + 8 * H * L, "flops": rows * (2 * fft + 6 * L)}
    # u, dy, y and du once, the parameters and window read and the parameters' gradient written;
    # transforms of u, dy and the filter, inverse transforms of y, du and the filter's gradient
    return {"bytes": 4 * rows * L * s + 12 * H * L, "flops": rows * (4 * fft + 18 * L) + 2 * H * fft}


def tolerance(case):
    # The convolution kernels' operands are fp16 and their sums fp32: 3.3e-4 to 4.7e-4 from 64
    # bits with fp32 input and output, 1.7e-3 with bf16 ones (the rounding of the result). The
    # transforms run in fp64 with complex64 between their stages: 5e-8 to 9e-8.
    if case["kind"] in ("conv", "train"):
        return {"rel": 1.8e-3 if case["io"] == "fp32" else 7e-3}
    return {"rel": 4e-7}


def _causal(a, b, L):
    """IDFT(DFT(a) b) for rows of length L zero-padded to 2L, in 64 bits."""
    return torch.fft.irfft(torch.fft.rfft(a, 2 * L) * b, 2 * L)[..., :L]


def exact(case, seed):
    d = _inputs(case, seed)
    if case["kind"] == "fft":
        x = d["x"].to(torch.complex128)
        return torch.fft.ifft(x) if case["inverse"] else torch.fft.fft(x)
    if case["kind"] == "conv2d":
        K = torch.fft.rfft2(d["k"].double())
        return torch.fft.irfft2(torch.fft.rfft2(d["u"].double()) * K, s=(case["N0"], case["N1"]))
    B, H, L = case["B"], case["H"], case["L"]
    out = {"y": torch.empty(B, H, L, device="cuda", dtype=torch.float64)}
    if case["kind"] == "train":
        out["du"] = torch.empty_like(out["y"])
        out["dw"] = torch.empty(H, L, device="cuda", dtype=torch.float64)
    # the filter is the product of its parameters and window in the layer's own type
    k = d["w"] * d["window"]
    step = max(1, (1 << 25) // (B * L))  # channels at a time
    for h in range(0, H, step):
        c = slice(h, h + step)
        u = d["u"][:, c].double()
        K = torch.fft.rfft(k[c].double(), 2 * L)
        out["y"][:, c] = _causal(u, K, L)
        if case["kind"] == "train":
            dy = d["dy"][:, c].double()
            out["du"][:, c] = _causal(dy, K.conj(), L)
            corr = _causal(dy, torch.fft.rfft(u, 2 * L).conj(), L)
            out["dw"][c] = corr.sum(0) * d["window"][c].double()
    return out if case["kind"] == "train" else out["y"]
