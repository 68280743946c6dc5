"""The anti-causal correlation (sffft_corr_*, torch.ops.sffft.corr): the convolution kernels with
conjugate DFT and twiddle tables on the convolution's own spectrum.

y[m] = sum_{n >= m} u[n] k[n - m] against an fp64 FFT, for every compiled plan (wave, workgroup and
multi-pass kernels, one and two sequences per transform, both accumulation modes), and as the
gradient it serves."""
import ctypes

import pytest
import torch

import sffft_amd as sf
from sffft_amd import torch_ops


def reference(u, k):
    L = u.shape[-1]
    U, K = torch.fft.rfft(u.double().cpu(), 2 * L), torch.fft.rfft(k.double().cpu(), 2 * L)
    return torch.fft.irfft(U * K.conj(), 2 * L)[..., :L]


def test_argument_errors_need_no_gpu():
    lib = sf.lib()
    null, good = ctypes.c_void_p(0), ctypes.c_void_p(1 << 20)
    p = sf.make_plan("64x32", 4, seqs=2)
    assert lib.sffft_corr_f32(null, good, good, 8, 768, 1024, ctypes.byref(p), null) == sf.SFFFT_EINVAL
    assert lib.sffft_corr_bf16(good, good, good, 7, 768, 1024, ctypes.byref(p), null) == sf.SFFFT_EINVAL  # B odd
    legacy = p.replace(cached=0)
    assert lib.sffft_corr_f32(good, good, good, 8, 768, 1024, ctypes.byref(legacy), null) == sf.SFFFT_ENOPLAN


@pytest.mark.gpu
@pytest.mark.parametrize("io", ["fp32", "bf16"])
@pytest.mark.parametrize("L", sf.LENGTHS + (32768,))
def test_matches_fp64(dev, L, io):
    B, H = 4, 5
    g = torch.Generator(device=dev).manual_seed(L)
    u = torch.randn(B, H, L, device=dev, generator=g).to(torch.bfloat16 if io == "bf16" else torch.float32)
    k = torch.randn(H, L, device=dev, generator=g) * torch.exp(-torch.arange(L, device=dev) * (8.0 / L))
    ref = reference(u, k)
    plans = [sf.default_plan(L)] if L > 16384 else sf.plans(L)
    for plan in plans:
        for acc in (0, 1) if plan.mode != 2 else (0,):
            p = torch_ops.plan_fields(plan.replace(acc=acc))
            kf = torch.ops.sffft.spectrum(k, p)
            y = torch.ops.sffft.corr(u, kf, p)
            err = ((y.double().cpu() - ref).norm() / ref.norm()).item()
            print(f"corr L={L} {io} {plan!r} acc={acc} rel_l2={err:.2e}", flush=True)
            # the bounds of the convolution itself (fp16 operands; the driver's caps for acc = 1)
            assert err <= {("fp32", 0): 5e-4, ("bf16", 0): 3e-3, ("fp32", 1): 2e-3, ("bf16", 1): 6e-3}[io, acc]


@pytest.mark.gpu
def test_in_kernel_tables_take_the_conjugate_spectrum(dev):
    u, k = torch.randn(2, 3, 1024, device=dev), torch.randn(3, 1024, device=dev)
    for plan in (sf.make_plan("64x32", 4, seqs=2), sf.make_plan("64x32", 4, seqs=2, mode=1)):
        p = torch_ops.plan_fields(plan.replace(cached=0))
        kf = torch.ops.sffft.spectrum(k, p)
        assert torch.equal(torch.ops.sffft.corr(u, kf, p), torch.ops.sffft.conv(u, torch.conj_physical(kf), p))


@pytest.mark.gpu
def test_opcheck_and_adjoint(dev):
    u, k = torch.randn(2, 3, 256, device=dev), torch.randn(3, 256, device=dev)
    p = torch_ops.plan_fields(sf.default_plan(256, "fp32", 2))
    kf = torch.ops.sffft.spectrum(k, p)
    torch.library.opcheck(torch.ops.sffft.corr.default, (u.clone().requires_grad_(), kf, p))
    torch.library.opcheck(torch.ops.sffft.longconv.default,
                          (u.clone().requires_grad_(), k.clone().requires_grad_(), kf, p))
    torch.library.opcheck(torch.ops.sffft.filter_grad.default, (u, u))
    v = u.clone().requires_grad_()
    (g,) = torch.autograd.grad(torch.ops.sffft.corr(v, kf, p), v, u)
    assert torch.equal(g, torch.ops.sffft.conv(u, kf, p))


@pytest.mark.gpu
def test_third_derivative(dev):
    """The filter gradient is linear in dy and its adjoint in dy linear in what comes back, so the
    gradients of gradients go on: <dk(u, dy), c> differentiated by dy is conv(u, c), and that by c
    the filter gradient again."""
    u, dy = torch.randn(2, 3, 256, device=dev), torch.randn(2, 3, 256, device=dev, requires_grad=True)
    k, c = (torch.randn(3, 256, device=dev, requires_grad=True) for _ in range(2))
    (dk,) = torch.autograd.grad(torch_ops.LongConv()(u, k), k, dy, create_graph=True)
    (g,) = torch.autograd.grad((dk * c).sum(), dy, create_graph=True)
    w = torch.randn_like(g)
    (dc,) = torch.autograd.grad((g * w).sum(), c)
    ref = torch.ops.sffft.filter_grad(u, w)
    assert ((dc - ref).norm() / ref.norm()).item() <= 1e-6


BACKWARD_CAPTURE = """
import torch
import sffft_amd as sf
from sffft_amd import torch_ops

L = 512
for plan in (sf.make_plan("64x16", 12, seqs=2, mode=1, channels=3), sf.default_plan(L), sf.long_plan("32x32x32")):
    L = plan.r0 * plan.r1 * plan.r2 // 2
    p = torch_ops.plan_fields(plan)
    u, k = torch.randn(2, 3, L, device="cuda"), torch.randn(3, L, device="cuda")
    kf = torch.ops.sffft.spectrum(k, p)
    torch.ops.sffft.conv(u, kf, p)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        y = torch.ops.sffft.corr(u, kf, p)
        dk = torch.ops.sffft.filter_grad(u, u)
    for _ in range(3):
        y.zero_()
        torch.ops.sffft.conv(u * 0.5, kf, p)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, torch.ops.sffft.corr(u, kf, p))
        assert torch.equal(dk, torch.ops.sffft.filter_grad(u, u))
print("captured")
"""


@pytest.mark.gpu
def test_backward_capture_after_an_eager_forward(dev):
    """The conjugate tables exist once the forward ones do: a capture of the backward pass needs no
    eager backward before it. In a process of its own, which has run no backward pass of any plan."""
    import os
    import subprocess
    import sys

    r = subprocess.run([sys.executable, "-c", BACKWARD_CAPTURE], capture_output=True, text=True, timeout=100,
                       cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
    assert r.returncode == 0 and "captured" in r.stdout, r.stderr[-2000:]
