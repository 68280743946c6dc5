"""The fused filter gradient (sffft_filter_grad_*, torch.ops.sffft.filter_grad).

dk[h, j] = sum_b sum_{n >= j} dy[b, h, n] u[b, h, n - j] against an fp64 FFT correlation, at
every compiled length (teams within one wavefront, teams of several, both halves in a workgroup
or in the grid) and at batches and channel counts that leave a pair, a subset of the batch, a
channel slot or a batch split partly empty.
"""
import ctypes

import pytest
import torch

import sffft_amd as sf
from sffft_amd import torch_ops


def reference(u, dy):
    L = u.shape[-1]
    U, D = (torch.fft.rfft(x.double().cpu(), 2 * L) for x in (u, dy))
    return torch.fft.irfft((D * U.conj()).sum(0), 2 * L)[..., :L]


def test_argument_errors_need_no_gpu():
    lib = sf.lib()
    E = sf.SFFFT_EINVAL
    null = ctypes.c_void_p(0)
    u, dy, dk, w = (ctypes.c_void_p((1 << 40) + i * (1 << 34)) for i in range(4))
    # one half per workgroup from L = 4096 on: two parts to sum, and a workspace for them
    assert lib.sffft_filter_grad_work_bytes(8, 768, 1024) == 0
    need = lib.sffft_filter_grad_work_bytes(8, 768, 4096)
    assert need == 2 * 768 * 4096 * 4
    assert lib.sffft_filter_grad_work_bytes(8, 768, 1000) == lib.sffft_filter_grad_work_bytes(8, 0, 4096) == 0
    f = lib.sffft_filter_grad_f32
    assert f(null, dy, dk, w, need, 8, 768, 4096, null) == E
    assert f(u, dy, dk, w, need, 0, 768, 4096, null) == E
    assert f(u, dy, dk, w, need, 8, 768, 1000, null) == E
    assert f(u, dy, dk, w, need, 8, 768, 32768, null) == E                     # multi-pass lengths: not here
    assert f(u, dy, dk, null, 0, 8, 768, 4096, null) == E                      # workspace missing
    assert f(u, dy, dk, w, need - 4, 8, 768, 4096, null) == E                  # too small
    assert f(u, dy, u, w, need, 8, 768, 4096, null) == E                       # dk overlaps u
    assert f(u, dy, dk, dy, need, 8, 768, 4096, null) == E                     # workspace overlaps dy
    assert f(u, dy, ctypes.c_void_p((1 << 40) + (1 << 36) + 4), w, need, 8, 768, 4096, null) == E  # dk misaligned
    assert f(ctypes.c_void_p((1 << 40) + 2), dy, dk, w, need, 8, 768, 4096, null) == E


@pytest.mark.gpu
@pytest.mark.parametrize("io", ["fp32", "bf16"])
@pytest.mark.parametrize("L", sf.LENGTHS)
def test_matches_fp64(dev, L, io):
    g = torch.Generator(device=dev).manual_seed(L)
    for B, H in ((1, 1), (2, 5), (3, 2), (9, 7), (16, 3)):
        print(f"filter_grad B={B} H={H} L={L} {io}", flush=True)
        u, dy = (torch.randn(B, H, L, device=dev, generator=g).to(torch.bfloat16 if io == "bf16" else torch.float32)
                 for _ in range(2))
        dk = torch.ops.sffft.filter_grad(u, dy)
        ref = reference(u, dy)
        err = ((dk.double().cpu() - ref).norm(dim=1) / ref.norm(dim=1)).max().item()
        # fp32 transforms: three passes (u, dy, inverse) of at most four radix-16 stages, each with
        # about 8 roundings of 2^-24 on the way of a value: rms 2^-24 sqrt(3 * 4 * 8) = 6e-7, and
        # a factor of 3 for the worst channel
        assert err <= 2e-6, (B, H, err)
        assert torch.equal(dk, torch.ops.sffft.filter_grad(u, dy))


@pytest.mark.gpu
@pytest.mark.parametrize("L", sf.LENGTHS)
def test_rows_of_unequal_size(dev, L):
    """Two batch rows share a transform: the error of a row must not depend on its partner's size. Rows of
    u scaled by s and 1/s in turn and those of dy by the inverse leave every row's product as it is, so the
    bound is that of equal rows; rows of few samples and empty ones beside dense ones likewise."""
    g = torch.Generator(device=dev).manual_seed(L + 1)

    def check(u, dy, what):
        ref = reference(u, dy)
        err = ((torch.ops.sffft.filter_grad(u, dy).double().cpu() - ref).norm(dim=1) / ref.norm(dim=1)).max().item()
        assert err <= 2e-6, (what, err)  # as in test_matches_fp64

    for B, H in ((2, 3), (5, 4), (16, 3)):
        for s in (3.0, 30.0, 1000.0, 1e6):
            u, dy = (torch.randn(B, H, L, device=dev, generator=g) for _ in range(2))
            c = torch.tensor([s if b % 2 else 1 / s for b in range(B)], device=dev)[:, None, None]
            check(u * c, dy / c, (B, H, s))
            check(u / c, dy * c, (B, H, 1 / s))
    u, dy = (torch.randn(4, 3, L, device=dev, generator=g) for _ in range(2))
    u[0::2] = 0
    u[0::2, :, 5] = 1.0
    dy[1::2] /= 100 * L**0.5
    check(u, dy, "single samples")
    u[2] = 0
    u[1] = 0
    check(u, dy, "empty rows")


@pytest.mark.gpu
@pytest.mark.parametrize("L", [128, 256, 512, 1024, 2048, 16384])
def test_channels_are_independent(dev, L):
    """Unequal, infinite or NaN rows of one channel leave the other channels' bits alone, though channels
    share workgroups and, below L = 1024, wavefronts."""
    g = torch.Generator(device=dev).manual_seed(L + 2)
    u, dy = (torch.randn(5, 6, L, device=dev, generator=g) for _ in range(2))
    base = torch.ops.sffft.filter_grad(u, dy)
    for bad in (1e4, float("inf"), float("nan")):
        v = u.clone()
        v[1, 2] *= bad
        out = torch.ops.sffft.filter_grad(v, dy)
        keep = [h for h in range(6) if h != 2]
        assert torch.equal(out[keep], base[keep]), bad
        assert torch.isfinite(out[2]).all().item() == (bad == 1e4)


@pytest.mark.gpu
def test_any_alignment_and_stride(dev):
    """Rows at any element offset, and non-contiguous operands, as the composed path took them."""
    x = torch.randn(4 * 3 * 512 + 1, device=dev)
    u, dy = x[1:].view(4, 3, 512), x[:-1].view(4, 512, 3).transpose(1, 2)
    ref = reference(u, dy)
    assert ((torch_ops.filter_grad(u, dy).double().cpu() - ref).norm() / ref.norm()).item() <= 2e-6
    # an expanded output gradient, as sum().backward() makes
    one = torch.ones((), device=dev).expand(4, 3, 512)
    ref = reference(u, one)
    assert ((torch_ops.filter_grad(u, one).double().cpu() - ref).norm() / ref.norm()).item() <= 2e-6


@pytest.mark.gpu
@pytest.mark.parametrize("L", [128, 512, 1024, 4096])
def test_race_check_build_agrees(dev, L):
    """Bit-identical to the build whose wavefront-level LDS hand-offs are real waits."""
    B, H = 8, 64
    u, dy = (torch.randn(B, H, L, device=dev) for _ in range(2))
    out = []
    for lib in (sf.lib(), sf.load_library(sf.DEBUG_LIB_PATH)):
        dk = torch.empty(H, L, device=dev)
        wb = lib.sffft_filter_grad_work_bytes(B, H, L)
        work = torch.empty(max(wb, 16), dtype=torch.uint8, device=dev)
        p = [ctypes.c_void_p(t.data_ptr()) for t in (u, dy, dk, work)]
        s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        assert lib.sffft_filter_grad_f32(*p, wb, B, H, L, s) == 0
        torch.cuda.synchronize()
        out.append(dk)
    assert torch.equal(*out)


@pytest.mark.gpu
@pytest.mark.parametrize("composed", [False, True])
def test_second_derivative(dev, composed):
    """With the gradient's own gradient recorded, d(dk)/d(dy) is still there: through LongConv's backward
    pass, whose fused filter gradient has an adjoint of its own, and through torch_ops.filter_grad on a dy
    that records a gradient, which takes the composition of differentiable operators."""
    u, k = torch.randn(2, 3, 256, device=dev), torch.randn(3, 256, device=dev, requires_grad=True)
    dy = torch.randn(2, 3, 256, device=dev, requires_grad=True)
    if composed:
        dk = torch_ops.filter_grad(u, dy)
        ref = reference(u, dy.detach())
        assert ((dk.detach().double().cpu() - ref).norm() / ref.norm()).item() <= 5e-4  # fp16 operands
    else:
        (dk,) = torch.autograd.grad(torch_ops.LongConv()(u, k), k, dy, create_graph=True)
    c = torch.randn(3, 256, device=dev)
    (g,) = torch.autograd.grad((dk * c).sum(), dy)
    # d/d(dy) of sum_j c[h, j] dk[h, j]: the causal convolution of u with c
    U, C = torch.fft.rfft(u.double(), 512), torch.fft.rfft(c.double(), 512)
    ref = torch.fft.irfft(U * C, 512)[..., :256]
    assert ((g.double() - ref).norm() / ref.norm()).item() <= 5e-4
