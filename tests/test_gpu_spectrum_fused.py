"""The one-launch filter spectrum against the staged launches (padding, transform, gather), bit
for bit: every plan whose transform it takes, real, conjugate and complex filters, channel counts
that leave a workgroup partly empty. A spectrum buffer aligned to 8 bytes only takes the staged
launches, which gives the reference."""
import ctypes

import pytest
import torch

import sffft_amd as sf

pytestmark = pytest.mark.gpu


def plans(L):
    out = list(sf.plans(L))
    for r0 in (16, 32, 64):  # the multi-pass plans of the same length
        for row in ("16x16", "32x32", "64x32", "64x64"):
            p = sf.long_plan(f"{r0}x{row}")
            if p.r0 * p.r1 * p.r2 == 2 * L:
                out.append(p)
    return out


@pytest.mark.parametrize("L", [L for L in sf.LENGTHS if L <= 8192])
def test_fused_equals_staged(dev, L):
    lib = sf.lib()
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for H in (1, 7):
        kr, ki = torch.randn(H, L, device=dev), torch.randn(H, L, device=dev)
        n = H * 2 * L
        for p in plans(L):
            for fn, filters in (("sffft_spectrum", (kr,)), ("sffft_spectrum_conj", (kr,)),
                                ("sffft_spectrum_complex", (kr, ki))):
                if len(filters) == 2 and p.seqs != 2:
                    continue
                print(f"{fn} L={L} H={H} {p!r}", flush=True)
                got = []
                for off in (0, 1):
                    kf = torch.full((n + 1,), 7.0 + 3.0j, dtype=torch.complex64, device=dev)[off:off + n]
                    work = torch.empty(n, dtype=torch.complex64, device=dev)
                    a = [ctypes.c_void_p(t.data_ptr()) for t in (*filters, kf, work)]
                    rc = getattr(lib, fn)(*a[:-2], H, L, ctypes.byref(p), *a[-2:], s)
                    assert rc == 0
                    got.append(torch.view_as_real(kf))
                assert torch.equal(*got), (fn, H, repr(p))


def test_filter_inside_the_spectrum_buffer(dev):
    """The filter's rows may lie in the buffer that its spectrum overwrites, as before."""
    L, H = 1024, 5
    plan = sf.default_plan(L)
    k = torch.randn(H, L, device=dev)
    ref = sf.spectrum(k, L, plan)
    kf = torch.empty(H, 2 * L, dtype=torch.complex64, device=dev)
    inside = torch.view_as_real(kf).view(-1)[: H * L]
    inside.copy_(k.view(-1))
    work = torch.empty_like(kf)
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    a = [ctypes.c_void_p(t.data_ptr()) for t in (inside, kf, work)]
    assert sf.lib().sffft_spectrum(a[0], H, L, ctypes.byref(plan), a[1], a[2], s) == 0
    assert torch.equal(torch.view_as_real(kf), torch.view_as_real(ref))
