"""The four-launch 2-D circular convolution of real images (sizes of its path) and the complex
transforms (sizes outside it) against an fp64 FFT convolution: single and several stages along
either axis, images that leave a workgroup partly empty, every image on its own."""
import pytest
import torch

import sffft_amd as sf

pytestmark = pytest.mark.gpu


def reference(u, k):
    U, K = torch.fft.rfft2(u.double().cpu()), torch.fft.rfft2(k.double().cpu())
    return torch.fft.irfft2(U * K, s=u.shape[-2:])


@pytest.mark.parametrize("N0,N1", [(16, 32), (32, 32), (16, 64), (64, 128), (128, 256), (256, 512), (512, 32),
                                   (32, 1024), (16, 2048), (16, 4096), (512, 512),
                                   (8, 32), (16, 16), (1024, 32), (16, 8192)])  # the last four: complex transforms
def test_matches_fp64(dev, N0, N1):
    g = torch.Generator(device=dev).manual_seed(N0 * N1)
    for B, H in ((1, 1), (2, 3), (3, 1)):
        print(f"circconv2d B={B} H={H} {N0}x{N1}", flush=True)
        u = torch.randn(B, H, N0, N1, device=dev, generator=g)
        k = torch.randn(H, N0, N1, device=dev, generator=g)
        y = sf.circconv2d(u, k)
        ref = reference(u, k)
        # complex64 between launches, fp64 within: at most a dozen roundings of 2^-24, rms 2e-7
        assert ((y.double().cpu() - ref).norm() / ref.norm()).item() <= 2e-7
        assert torch.equal(y, sf.circconv2d(u, k))


def test_images_do_not_mix(dev):
    u, k = torch.randn(2, 2, 64, 64, device=dev), torch.randn(2, 64, 64, device=dev)
    y = sf.circconv2d(u, k)
    v = u.clone()
    v[1, 0, 3, 5] = float("nan")
    z = sf.circconv2d(v, k)
    assert torch.isnan(z[1, 0]).all()
    for b, h in ((0, 0), (0, 1), (1, 1)):
        assert torch.equal(z[b, h], y[b, h])


def test_delta_shifts(dev):
    """A filter of one sample shifts the image, along both axes and around the ends."""
    u = torch.randn(1, 1, 32, 64, device=dev)
    k = torch.zeros(1, 32, 64, device=dev)
    k[0, 5, 63] = 1.0
    y = sf.circconv2d(u, k)
    assert (y - torch.roll(u, (5, 63), (2, 3))).abs().max().item() <= 1e-5
