"""Small 2D planes, whole images in LDS (csrc/fftconv2d_plane.h), against float64 FFT convolutions of the same inputs:
every transform size, odd and unaligned rows, filters to twice the image, a periodic first axis, per-sample filters,
several images a workgroup and a split batch, with and without the gates."""

import pytest
import torch

from nvsubquadratic_amd.fftconv_hip import fftconv2d_bhl
from nvsubquadratic_amd.gated_fftconv_hip import hyena_gated_fftconv2d_bhl
from nvsubquadratic_amd.mixed_fftconv_hip import mixed_fftconv2d_fp32_bhl


pytestmark = pytest.mark.gpu

# One or two roundings to the I/O type a value (gated: four); fp32 FFTs of up to 2^14 points.
TOL = {torch.float32: 2e-6, torch.bfloat16: 1e-2, torch.float16: 1.5e-3}


def _ref(x, k, s, periodic0):
    S, K = x.shape[2:], k.shape[2:]
    F = [S[0] if periodic0 else S[0] + K[0], S[1] + K[1]]
    y = torch.fft.irfftn(torch.fft.rfftn(x, s=F) * torch.fft.rfftn(k, s=F), s=F)
    y = torch.roll(y, -((K[0] - 1) // 2), dims=2) if periodic0 else y[:, :, K[0] // 2:K[0] // 2 + S[0]]
    return y[..., K[1] // 2:K[1] // 2 + S[1]] + s.view(1, -1, 1, 1) * x


def _check(got, want, dtype):
    # The last gradient, the shortcut's, is one sum per channel of every g x (gated: dy1 z, RMS about 1/4), whose size
    # is sqrt(count) / 4 or more unless it cancels; its rounding error follows the terms, not the sum.
    for i, (a, r) in enumerate(zip(got, want)):
        size = r.norm().item()
        if i == len(want) - 1:
            size = max(size, (got[0].numel() ** 0.5) / 4)
        err = (a.double() - r).norm().item() / size
        assert err < TOL[dtype], (i, err)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,H,S,K,periodic0,film", [
    (1, 1, (1, 1), (1, 1), False, False),
    (3, 2, (7, 7), (13, 13), False, False),       # 16 x 16 grown to one wave
    (5, 3, (9, 20), (5, 39), False, False),       # 16 x 64: wider than half the row
    (70, 2, (14, 14), (27, 27), False, False),    # 32 x 32, batch split over workgroups
    (2, 600, (11, 30), (22, 60), False, False),   # 32 x 64, filter twice the image, two images a workgroup
    (2, 3, (16, 60), (16, 61), True, False),      # periodic 16 x 128
    (4, 2, (64, 16), (64, 31), True, False),      # periodic 64 x 32
    (3, 2, (40, 5), (41, 9), False, False),       # 64 x 16
    (2, 3, (33, 31), (47, 33), False, True),      # 64 x 64, per-sample filters
    (2, 2, (60, 7), (9, 7), False, False),        # 128 x 16, filter shorter than the image
    (2, 2, (128, 24), (127, 17), True, False),    # periodic 128 x 64
    (2, 2, (85, 85), (85, 85), False, False),     # 128 x 128
    (2, 2, (101, 100), (50, 56), False, False),
])
def test_plane_against_float64(B, H, S, K, periodic0, film, dtype):
    gen = torch.Generator(device="cuda").manual_seed(S[0] * 1000 + S[1])
    x, g, kg, v = (torch.randn(B, H, *S, device="cuda", generator=gen).to(dtype) for _ in range(4))
    k = torch.randn(B if film else 1, H, *K, device="cuda", generator=gen) / (K[0] * K[1]) ** 0.5
    s = torch.randn(H, device="cuda", generator=gen).to(dtype)

    def conv(*a):
        if periodic0:
            return mixed_fftconv2d_fp32_bhl(a[0], a[1], (True, False), a[2])
        return fftconv2d_bhl(*a)

    args = [t.clone().requires_grad_() for t in (x, k, s)]
    y = conv(*args)
    got = (y, *torch.autograd.grad(y, args, g))
    a6 = [t.double().requires_grad_() for t in (x, k, s)]
    y6 = _ref(*a6, periodic0)
    _check(got, (y6, *torch.autograd.grad(y6, a6, g.double())), dtype)
    with torch.no_grad():
        assert torch.equal(conv(x, k, s), y)

    args = [t.clone().requires_grad_() for t in (x, kg, v, k, s)]
    y = hyena_gated_fftconv2d_bhl(*args, "silu", "sigmoid", periodic=(periodic0, False))
    got = (y, *torch.autograd.grad(y, args, g))
    a6 = [t.double().requires_grad_() for t in (x, kg, v, k, s)]
    y6 = _ref(a6[0] * torch.nn.functional.silu(a6[1]), a6[3], a6[4], periodic0) * torch.sigmoid(a6[2])
    _check(got, (y6, *torch.autograd.grad(y6, a6, g.double())), dtype)


def test_images_do_not_mix():
    """A non-finite image leaves the outputs and input gradients of the others as they are."""
    x = torch.randn(6, 2, 14, 14, device="cuda")
    k = torch.randn(1, 2, 27, 27, device="cuda")
    clean = fftconv2d_bhl(x, k)
    x[2, 0, 3, 3] = float("inf")
    y = fftconv2d_bhl(x, k)
    keep = [0, 1, 3, 4, 5]
    assert torch.equal(y[keep], clean[keep]) and torch.equal(y[2, 1], clean[2, 1])
    assert not torch.isfinite(y[2, 0]).any()
