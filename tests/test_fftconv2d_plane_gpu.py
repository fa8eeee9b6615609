"""Small 2D planes, whole images in LDS (csrc/fftconv2d_plane.h), against float64 FFT convolutions of the same inputs:
every transform size, odd and unaligned rows, filters to twice the image, a periodic first axis, per-sample filters,
several images a workgroup and a split batch, with and without the gates."""

import pytest
import torch

from nvsubquadratic_amd import _lib
from nvsubquadratic_amd.fftconv_hip import _nd_state_bytes, fftconv2d_bhl
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
    (2, 600, (11, 30), (22, 60), False, False),   # 32 x 64, filter twice the image
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


def _max_shares(B, H, S, K, periodic0):
    """Workgroups a channel's batch is split over at most: 2^25 points in all (plane2_max_split)."""
    def up(n):
        return 1 << max(4, (n - 1).bit_length())

    points = (S[0] if periodic0 else up(S[0] + (K[0] + 1) // 2)) * up(S[1] + (K[1] + 1) // 2)
    return max(1, min(B, (1 << 25) // max(1024, points) // H))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,H,S,K,periodic0", [
    (13, 8192, (14, 14), (27, 27), False),  # at most four shares
    (11, 8400, (16, 21), (15, 20), True),   # at most three
    (13, 2048, (30, 21), (59, 41), False),  # 64 x 64: four
])
def test_several_images_a_workgroup(B, H, S, K, periodic0, dtype):
    """A workgroup takes one image after the other: the next one's samples are loaded during a transform, the tile and
    the raw image are reused and the filter gradient is summed in registers; the last share is a ragged one.  Sampled
    channels against float64, with and without the gates, and a non-finite image, which must leave the outputs and
    input gradients of the other images of its channel as they are, bit for bit."""
    assert -(-B // _max_shares(B, H, S, K, periodic0)) >= 3
    gen = torch.Generator(device="cuda").manual_seed(H)
    x, g, kg, v = (torch.randn(B, H, *S, device="cuda", generator=gen).to(dtype) for _ in range(4))
    k = torch.randn(1, H, *K, device="cuda", generator=gen) / (K[0] * K[1]) ** 0.5
    s = torch.randn(H, device="cuda", generator=gen).to(dtype)
    ch = torch.tensor([0, 1, H // 2 + 3, H - 1], device="cuda")
    per = (periodic0, False)

    def plain(x, k, s):
        return mixed_fftconv2d_fp32_bhl(x, k, per, s) if periodic0 else fftconv2d_bhl(x, k, s)

    def gated(x, kg, v, k, s):
        return hyena_gated_fftconv2d_bhl(x, kg, v, k, s, "silu", "sigmoid", periodic=per)

    for op, ts in ((plain, (x, k, s)), (gated, (x, kg, v, k, s))):
        def call(x0):
            args = [t.clone().requires_grad_() for t in (x0, *ts[1:])]
            y = op(*args)
            return (y, *torch.autograd.grad(y, args, g))

        got = call(x)
        a6 = [t.index_select(0 if t.dim() == 1 else 1, ch).double().requires_grad_() for t in ts]
        if op is plain:
            y6 = _ref(*a6, periodic0)
        else:
            y6 = _ref(a6[0] * torch.nn.functional.silu(a6[1]), a6[3], a6[4], periodic0) * torch.sigmoid(a6[2])
        want = (y6, *torch.autograd.grad(y6, a6, g[:, ch].double()))
        _check([t.index_select(0 if t.dim() == 1 else 1, ch) for t in got], want, dtype)
        bad = x.clone()
        bad[1, 0, 3, 3] = float("inf")
        other = call(bad)
        keep = [b for b in range(B) if b != 1]
        for a, b in zip(got[:2], other[:2]):
            assert torch.equal(a[keep], b[keep]) and torch.equal(a[:, 1:], b[:, 1:])
        assert not torch.isfinite(other[0][1, 0]).any()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,H,S,K", [(16, 256, (53, 34), (27, 17)), (13, 256, (19, 48), (37, 95))])
def test_rectangles_whose_backward_runs_the_passes(B, H, S, K, dtype):
    """128 x 64 and 64 x 128 planes of the mixed-radix plan with many images: the backward, and a forward that keeps
    state for it, run that plan's passes; inference runs the plane."""
    gen = torch.Generator(device="cuda").manual_seed(B)
    x, g, kg, v = (torch.randn(B, H, *S, device="cuda", generator=gen).to(dtype) for _ in range(4))
    k = torch.randn(1, H, *K, device="cuda", generator=gen) / (K[0] * K[1]) ** 0.5
    s = torch.randn(H, device="cuda", generator=gen).to(dtype)
    assert _nd_state_bytes(x, k.view(H, *K), 1, 0, True) > 0
    ch = torch.tensor([0, 77, H - 1], device="cuda")
    cut = [t.index_select(0 if t.dim() == 1 else 1, ch).double().requires_grad_() for t in (x, k, s)]
    args = [t.clone().requires_grad_() for t in (x, k, s)]
    y = fftconv2d_bhl(*args)
    got = (y, *torch.autograd.grad(y, args, g))
    y6 = _ref(*cut, False)
    want = (y6, *torch.autograd.grad(y6, cut, g[:, ch].double()))
    _check([t.index_select(0 if t.dim() == 1 else 1, ch) for t in got], want, dtype)
    with torch.no_grad():
        _check([fftconv2d_bhl(x, k, s)[:, ch]], [y6.detach()], dtype)
    args = [t.clone().requires_grad_() for t in (x, kg, v, k, s)]
    y = hyena_gated_fftconv2d_bhl(*args, "silu", "sigmoid")
    got = (y, *torch.autograd.grad(y, args, g))
    cut = [t.index_select(0 if t.dim() == 1 else 1, ch).double().requires_grad_() for t in (x, kg, v, k, s)]
    y6 = _ref(cut[0] * torch.nn.functional.silu(cut[1]), cut[3], cut[4], False) * torch.sigmoid(cut[2])
    want = (y6, *torch.autograd.grad(y6, cut, g[:, ch].double()))
    _check([t.index_select(0 if t.dim() == 1 else 1, ch) for t in got], want, dtype)


def test_planes_keep_no_state():
    """A training forward of a plane allocates no spectrum for its backward (64 x 384 x 14^2 kept 200 MB)."""
    x = torch.empty(64, 384, 14, 14, device="cuda", dtype=torch.bfloat16)
    k = torch.empty(384, 27, 27, device="cuda")
    assert _nd_state_bytes(x, k, 1, 0, True) == 0
    lib, S, K = _lib.get_lib(), _lib.i64_array((14, 14)), _lib.i64_array((27, 27))
    need = [lib.nsq_fftconv_nd_workspace_bytes(2, 64, 384, S, K, 1, d) for d in (_lib.NSQ_DIR_FWD, _lib.NSQ_DIR_BWD)]
    assert need[1] == need[0] > 0  # a backward that transforms again needs no second spectrum
    big = torch.empty(2, 8, 200, 200, device="cuda")
    assert _nd_state_bytes(big, torch.empty(8, 200, 200, device="cuda"), 1, 0, True) > 0


def test_per_sample_filters_beyond_65535_images():
    """More images than a grid's second axis holds."""
    B, S, K = 66000, (5, 6), (3, 5)
    gen = torch.Generator(device="cuda").manual_seed(1)
    x, g = (torch.randn(B, 1, *S, device="cuda", generator=gen) for _ in range(2))
    k, s = torch.randn(B, 1, *K, device="cuda", generator=gen), torch.randn(1, device="cuda", generator=gen)
    args = [t.clone().requires_grad_() for t in (x, k, s)]
    y = fftconv2d_bhl(*args)
    got = (y, *torch.autograd.grad(y, args, g))
    a6 = [t.double().requires_grad_() for t in (x, k, s)]
    y6 = _ref(*a6, False)
    _check(got, (y6, *torch.autograd.grad(y6, a6, g.double())), torch.float32)


def test_images_do_not_mix():
    """A non-finite image leaves the outputs of the others as they are (one image a workgroup)."""
    x = torch.randn(6, 2, 14, 14, device="cuda")
    k = torch.randn(1, 2, 27, 27, device="cuda")
    clean = fftconv2d_bhl(x, k)
    x[2, 0, 3, 3] = float("inf")
    y = fftconv2d_bhl(x, k)
    keep = [0, 1, 3, 4, 5]
    assert torch.equal(y[keep], clean[keep]) and torch.equal(y[2, 1], clean[2, 1])
    assert not torch.isfinite(y[2, 0]).any()
