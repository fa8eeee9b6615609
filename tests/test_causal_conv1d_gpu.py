"""GPU parity of the HIP direct causal conv and B2B block against the CPU oracle.

Mirrors tests/ops/test_causal_conv1d_custom.py (forward :63-110 incl. bias and
silu; B2B shape/finite :112-133, here extended to values) and
tests/modules/test_subq_ops_causal_conv1d.py (module forward/backward and the
construction errors :74-148).  Tolerances: the reference's atol=1e-3/rtol=1e-4
elementwise for fp32 plus rel-L2 <= 1e-4 (fp32) / 2e-2 (bf16).
"""

import numpy as np
import os
import pytest
import torch

from nvsubquadratic_amd.causal_conv1d_hip import b2b_causal_conv1d, causal_conv1d
from nvsubquadratic_amd.modules import HipCausalConv1d
from oracle.direct_ref import b2b_causal_conv1d_torch, causal_conv1d_torch
from oracle.fftconv_ref import rel_l2


pytestmark = pytest.mark.gpu
GOLDEN = os.path.join(os.path.dirname(__file__), "golden", "direct1d.npz")


@pytest.mark.parametrize("C,L,K", [(16, 64, 3), (36, 256, 3), (64, 128, 7), (8, 5000, 128), (4, 3000, 256), (3, 7, 9)])
@pytest.mark.parametrize("with_bias", [False, True])
@pytest.mark.parametrize("act", ["identity", "silu"])
def test_forward_backward_vs_reference(C, L, K, with_bias, act):
    torch.manual_seed(42)
    x = torch.randn(2, C, L, requires_grad=True)
    w = torch.randn(C, K, requires_grad=True)
    b = torch.randn(C, requires_grad=True) if with_bias else None
    y_ref = causal_conv1d_torch(x, w, b, act)
    g = torch.randn_like(y_ref)
    y_ref.backward(g)
    xg = x.detach().cuda().requires_grad_(True)
    wg = w.detach().cuda().requires_grad_(True)
    bg = b.detach().cuda().requires_grad_(True) if with_bias else None
    y = causal_conv1d(xg, wg, bg, act)
    y.backward(g.cuda())
    torch.testing.assert_close(y.cpu(), y_ref, atol=1e-3, rtol=1e-4)
    assert rel_l2(y_ref, y) < 1e-4
    assert rel_l2(x.grad, xg.grad) < 1e-4
    assert rel_l2(w.grad, wg.grad) < 1e-4
    if with_bias:
        assert rel_l2(b.grad, bg.grad) < 1e-4


def test_golden_fixtures():
    d = np.load(GOLDEN)
    for i in range(int(d["n_direct"])):
        x, w, b = (torch.tensor(d[f"d{i}_{n}"], dtype=torch.float32, device="cuda") for n in ("x", "w", "b"))
        assert rel_l2(d[f"d{i}_y"], causal_conv1d(x, w, b)) < 1e-5
        assert rel_l2(d[f"d{i}_y_silu"], causal_conv1d(x, w, b, "silu")) < 1e-5
    for i in range(int(d["n_b2b"])):
        x, wp, wm, sk = (torch.tensor(d[f"b{i}_{n}"], dtype=torch.float32, device="cuda")
                         for n in ("x", "wp", "wm", "skip"))
        assert rel_l2(d[f"b{i}_y"], b2b_causal_conv1d(x, wp, wm, sk)) < 1e-5


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_low_precision_io(dtype):
    torch.manual_seed(1)
    x = torch.randn(2, 32, 700, dtype=dtype)
    w = torch.randn(32, 4)
    y = causal_conv1d(x.cuda(), w.cuda(), None, "silu")
    assert y.dtype == dtype
    assert rel_l2(causal_conv1d_torch(x.float(), w, None, "silu"), y) < 2e-2


def test_batch_and_tile_independence_bitwise():
    torch.manual_seed(2)
    x = torch.randn(3, 8, 5000, device="cuda")
    w = torch.randn(8, 31, device="cuda")
    y = causal_conv1d(x, w)
    y1 = causal_conv1d(x[1:2].contiguous(), w)
    assert torch.equal(y[1:2], y1)


@pytest.mark.parametrize("K", [2, 3, 4, 5, 8, 9, 17, 33, 128, 256])
def test_halo_before_row_start_reads_zero(K):
    """Outputs whose window reaches before position 0 see only the zero padding.

    Rows are staged through raw buffers; positions before the row start must read
    as zero however the compiler splits the element offset (a negative offset plus
    a folded immediate can wrap back into range).
    """
    torch.manual_seed(11)
    B, C, L = 3, 5, 300
    x = torch.randn(B, C, L, requires_grad=True)
    w = torch.randn(C, K, requires_grad=True)
    y_ref = causal_conv1d_torch(x, w, None)
    g = torch.randn_like(y_ref)
    y_ref.backward(g)
    xg, wg = x.detach().cuda().requires_grad_(True), w.detach().cuda().requires_grad_(True)
    y = causal_conv1d(xg, wg)
    y.backward(g.cuda())
    assert rel_l2(y_ref[..., :K], y[..., :K]) < 1e-5
    assert rel_l2(y_ref, y) < 1e-5
    assert rel_l2(x.grad, xg.grad) < 1e-5
    assert rel_l2(w.grad, wg.grad) < 1e-5


@pytest.mark.parametrize("K", [1, 2, 3, 4, 5, 6, 7, 8, 9, 12, 15, 16])
@pytest.mark.parametrize("L", [1, 13, 4103, 18432])
def test_short_taps_backward_across_tiles_and_batches(K, L):
    """Up to 16 taps the whole backward is one register-resident pass whose
    weight/bias partials cover runs of (batch, tile) pairs; with 3 batches and
    up to 9 tiles per row those runs cross row ends.  Ragged lengths take the
    element-load path, multiples of 8 the vector path."""
    torch.manual_seed(100 + K)
    B, C = 3, 6
    x = torch.randn(B, C, L, dtype=torch.float64, requires_grad=True)
    w = torch.randn(C, K, dtype=torch.float64, requires_grad=True)
    b = torch.randn(C, dtype=torch.float64, requires_grad=True)
    y_ref = causal_conv1d_torch(x, w, b, "silu")
    g = torch.randn_like(y_ref)
    y_ref.backward(g)
    xg = x.detach().float().cuda().requires_grad_(True)
    wg = w.detach().float().cuda().requires_grad_(True)
    bg = b.detach().float().cuda().requires_grad_(True)
    y = causal_conv1d(xg, wg, bg, "silu")
    y.backward(g.float().cuda())
    assert rel_l2(y_ref, y.double()) < 1e-5
    assert rel_l2(x.grad, xg.grad.double()) < 1e-5
    assert rel_l2(w.grad, wg.grad.double()) < 1e-5
    assert rel_l2(b.grad, bg.grad.double()) < 1e-5


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("K", [4, 7, 13])
def test_short_taps_backward_low_precision_io(dtype, K):
    torch.manual_seed(5)
    x = torch.randn(2, 16, 3000).to(dtype)
    w = torch.randn(16, K)
    b = torch.randn(16)
    xr = x.float().requires_grad_(True)
    wr, br = w.clone().requires_grad_(True), b.clone().requires_grad_(True)
    y_ref = causal_conv1d_torch(xr, wr, br, "silu")
    g = torch.randn_like(y_ref).to(dtype)
    y_ref.backward(g.float())
    xg = x.cuda().requires_grad_(True)
    wg, bg = w.cuda().requires_grad_(True), b.cuda().requires_grad_(True)
    y = causal_conv1d(xg, wg, bg, "silu")
    y.backward(g.cuda())
    assert xg.grad.dtype == dtype
    assert rel_l2(y_ref, y.float()) < 2e-2
    assert rel_l2(xr.grad, xg.grad.float()) < 2e-2
    assert rel_l2(wr.grad, wg.grad) < 2e-2
    assert rel_l2(br.grad, bg.grad) < 2e-2


@pytest.mark.parametrize("K", [15, 16, 17, 33, 34, 65, 66, 129, 130, 256])
@pytest.mark.parametrize("act", ["identity", "silu"])
def test_tap_counts_across_matrix_core_plans(K, act):
    """Direct conv above 16 taps runs as banded Toeplitz MFMA products (forward,
    the silu pre-activation gradient, the input-gradient correlation and the
    weight gradient, on bands of 12, 20, 36 or 68 steps); up to 16 taps the
    register-window kernels run.  Ragged length, bias, two batches; forward and
    gradients against a float64 reference."""
    torch.manual_seed(200 + K)
    B, C, L = 2, 3, 4700
    x = torch.randn(B, C, L, dtype=torch.float64, requires_grad=True)
    w = (torch.randn(C, K, dtype=torch.float64) / K ** 0.5).requires_grad_(True)
    b = torch.randn(C, dtype=torch.float64, requires_grad=True)
    y_ref = causal_conv1d_torch(x, w, b, act)
    g = torch.randn_like(y_ref)
    y_ref.backward(g)
    xg, wg, bg = (t.detach().float().cuda().requires_grad_(True) for t in (x, w, b))
    y = causal_conv1d(xg, wg, bg, act)
    y.backward(g.float().cuda())
    assert rel_l2(y_ref, y.detach().double()) < 1e-5
    assert rel_l2(y_ref[..., :K + 2], y.detach()[..., :K + 2].double()) < 1e-5
    for ref, got in ((x, xg), (w, wg), (b, bg)):
        assert rel_l2(ref.grad, got.grad.double()) < 1e-5
    assert rel_l2(x.grad[..., -K - 2:], xg.grad[..., -K - 2:].double()) < 1e-5


@pytest.mark.parametrize("Kp,Km", [(2, 3), (4, 4), (5, 7), (8, 1), (1, 9), (7, 33)])
def test_b2b_halo_before_row_start_reads_zero(Kp, Km):
    """B2B forward and backward near the row start for several halo widths."""
    torch.manual_seed(12)
    B, C, L = 2, 3, 200
    x = torch.randn(B, 3 * C, L, requires_grad=True)
    wp = torch.randn(3 * C, Kp, requires_grad=True)
    wm = torch.randn(C, Km, requires_grad=True)
    sk = torch.randn(C, requires_grad=True)
    y_ref = b2b_causal_conv1d_torch(x, wp, wm, sk)
    g = torch.randn_like(y_ref)
    y_ref.backward(g)
    args = [t.detach().cuda().requires_grad_(True) for t in (x, wp, wm, sk)]
    y = b2b_causal_conv1d(*args)
    y.backward(g.cuda())
    assert rel_l2(y_ref, y) < 1e-4
    assert rel_l2(x.grad[..., :Kp + Km], args[0].grad[..., :Kp + Km]) < 1e-4
    for ref, got in zip((x, wp, wm, sk), args):
        assert rel_l2(ref.grad, got.grad) < 1e-4


# --------------------------------------------------------------------------- B2B
@pytest.mark.parametrize("B,C,L,Kp,Km", [(2, 16, 64, 3, 3), (4, 32, 128, 4, 4), (2, 16, 128, 8, 8),
                                         (1, 8, 3000, 3, 128), (2, 4, 257, 5, 256)])
def test_b2b_forward_backward(B, C, L, Kp, Km):
    torch.manual_seed(42)
    x = torch.randn(B, 3 * C, L, requires_grad=True)
    wp = (torch.randn(3 * C, Kp) / Kp ** 0.5).requires_grad_(True)
    wm = (torch.randn(C, Km) / Km ** 0.5).requires_grad_(True)
    sk = torch.randn(C, requires_grad=True)
    y_ref = b2b_causal_conv1d_torch(x, wp, wm, sk)
    g = torch.randn_like(y_ref)
    y_ref.backward(g)
    args = [t.detach().cuda().requires_grad_(True) for t in (x, wp, wm, sk)]
    y = b2b_causal_conv1d(*args)
    assert y.shape == (B, C, L) and torch.isfinite(y).all()
    y.backward(g.cuda())
    assert rel_l2(y_ref, y) < 1e-4
    for ref, got in zip((x, wp, wm, sk), args):
        assert rel_l2(ref.grad, got.grad) < 1e-4


def test_b2b_backward_every_channel_many_workgroups():
    """The fused adjoint (projection taps <= 4, matrix-core mixer) with many workgroups per CU in
    flight, fp32, checked channel by channel: each thread's k / v windows read x words that
    other waves stage, so a missing barrier there corrupts runs of positions in a few
    channels only -- invisible in one rel-L2 over all channels, caught per row here."""
    torch.manual_seed(7)
    B, C, L, Kp, Km = 4, 512, 8192, 3, 128
    x = torch.randn(B, 3 * C, L, requires_grad=True)
    wp = (torch.randn(3 * C, Kp) / Kp ** 0.5).requires_grad_(True)
    wm = (torch.randn(C, Km) / Km ** 0.5).requires_grad_(True)
    sk = torch.randn(C, requires_grad=True)
    y_ref = b2b_causal_conv1d_torch(x, wp, wm, sk)
    g = torch.randn_like(y_ref)
    y_ref.backward(g)
    args = [t.detach().cuda().requires_grad_(True) for t in (x, wp, wm, sk)]
    b2b_causal_conv1d(*args).backward(g.cuda())
    gx = args[0].grad.cpu().double()
    rx = x.grad.double()
    err_x = ((gx - rx).norm(dim=2) / rx.norm(dim=2)).max().item()  # worst (batch, channel) row
    err_wp = ((args[1].grad.cpu().double() - wp.grad.double()).norm(dim=1) / wp.grad.double().norm(dim=1)).max().item()
    assert err_x < 1e-4, err_x
    assert err_wp < 1e-4, err_wp
    for ref, got in zip((wm, sk), args[2:]):
        assert rel_l2(ref.grad, got.grad) < 1e-4


@pytest.mark.parametrize("Km", [15, 16, 17, 33, 34, 65, 66, 128, 129, 130, 256])
def test_b2b_mixer_tap_counts_across_matrix_core_plans(Km):
    """Mixer tap counts on both sides of each matrix-core step-count boundary.

    From 16 taps the mixer conv (forward), its adjoint correlation and its
    weight gradient run as banded Toeplitz products on the matrix cores with
    12, 20, 36 or 68 steps (up to 33, 65, 129, 257 taps); 15 taps stay on the
    FMA loop.  Ragged length (not a multiple of the 2048-output tile), several
    batches, nonzero skip; forward and all four gradients against float64.
    """
    torch.manual_seed(100 + Km)
    B, C, L = 3, 5, 4500
    x = torch.randn(B, 3 * C, L, dtype=torch.float64, requires_grad=True)
    wp = (torch.randn(3 * C, 3, dtype=torch.float64) / 3 ** 0.5).requires_grad_(True)
    wm = (torch.randn(C, Km, dtype=torch.float64) / Km ** 0.5).requires_grad_(True)
    sk = torch.randn(C, dtype=torch.float64, requires_grad=True)
    # the B2B composition of the oracle's conv, in float64
    p = causal_conv1d_torch(x, wp)
    q, k, v = p[:, :C], p[:, C:2 * C], p[:, 2 * C:]
    z = k * v
    y_ref = q * (causal_conv1d_torch(z, wm) + sk.view(1, C, 1) * z)
    gy = torch.randn_like(y_ref)
    y_ref.backward(gy)
    args = [t.detach().float().cuda().requires_grad_(True) for t in (x, wp, wm, sk)]
    y = b2b_causal_conv1d(*args)
    y.backward(gy.float().cuda())
    y = y.detach().double().cpu()
    assert rel_l2(y_ref, y) < 1e-5
    # the first outputs of a row and of a tile see the causal zero padding / the tile halo
    assert rel_l2(y_ref[..., :Km + 3], y[..., :Km + 3]) < 1e-5
    assert rel_l2(y_ref[..., 2048:2048 + Km], y[..., 2048:2048 + Km]) < 1e-5
    for ref, got in zip((x, wp, wm, sk), args):
        assert rel_l2(ref.grad, got.grad.double()) < 1e-5
    # gradients near the row end and across a tile boundary
    assert rel_l2(x.grad[..., -Km - 3:], args[0].grad[..., -Km - 3:].double()) < 1e-5
    assert rel_l2(x.grad[..., 2040:2060], args[0].grad[..., 2040:2060].double()) < 1e-5


def test_b2b_config2_shape_bf16_sample():
    """Config 2 (B=4, L=8192, 3*4096 channels, k=3 then k=128) on a channel sample, bf16 I/O."""
    torch.manual_seed(3)
    B, C, L = 4, 64, 8192
    x = torch.randn(B, 3 * C, L).to(torch.bfloat16)
    wp = torch.randn(3 * C, 3)
    wm = torch.randn(C, 128) / 128 ** 0.5
    sk = torch.zeros(C)
    y = b2b_causal_conv1d(x.cuda(), wp.cuda(), wm.cuda(), sk.cuda())
    assert y.dtype == torch.bfloat16
    assert rel_l2(b2b_causal_conv1d_torch(x.float(), wp, wm, sk), y) < 2e-2


# --------------------------------------------------------------------------- module
@pytest.mark.parametrize("C,L,K", [(36, 256, 3), (64, 512, 7), (16, 128, 4)])
def test_module_matches_reference_conv(C, L, K):
    torch.manual_seed(42)
    ref = torch.nn.Conv1d(C, C, K, groups=C, bias=True)
    fast = HipCausalConv1d(C, C, K, groups=C, bias=True).cuda()
    fast.load_state_dict(ref.state_dict())
    x = torch.randn(2, C, L, requires_grad=True)
    y_ref = causal_conv1d_torch(x, ref.weight.squeeze(1), ref.bias)
    y_ref.sum().backward()
    xg = x.detach().cuda().requires_grad_(True)
    y = fast(xg)
    y.sum().backward()
    torch.testing.assert_close(y.cpu(), y_ref, atol=1e-3, rtol=1e-4)
    torch.testing.assert_close(xg.grad.cpu(), x.grad, atol=1e-2, rtol=1e-3)
    torch.testing.assert_close(fast.weight.grad.cpu(), ref.weight.grad, atol=1e-2, rtol=1e-3)
    torch.testing.assert_close(fast.bias.grad.cpu(), ref.bias.grad, atol=1e-2, rtol=1e-3)


@pytest.mark.parametrize("dtype,tol", [(torch.bfloat16, 4e-3), (torch.float16, 5e-4)])
@pytest.mark.parametrize("Km", [16, 33, 34, 65, 66, 128, 129, 256])
def test_b2b_16bit_io_mixer_as_bf16_products(dtype, tol, Km):
    """16-bit I/O runs the B2B mixer on v_mfma_f32_16x16x32_bf16 with z and the taps split into bf16
    halves (three products per step, ~2^-17 relative per product).  Against float64 of the same
    16-bit inputs the error is the output rounding: ~1e-3 (bf16) and ~1.5e-4 (fp16) rel-L2; a band
    or split mistake (a lost lo term alone is ~2^-9) fails the fp16 bound.  Tap counts on both sides
    of every band step boundary, ragged length, nonzero skip, the row start and a tile halo."""
    torch.manual_seed(200 + Km)
    B, C, L = 3, 5, 4500
    x = torch.randn(B, 3 * C, L).to(dtype)
    wp = torch.randn(3 * C, 3) / 3 ** 0.5
    wm = torch.randn(C, Km) / Km ** 0.5
    sk = torch.randn(C)
    p = causal_conv1d_torch(x.double(), wp.double())
    q, k, v = p[:, :C], p[:, C:2 * C], p[:, 2 * C:]
    z = k * v
    y64 = q * (causal_conv1d_torch(z, wm.double()) + sk.double().view(1, C, 1) * z)
    y = b2b_causal_conv1d(x.cuda(), wp.cuda(), wm.cuda(), sk.cuda())
    assert y.dtype == dtype
    y = y.double().cpu()
    assert rel_l2(y64, y) < tol
    assert rel_l2(y64[..., :Km + 3], y[..., :Km + 3]) < tol
    assert rel_l2(y64[..., 2048:2048 + Km], y[..., 2048:2048 + Km]) < tol


@pytest.mark.parametrize("act", ["identity", "silu"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,C,L,K", [(1, 2048, 6 * 2048 + 8, 18), (1, 2048, 5 * 2048, 145), (3, 70, 4100, 210),
                                     (2, 1, 2049, 256), (1, 3, 255, 17), (2, 5, 2047, 81)])
def test_bands_as_split_bf16_products(B, C, L, K, dtype, act):
    """The matrix-core bands (operands as exact sums of bf16 values) against float64 of the same inputs: tap counts at
    the step boundaries, runs of tiles that start inside a row (2048 channels: three or five tiles a run) or span
    rows, one-sample tails, unaligned rows.  fp32 values (weight and bias gradients in every type) are sums of up to
    B L products: 1e-6 relative, a few fp32 roundings; 16-bit outputs are one rounding, half a unit in the last
    place at most 2^-9 / 2^-12 relative.  A weight or bias gradient is a sum of B L terms of unit size, typically
    sqrt(B L) and where it cancels (one channel's bias) anything below, while its rounding error follows the terms:
    those errors are taken relative to sqrt(B L) per entry where that is more."""
    gen = torch.Generator(device="cuda").manual_seed(K)
    x = torch.randn(B, C, L, device="cuda", generator=gen).to(dtype).requires_grad_()
    gy = torch.randn(B, C, L, device="cuda", generator=gen).to(dtype)
    w = (torch.randn(C, K, device="cuda", generator=gen) / K ** 0.5).requires_grad_()
    b = torch.randn(C, device="cuda", generator=gen).requires_grad_()
    y = causal_conv1d(x, w, b, act)
    got = (y, *torch.autograd.grad(y, (x, w, b), gy))

    x6, w6, b6 = (t.detach().double().requires_grad_() for t in (x, w, b))
    n = L + K
    p = torch.fft.irfft(torch.fft.rfft(x6, n=n) * torch.fft.rfft(w6.flip(-1), n=n), n=n)[..., :L] + b6.view(1, C, 1)
    y6 = p * torch.sigmoid(p) if act == "silu" else p
    want = (y6, *torch.autograd.grad(y6, (x6, w6, b6), gy.double()))
    tol = {torch.float32: 1e-6, torch.bfloat16: 2.0 ** -9, torch.float16: 2.0 ** -12}[dtype]
    for i, (a, r) in enumerate(zip(got, want)):
        size = r.norm().item() if i < 2 else max(r.norm().item(), (r.numel() * B * L) ** 0.5)
        err = (a.double() - r).norm().item() / size
        assert err < (tol if i < 2 else 1e-6), (i, err)


def _taps64(x, w, b, act):
    """The conv tap by tap in float64: no zero tap meets a sample."""
    K = w.shape[1]
    xp = torch.nn.functional.pad(x, (K - 1, 0))
    p = (xp.unfold(2, K, 1) * w[None, :, None, :]).sum(-1) + b.view(1, -1, 1)
    return p * (1.0 / (1.0 + torch.exp(-p))) if act == "silu" else p


def _same_kind(ref, got, skip=None):
    """NaN where the reference has NaN, the same infinities, close elsewhere."""
    ref, got = ref.double().cpu(), got.double().cpu()
    keep = torch.ones_like(ref, dtype=torch.bool) if skip is None else ~skip
    assert torch.equal(torch.isnan(ref)[keep], torch.isnan(got)[keep])
    inf = torch.isinf(ref) & keep
    assert torch.equal(ref[inf], got[inf])
    fin = torch.isfinite(ref) & keep
    assert torch.isfinite(got[fin]).all()
    return fin


@pytest.mark.parametrize("act", ["identity", "silu"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,C,L,K", [(1, 3, 400, 5), (2, 2, 4501, 9), (2, 2, 4504, 16), (1, 3, 2500, 17), (2, 3, 6200, 64),
                                     (1, 2, 4300, 256), (1, 2048, 5 * 2048, 18)])
def test_non_finite_samples_reach_their_own_outputs(B, C, L, K, dtype, act):
    """An inf or NaN in x, in the upstream gradient or in a tap reaches the results that a sum over the taps gives, as
    the same kind of value, and no other: not the outputs before it, nor the rest of its tile.  (Up to 16 taps the
    register kernels pad the taps with zeros, which meet samples up to 16 before their own.)  Values elsewhere as
    without it; 2048 channels: runs of tiles that start inside a row."""
    print(f"B={B} C={C} L={L} K={K} {dtype} {act}", flush=True)
    gen = torch.Generator().manual_seed(K)
    x = torch.randn(B, C, L, generator=gen).to(dtype)
    gy = torch.randn(B, C, L, generator=gen).to(dtype)
    w, b = torch.randn(C, K, generator=gen) / K ** 0.5, torch.randn(C, generator=gen)
    n = min(C, 3)  # channels checked
    p1, p2 = L // 3, (2 * L) // 3
    x[0, 0, p1], x[0, 0, p1 + 40], x[0, 1, p2] = float("inf"), float("-inf"), float("nan")
    gy[0, 1, p1], gy[0, 0, p2] = float("-inf"), float("nan")
    if C == 3:
        w[2, K // 2] = float("inf")
    xg, wg, bg = (t.cuda().requires_grad_() for t in (x, w, b))
    y = causal_conv1d(xg, wg, bg, act)
    gx, gw, gb = torch.autograd.grad(y, (xg, wg, bg), gy.cuda())

    x6, w6, b6 = (t[:, :n].double() if t.dim() == 3 else t[:n].double() for t in (x, w, b))
    p = _taps64(x6, w6, b6, "identity")
    s = 1.0 / (1.0 + torch.exp(-p))
    g6 = gy[:, :n].double()
    gp = g6 * (s * (1.0 + p * (1.0 - s))) if act == "silu" else g6
    want_gx = (torch.nn.functional.pad(gp, (0, K - 1)).unfold(2, K, 1) * w6.flip(1)[None, :, None, :]).sum(-1)
    xw = torch.nn.functional.pad(x6, (K - 1, 0)).unfold(2, K, 1)  # [B, n, L, K]
    want_gw, want_gb = (gp.unsqueeze(-1) * xw).sum((0, 2)), gp.sum((0, 2))
    want_y = p * s if act == "silu" else p
    pad = 16 - K if K <= 16 else 0

    def near(bad):  # positions within `pad` of a non-finite result
        m = torch.zeros_like(bad)
        for i in range(1, pad + 1):
            m |= torch.roll(bad, i, -1) | torch.roll(bad, -i, -1)
        return m & ~bad

    tol = {torch.float32: 2e-5, torch.bfloat16: 2e-2, torch.float16: 4e-3}[dtype]
    for want, got in ((want_y, y[:, :n]), (want_gx, gx[:, :n])):
        fin = _same_kind(want, got, near(~torch.isfinite(want)) if pad else None)
        a, r = got.double().cpu()[fin], want[fin]
        assert (a - r).norm() < tol * r.norm()
    if not pad:
        for want, got in ((want_gw, gw[:n]), (want_gb, gb[:n])):
            _same_kind(want, got)


@pytest.mark.parametrize("K", [9, 64, 256])
def test_values_above_the_largest_bf16_stay_finite(K):
    """fp32 values between the largest bf16 and the largest fp32 (which round to infinity in bf16) as samples, taps and
    gradients: results as in float64."""
    B, C, L = 1, 2, 3000
    gen = torch.Generator().manual_seed(K)
    x, gy = torch.randn(B, C, L, generator=gen), torch.randn(B, C, L, generator=gen)
    w, b = torch.randn(C, K, generator=gen) * 1e-3, torch.randn(C, generator=gen)
    big = float(torch.finfo(torch.float32).max)
    x[0, 0, 700], gy[0, 0, 1500], w[1, 3] = big, -big, big
    x[0, 1] *= 1e-3
    gy[0, 1] *= 1e-3
    args = [t.cuda().requires_grad_() for t in (x, w, b)]
    y = causal_conv1d(*args)
    got = (y, *torch.autograd.grad(y, args, gy.cuda()))
    args6 = [t.double().requires_grad_() for t in (x, w, b)]
    y6 = _taps64(*args6, "identity")
    want = (y6, *torch.autograd.grad(y6, args6, gy.double()))
    for i, (a, r) in enumerate(zip(got, want)):
        for c in range(C):  # the channels differ in size by 1e38
            ac, rc = (t[:, c] if t.dim() == 3 else t[c] for t in (a.double().cpu(), r))
            if rc.abs().max() < 1e38:  # an overflowing sum is an infinity in any order
                assert torch.isfinite(ac).all(), (i, c)
                assert (ac - rc).norm() <= 1e-5 * rc.norm(), (i, c)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_split_products_round_to_nearest(dtype):
    """One non-zero tap: each output is one product of a sample and a tap, taken as products of their bf16 parts.  With
    parts rounded to nearest the products left out are at most 2^-24 of it and of either sign; the kept ones are exact,
    their fp32 sums lose up to half a unit in the last place (2^-24) where they are rounded and a whole one where the
    matrix unit cuts off the bits of a smaller term.  Checked: no error above 3 * 2^-24, and no mean error above 2^-25
    over 2^19 products of one sign.  Measured: 2.4 and -0.25 in units of 2^-24 (parts cut off: 8.8 and -0.88)."""
    gen = torch.Generator().manual_seed(3)
    C, L, K = 64, 8192, 33
    x = (1 + torch.rand(1, C, L, generator=gen)).to(dtype)
    w = torch.zeros(C, K)
    w[:, K - 1] = 1 + torch.rand(C, generator=gen)
    x[0, :, 0] = 1 + 2.0 ** -7 - 2.0 ** -23 if dtype == torch.float32 else x[0, :, 0]
    w[0, K - 1] = 1 + 2.0 ** -7 - 2.0 ** -23
    want = x.double() * w[:, -1:].double()
    if dtype == torch.float32:
        y = causal_conv1d(x.cuda(), w.cuda())
    else:  # the fp16 result is one rounding to 11 bits: take the fp32 weight gradient, one product a tap
        xg, wg = x.cuda(), w.cuda().requires_grad_()
        gy = torch.zeros(1, C, L, dtype=dtype)
        gy[..., L // 2] = (1 + torch.rand(C, generator=gen)).to(dtype)
        gw, = torch.autograd.grad(causal_conv1d(xg, wg), wg, gy.cuda())
        y = gw.flip(1)
        want = gy[0, :, L // 2, None].double() * x[0, :, L // 2 - K + 1:L // 2 + 1].double().flip(1)
    err = (y.double().cpu() - want) / want
    print("max", float(err.abs().max()) * 2 ** 24, "mean", float(err.mean()) * 2 ** 24)
    assert err.abs().max() <= 3 * 2.0 ** -24
    if dtype == torch.float32:
        assert err.mean().abs() <= 2.0 ** -25


@pytest.mark.parametrize("act", ["identity", "silu"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("L", [3, 8, 2045, 2047, 2048, 2049, 2052, 4100])
def test_unaligned_rows(L, dtype, act):
    """Rows that start at any element and end inside a vector of 4 or 8: odd lengths, and tensors one to three elements
    into their storage, against the same values in aligned storage where that exists, else float64.  What lies beside
    the tensor in its storage is NaN: nothing outside a row is read, and nothing is written there."""
    gen = torch.Generator().manual_seed(L)
    B, C, K = 2, 3, 17
    nan = float("nan")

    def at(t, off):  # a contiguous copy of t, `off` elements into a NaN-filled storage
        flat = torch.full((t.numel() + 16,), nan, device="cuda", dtype=t.dtype)
        v = flat[off:off + t.numel()].view(t.shape)
        v.copy_(t)
        return v

    x, gy = (torch.randn(B, C, L, generator=gen).to(dtype) for _ in range(2))
    w, b = torch.randn(C, K, generator=gen) / K ** 0.5, torch.randn(C, generator=gen)
    x6, w6, b6 = (t.double().requires_grad_() for t in (x, w, b))
    y6 = _taps64(x6, w6, b6, act)
    want = (y6, *torch.autograd.grad(y6, (x6, w6, b6), gy.double()))
    tol = {torch.float32: 1e-6, torch.bfloat16: 2.0 ** -9, torch.float16: 2.0 ** -12}[dtype]
    for off in range(4):
        args = [at(x, off).requires_grad_(), w.cuda().requires_grad_(), b.cuda().requires_grad_()]
        y = causal_conv1d(*args, act)
        got = (y, *torch.autograd.grad(y, args, at(gy, (off + 1) % 4)))
        for i, (r, a) in enumerate(zip(want, got)):
            err = (a.double().cpu() - r).norm() / r.norm()
            assert err < (tol if i < 2 else 2e-6), (off, i, float(err))
