"""The block-tiled pointwise convolution of wide layers (48 rows and channels
and more): every edge of its tiles against float64, and non-finite operands
against fp32 arithmetic.

Bars: an fp32 sum of k products is within (k + 2) 2^-24 sum |a||b| of the
exact one in any order; a product split into three bf16 parts is within
2^-24 |a||b| of exact like a rounded one.  The weight gradient adds fp32 sums
over chunks of at most 1024 pixels in float64.
"""
import numpy as np
import pytest

from test_gpu_parity import EPS, assert_stats, assert_vals, dev, host
from test_gpu_pw_conv import kernels

pytestmark = pytest.mark.gpu

U32 = 2.0 ** -24

SHAPES = [
    # (N, C_in, C_out, HW)
    (1, 48, 48, 4096),     # the narrowest: one partial row tile
    (3, 49, 65, 1537),     # nothing a multiple of anything; a 1-row second tile
    (2, 51, 130, 2055),    # three row tiles, HW % 4 = 3
    (1, 64, 64, 4098),     # whole row tile, a pixel tile of 2
    (1, 160, 200, 4100),   # five K steps, two ci tiles in the weight gradient
    (1, 132, 256, 2817),   # K % 32 = 4; a pixel tile of one pixel
    (5, 128, 72, 1000),    # several samples, ragged rows
    # chunks of 384 and 136 pixels: items of 128, 128, 128 | 128, 8 in a block,
    # four row tiles, the last of 8 rows
    (256, 200, 200, 520),
]


@pytest.fixture(autouse=True)
def no_simt(gpu, request):
    """The block-tiled kernels also where k_pw_small would run."""
    old = gpu.tune_get(gpu.TUNE_PW_SMALL)
    if "leaves_small" not in request.node.name:
        gpu.tune(gpu.TUNE_PW_SMALL, 0)
    yield
    gpu.tune(gpu.TUNE_PW_SMALL, old)


def data(seed, N, C_in, C_out, HW):
    r = np.random.default_rng(seed)
    x = (r.standard_normal((N, C_in, HW)) * np.exp(r.standard_normal((N, C_in, 1)))).astype(np.float32)
    w = (r.uniform(-1.0, 1.0, (C_out, C_in)) / np.sqrt(C_in)).astype(np.float32)
    b = r.uniform(-0.5, 0.5, C_out).astype(np.float32)
    dz = r.standard_normal((N, C_out, HW)).astype(np.float32)
    return x, w, b, dz


def check(got, truth, bound, what):
    ratio = np.abs(np.asarray(got, np.float64) - truth) / np.maximum(bound, 2.0 ** -149)
    assert ratio.max() <= 1.0, f"{what}: {ratio.max():.2f} of the bound"


@pytest.mark.parametrize("shape", SHAPES)
def test_pw_gemm_matches_float64(gpu, oracle, shape):
    N, C_in, C_out, HW = shape
    x, w, b, dz = data(7, *shape)
    X, W, D = x.astype(np.float64), w.astype(np.float64), dz.astype(np.float64)
    dzd, xd, wd = dev(dz), dev(x), dev(w)
    names, z = kernels(gpu, lambda: gpu.pw_conv_forward(xd, wd, dev(b)))
    assert "pw_conv_tiled" in names, names
    zb = (C_in + 2) * U32 * (np.abs(W) @ np.abs(X) + np.abs(b)[:, None])
    check(host(z), W @ X + b[:, None], zb, "z")

    G = 1 if C_out % 2 else 2
    gamma, beta = np.linspace(0.5, 1.5, C_out, dtype=np.float32), np.zeros(C_out, np.float32)
    names, (z2, y, st) = kernels(gpu, lambda: gpu.pw_conv_gn_silu_forward(
        xd, wd, dev(b), dev(gamma), dev(beta), G, eps=EPS))
    assert "pw_conv_gn_stats_tiled" in names, names
    check(host(z2), W @ X + b[:, None], zb, "z with statistics")
    ty, tm, tr = oracle.gn_silu_fwd_f64(host(z2), gamma, beta, N, C_out, HW, G, EPS)
    assert_vals(host(y), ty, "y")
    assert_stats(host(st.mean), host(st.rstd), tm, tr)

    old = np.linspace(-1.0, 1.0, N * C_in * HW, dtype=np.float32).reshape(N, C_in, HW)
    for acc in (False, True):
        names, (dx_, dw_, db_) = kernels(gpu, lambda: gpu.pw_conv_backward(
            dzd, xd, wd, dx=dev(old), accumulate_dx=acc))
        assert {"pw_conv_dgrad_tiled", "pw_conv_wgrad_tiled"} <= names, names
        bx = (C_out + 3) * U32 * (np.abs(W).T @ np.abs(D) + np.abs(old))
        check(host(dx_), W.T @ D + (old if acc else 0.0), bx, "dx")
    tw = np.einsum("nop,ncp->oc", D, X, optimize=True)
    bw = 1026 * U32 * np.einsum("nop,ncp->oc", np.abs(D), np.abs(X), optimize=True)
    check(host(dw_), tw, bw, "dw")
    check(host(db_), D.sum((0, 2)), 1026 * U32 * np.abs(D).sum((0, 2)), "db")


@pytest.mark.parametrize("ex, ew", [(-112, 0), (-122, 0), (0, -118), (-112, 100), (100, -120),
                                    (-60, -60), (60, 50), (90, 20), (115, -100)])
def test_pw_gemm_operands_of_any_size(gpu, ex, ew):
    """Operands anywhere in fp32's range keep their 24 bits, however small the
    parts that they split into: the bar of the other tests at every scale
    (and, where a product is below 2^-126, fp32's spacing there)."""
    N, C_in, C_out, HW = 1, 64, 96, 4096
    x, w, _, dz = data(13, N, C_in, C_out, HW)
    # exact scales, powers of two
    x, dz, w = (np.ldexp(v, e).astype(np.float32) for v, e in ((x, ex), (dz, ex), (w, ew)))
    X, W, D = x.astype(np.float64), w.astype(np.float64), dz.astype(np.float64)
    tiny = 2.0 ** -149
    z = gpu.pw_conv_forward(dev(x), dev(w))
    check(host(z), W @ X, (C_in + 2) * (U32 * (np.abs(W) @ np.abs(X)) + tiny), "z")
    dx, _, _ = gpu.pw_conv_backward(dev(dz), dev(x), dev(w), want_dw=False, want_db=False)
    check(host(dx), W.T @ D, (C_out + 2) * (U32 * (np.abs(W).T @ np.abs(D)) + tiny), "dx")
    # the weight gradient of operands this far apart: dz of w's scale
    dz = np.ldexp(data(13, N, C_in, C_out, HW)[3], ew).astype(np.float32)
    D = dz.astype(np.float64)
    _, dw, _ = gpu.pw_conv_backward(dev(dz), dev(x), dev(w), want_dx=False, want_db=False)
    check(host(dw), np.einsum("nop,ncp->oc", D, X, optimize=True),
          1026 * (U32 * np.einsum("nop,ncp->oc", np.abs(D), np.abs(X), optimize=True) + tiny), "dw")


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, 3.4e38])
def test_pw_gemm_non_finite_operands(gpu, value):
    """An output that an infinity, a NaN or a value that bf16 rounds to
    infinity reaches is what fp32 products and sums give; the others are
    untouched."""
    N, C_in, C_out, HW = 1, 64, 96, 4096
    x, w, _, dz = data(11, N, C_in, C_out, HW)
    clean = host(gpu.pw_conv_forward(dev(x), dev(w)))
    dxc, dwc, _ = gpu.pw_conv_backward(dev(dz), dev(x), dev(w))
    x[0, 5, 777] = value
    dz[0, 70, 1234] = value
    w[3, 5] = 0.0  # inf * 0
    with np.errstate(all="ignore"):
        z = host(gpu.pw_conv_forward(dev(x), dev(w)))
        want = w @ x[0, :, 777]
        np.testing.assert_allclose(z[0, :, 777], want, rtol=1e-5)
        # with the statistics: the same z, and groups that it does not reach
        G = 8
        z2, y, st = gpu.pw_conv_gn_silu_forward(dev(x), dev(w), None,
                                                dev(np.ones(C_out, np.float32)),
                                                dev(np.zeros(C_out, np.float32)), G, eps=EPS)
        np.testing.assert_array_equal(host(z2), z)
        reached = (~np.isfinite(z[0])).any(1).reshape(G, -1).any(1)
        assert np.array_equal(np.isnan(host(st.mean)) | np.isinf(host(st.mean)), reached)
        assert np.isfinite(host(y)[0][~np.repeat(reached, C_out // G)]).all()
        keep = np.arange(HW) != 777
        np.testing.assert_allclose(z[0][4:70, keep], clean[0][4:70, keep], rtol=1e-4, atol=1e-4)
        dx, dw, _ = gpu.pw_conv_backward(dev(dz), dev(x), dev(w))
        np.testing.assert_allclose(host(dx)[0, :, 1234], w.T @ dz[0, :, 1234], rtol=1e-5)
        keep = np.arange(HW) != 1234
        assert np.isfinite(host(dx)[0][:, keep]).all()
        bad = ~np.isfinite(host(dw))
        if not np.isfinite(value):
            assert bad[70].all() and bad[:, 5].all() and bad.sum() == C_in + C_out - 1
        else:
            rest = np.ones((C_out, C_in), bool)
            rest[70], rest[:, 5] = False, False
            assert np.isfinite(host(dw)[rest]).all()
    # columns and rows that nothing non-finite reaches
    np.testing.assert_allclose(host(dw)[:70, 6:], host(dwc)[:70, 6:], rtol=1e-3, atol=1e-3)


@pytest.mark.parametrize("shape, forward, fused, dgrad", [
    # (N, C_in, C_out, HW), whether the block-tiled kernel runs: 32 tiles of
    # 128 pixels and more each
    ((32, 512, 512, 1), False, False, False),    # 1 pixel of a tile: 7 against 30 us
    ((16, 256, 256, 4), False, False, False),
    ((32, 64, 64, 49), False, False, False),
    ((8, 64, 64, 400), False, False, False),     # 12.5 * 2^20 multiply-adds, the line at 14
    ((16, 64, 64, 256), True, False, True),      # 16 * 2^20; the fused form's line at 18
    ((32, 128, 128, 49), True, False, True),     # 24.5 * 2^20, the lines at 21 and 25
    ((128, 512, 512, 1), False, False, False),   # 2^25, 1024 tiles
    ((1, 64, 64, 4096), True, True, True),       # units of more than 16384: statistics fused
    ((1, 128, 256, 4096), True, True, True),
])
def test_pw_gemm_leaves_small_layers(gpu, shape, forward, fused, dgrad):
    import torch
    N, C_in, C_out, HW = shape
    x, w, b, dz = (dev(v) for v in data(5, *shape))
    ga, be = torch.ones(C_out, device="cuda"), torch.zeros(C_out, device="cuda")
    got, _ = kernels(gpu, lambda: gpu.pw_conv_forward(x, w, b))
    assert ("pw_conv_tiled" in got) == forward, got
    got, _ = kernels(gpu, lambda: gpu.pw_conv_gn_silu_forward(x, w, b, ga, be, 8))
    assert ("pw_conv_gn_stats_tiled" in got) == fused, got
    got, _ = kernels(gpu, lambda: gpu.pw_conv_backward(dz, x, w, want_dw=False, want_db=False))
    assert ("pw_conv_dgrad_tiled" in got) == dgrad, got
