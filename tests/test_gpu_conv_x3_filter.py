"""Backward filter of float layers on the bfloat16 matrix cores at float precision (csrc/wgrad_same.h) against the checker, whose sums
are in double: at most one rounding of 2^-24 per eight slots of a reduction of K, 2^-24 sqrt(K / 8) of the result by 2-norm."""
import numpy as np
import pytest

import oracle
import vdnn_implementation_amd.backend as be
from gpu_util import Dev, announce
from vdnn_implementation_amd.backend import check, lib

pytestmark = pytest.mark.gpu

# n, c, h, w, k, window
GEOMS = [
    (48, 64, 12, 12, 128, 3),     # whole tiles
    (41, 72, 9, 7, 200, 3),       # slices of five image rows, channels that end within a tile, samples of fewer slots than a split
    (7, 40, 29, 31, 104, 5),      # odd planes, two slots behind a row
    (40, 128, 5, 41, 64, 3),      # few rows
    (1, 136, 33, 65, 72, 5),      # one sample, one channel group beyond two tiles
]


@pytest.fixture(scope="module")
def ctx():
    with be.Context(pool_bytes=256 << 20) as c:
        yield c


def norm_error(got, want):
    return np.linalg.norm(got.astype(np.float64) - want) / np.linalg.norm(want.astype(np.float64))


def tensors(geom, seed):
    n, c, h, w, k, r = geom
    rng = np.random.default_rng(seed)
    x = np.maximum(rng.standard_normal((n, c, h, w)), 0).astype(np.float32)
    dy = rng.standard_normal((n, k, h, w)).astype(np.float32)
    full = (n, c, h, w, k, r, r, r // 2, r // 2, 1, 1)
    return be.shape(*full), oracle.shape(*full), x, dy, (k, c, r, r)


@pytest.mark.parametrize("geom", GEOMS, ids=lambda g: "x".join(map(str, g)))
def test_filter_and_bias_gradient_against_oracle(ctx, geom):
    g, og, x, dy, shape = tensors(geom, geom[0] * 100 + geom[1])
    k = shape[0]
    reduction = dy.size // k
    want_w = oracle.conv_bwd_filter_sgd(og, x, dy, np.zeros(shape, np.float32), 1.0)
    want_b = oracle.conv_bwd_bias_sgd(og, dy, np.zeros(k, np.float32), 1.0)
    alpha = np.float32(-0.37)
    rng = np.random.default_rng(1)
    w0, b0 = rng.standard_normal(shape).astype(np.float32), rng.standard_normal(k).astype(np.float32)
    assert lib.vdnn_conv_bwd_filter_sums_bias(g, 0, 0)
    with Dev(ctx) as d:
        dx_, ddy, gw, gb, wu, bu = d.up(x), d.up(dy), d.empty(shape), d.empty((k,)), d.up(w0), d.up(b0)
        be.profile_enable(ctx.handle, True)
        announce("x3 bwd filter", geom)
        check(lib.vdnn_conv_bwd_filter_bias(ctx.handle, None, g, 0, dx_.ptr, ddy.ptr, gw.ptr, gb.ptr, None, 0))
        got_w, got_b = gw.download(shape), gb.download((k,))
        assert norm_error(got_w, want_w) <= 2.0 ** -24 * np.sqrt(reduction / 8)
        # a bias gradient is a float sum of its own: chains of sixteen additions, then of their sums
        assert norm_error(got_b, want_b) <= 2.0 ** -24 * np.sqrt(reduction / 8)
        check(lib.vdnn_conv_bwd_filter_bias(ctx.handle, None, g, 0, dx_.ptr, ddy.ptr, gw.ptr, gb.ptr, None, 0))
        assert np.array_equal(gw.download(shape), got_w) and np.array_equal(gb.download((k,)), got_b)
        check(lib.vdnn_conv_bwd_filter_bias_sgd(ctx.handle, None, g, 0, dx_.ptr, ddy.ptr, wu.ptr, bu.ptr, alpha, None, 0))
        # (the update is one multiply-add of the same gradient)
        assert np.allclose(wu.download(shape), w0 + alpha * got_w.astype(np.float64), rtol=0, atol=2.0 ** -23 * np.abs(w0 + alpha * got_w).max())
        assert np.allclose(bu.download((k,)), b0 + alpha * got_b.astype(np.float64), rtol=0, atol=2.0 ** -23 * np.abs(b0 + alpha * got_b).max())
        ran = be.profile_collect(ctx.handle)
        be.profile_enable(ctx.handle, False)
        assert ran["conv_bwd_filter_x3_%dx%d" % shape[2:]]["launches"] == 3


@pytest.mark.parametrize("geom", [GEOMS[0], GEOMS[2]], ids=lambda g: "x".join(map(str, g)))
def test_values_without_three_parts(ctx, geom):
    """Infinities, NaN and floats that round to an infinite bfloat16 value reach the gradients that they reach in the checker.
    (A gradient of the output at the edge of its plane meets the padding's zeros on the device, products that the checker leaves
    out: those that are not finite lie inside.)"""
    g, og, x, dy, shape = tensors(geom, 7)
    n, c, h, w, k, r = geom
    x[0, 1, 3, 0], x[n - 1, 5, h - 1, w - 1], x[0, 9, 2, 2] = np.inf, np.nan, 3.4e38
    dy[0, 2, 4, 4], dy[n - 1, 7, 5, 5], dy[0, 11, 2, 2] = -np.inf, np.nan, 1e-30
    want = oracle.conv_bwd_filter_sgd(og, x, dy, np.zeros(shape, np.float32), 1.0)
    with Dev(ctx) as d:
        dx_, ddy, gw = d.up(x), d.up(dy), d.empty(shape)
        announce("x3 bwd filter special values", geom)
        check(lib.vdnn_conv_bwd_filter(ctx.handle, None, g, 0, dx_.ptr, ddy.ptr, gw.ptr, None, 0))
        got = gw.download(shape)
    assert np.isnan(want).any() and np.isinf(want).any()
    # products with the value next to the largest float may or may not overflow on the way: its channel is left out
    rest = np.ones(c, bool)
    rest[9] = False
    assert np.array_equal(np.isnan(got[:, rest]), np.isnan(want[:, rest]))
    assert np.array_equal(np.isposinf(got[:, rest]), np.isposinf(want[:, rest])) and np.array_equal(np.isneginf(got[:, rest]), np.isneginf(want[:, rest]))
    ordinary = np.isfinite(want) & (np.abs(want) < 1e6)
    assert norm_error(got[ordinary], want[ordinary]) <= 2.0 ** -24 * np.sqrt(n * h * w / 2)
