"""Edges of the 32x32 blocks that a tile's result leaves in (rows and columns that end inside one) and counts of slices around those
on their way from memory, against the checker, whose sums are in double. A sum of K products meets a rounding of 2^-24 per two
products on the float matrix cores; random signs make that 2^-24 sqrt(K / 2) of the result by 2-norm."""
import numpy as np
import pytest

import oracle
import vdnn_implementation_amd.backend as be
from gpu_util import Dev, announce
from vdnn_implementation_amd.backend import check, lib

pytestmark = pytest.mark.gpu

# n, c, h, w, k, window: 1x1 layers have c / 16 slices forward, k / 16 backward
CONVS = [(2, 16, 9, 7, 1, 1), (1, 80, 8, 8, 31, 1), (3, 96, 5, 13, 33, 1), (1, 112, 11, 3, 64, 1), (2, 128, 6, 6, 96, 1), (1, 144, 7, 9, 112, 1),
         (2, 33, 10, 10, 65, 3), (1, 160, 17, 15, 130, 3), (40, 24, 33, 31, 40, 3), (7, 64, 54, 54, 190, 3),
         (60, 33, 60, 60, 40, 3), (24, 66, 50, 50, 200, 3)]  # the larger tiles, odd and even counts of slices
FCS = [(1, 16, 1), (5, 99, 33), (33, 96, 31), (64, 112, 64), (65, 128, 130), (100, 1000, 97), (130, 4096, 300),
       (61, 9010, 4700), (200, 5009, 2600)]  # the larger tiles, odd and even counts of slices in a split


# rows around the eights that a block's result leaves in, forward (filters) and backward data (channels), in the 64x64 and the large tiles
FEW_ROWS = [(2, 7, 30, 30, 9, 3), (3, 17, 21, 19, 8, 1), (2, 24, 13, 17, 25, 3), (1, 15, 40, 40, 16, 5), (30, 8, 90, 91, 1, 3), (40, 9, 80, 80, 7, 1), (9, 16, 90, 91, 24, 3),
            (1, 300, 24, 23, 6, 1), (12, 150, 6, 5, 9, 3)]  # the last two with split sums
FEW_ROWS_FC = [(1, 9, 61), (7, 33, 130), (8, 700, 40), (9, 3000, 129), (17, 640, 800), (25, 5893, 753)]


@pytest.fixture(scope="module")
def ctx():
    with be.Context(pool_bytes=512 << 20) as c:
        yield c


def within(got, want, products):
    error = np.linalg.norm(got.astype(np.float64) - want) / np.linalg.norm(np.asarray(want, np.float64))
    return error <= 2.0 ** -24 * max(np.sqrt(products / 2), 4)  # (a few products: the roundings of bias, update and result)


@pytest.mark.parametrize("geom", CONVS + FEW_ROWS, ids=lambda g: "x".join(map(str, g)))
def test_convolution(ctx, geom):
    n, c, h, w, k, r = geom
    rng = np.random.default_rng(n + c + k)
    full = (n, c, h, w, k, r, r, r // 2, r // 2, 1, 1)
    g, og = be.shape(*full), oracle.shape(*full)
    x = np.maximum(rng.standard_normal((n, c, h, w)), 0).astype(np.float32)
    f, b = rng.standard_normal((k, c, r, r)).astype(np.float32), rng.standard_normal(k).astype(np.float32)
    want_y = oracle.conv_fwd(og, x, f, b)
    dy = rng.standard_normal(want_y.shape).astype(np.float32)
    want_dx = oracle.conv_bwd_data(og, dy, f)
    want_w = oracle.conv_bwd_filter_sgd(og, x, dy, f, -0.5)
    with Dev(ctx) as d:
        dx_, df, db, ddy = d.up(x), d.up(f), d.up(b), d.up(dy)
        y, gx = d.empty(want_y.shape), d.empty(x.shape)
        announce("tile epilogues", geom)
        check(lib.vdnn_conv_fwd(ctx.handle, None, g, 0, dx_.ptr, df.ptr, db.ptr, y.ptr, None, 0))
        plain = y.download(want_y.shape)
        assert within(plain, want_y, c * r * r)
        check(lib.vdnn_conv_fwd_relu(ctx.handle, None, g, 0, dx_.ptr, df.ptr, db.ptr, y.ptr, None, 0))
        assert np.array_equal(y.download(want_y.shape), np.maximum(plain, 0))
        check(lib.vdnn_conv_bwd_data(ctx.handle, None, g, 0, ddy.ptr, df.ptr, gx.ptr, None, 0))
        plain = gx.download(x.shape)
        assert within(plain, want_dx, k * r * r)
        check(lib.vdnn_conv_bwd_filter_sgd(ctx.handle, None, g, 0, dx_.ptr, ddy.ptr, df.ptr, -0.5, None, 0))
        assert within(df.download(f.shape), want_w, n * h * w)
        df2 = d.up(f)
        check(lib.vdnn_conv_bwd_data_relu(ctx.handle, None, g, 0, ddy.ptr, df2.ptr, dx_.ptr, dx_.ptr, None, 0))  # over the gating input
        assert np.array_equal(dx_.download(x.shape), np.where(x > 0, plain, 0))


@pytest.mark.parametrize("sizes", FCS + FEW_ROWS_FC, ids=lambda s: "x".join(map(str, s)))
def test_fully_connected(ctx, sizes):
    n, ci, co = sizes
    rng = np.random.default_rng(n + ci + co)
    x, f, b = np.maximum(rng.standard_normal((n, ci)), 0).astype(np.float32), rng.standard_normal((co, ci)).astype(np.float32), rng.standard_normal(co).astype(np.float32)
    dy = rng.standard_normal((n, co)).astype(np.float32)
    x64, f64, dy64 = x.astype(np.float64), f.astype(np.float64), dy.astype(np.float64)
    with Dev(ctx) as d:
        dx_, df, db, ddy = d.up(x), d.up(f), d.up(b), d.up(dy)
        y, gx = d.empty((n, co)), d.empty((n, ci))
        announce("tile epilogues, fully connected", sizes)
        check(lib.vdnn_fc_fwd(ctx.handle, None, n, ci, co, dx_.ptr, df.ptr, db.ptr, y.ptr))
        plain = y.download((n, co))
        assert within(plain, x64 @ f64.T + b, ci)
        check(lib.vdnn_fc_fwd_relu(ctx.handle, None, n, ci, co, dx_.ptr, df.ptr, db.ptr, y.ptr))
        assert np.array_equal(y.download((n, co)), np.maximum(plain, 0))
        check(lib.vdnn_fc_bwd_data(ctx.handle, None, n, ci, co, ddy.ptr, df.ptr, gx.ptr))
        plain = gx.download((n, ci))
        assert within(plain, dy64 @ f64, co)
        check(lib.vdnn_fc_bwd_weight_sgd(ctx.handle, None, n, ci, co, dx_.ptr, ddy.ptr, df.ptr, -0.5))
        assert within(df.download((co, ci)), f64 - 0.5 * (dy64.T @ x64), n)
        df2 = d.up(f)
        check(lib.vdnn_fc_bwd_data_relu(ctx.handle, None, n, ci, co, ddy.ptr, df2.ptr, dx_.ptr, dx_.ptr))
        assert np.array_equal(dx_.download((n, ci)), np.where(x > 0, plain, 0))
