"""GPU parity: a seeded sweep of 3x3 / stride 1 / padding 1 geometries through the kernels written for them (the windowed
forward / backward data of bfloat16 layers, the row-per-workgroup backward filter in both element types, the streaming
first-layer kernels), against the CPU checker through the C ABI.

The shapes are drawn so that every variant is met several times: rows of whole groups of eight, four and two pixels,
rows shorter and longer than a slice and than a tile, planes that are and are not multiples of the slice, one to three
input channels, channel counts of one and several blocks, ragged output-channel tiles, reductions short enough for one
split and long enough for many. Tolerances as in test_gpu_kernels.py / test_gpu_bf16.py.
"""
import numpy as np
import pytest

import oracle
import vdnn_implementation_amd.backend as be
from gpu_util import announce, gpu_conv_bwd_data, gpu_conv_bwd_filter, gpu_conv_fwd
from test_gpu_bf16 import Dev, get_act, rnd
from util import assert_close, assert_close_bf16
from vdnn_implementation_amd.backend import check, lib

pytestmark = pytest.mark.gpu
TOL = 1e-4


@pytest.fixture(scope="module")
def ctx():
    c = be.Context(pool_bytes=4 << 30)
    yield c
    c.close()


@pytest.fixture(autouse=True)
def accurate_oracle():
    oracle.set_accumulate_double(True)
    yield
    oracle.set_accumulate_double(False)


def sweep(seed, count):
    rng = np.random.default_rng(seed)
    out = []
    widths = [14, 16, 18, 20, 24, 28, 30, 32, 36, 40, 44, 56, 64, 72, 130]
    while len(out) < count:
        w = int(rng.choice(widths))
        h = int(rng.integers(2, 13))
        if rng.random() < 0.25:
            c = int(rng.integers(1, 4))                   # the first-layer kernels
            k = int(rng.choice([8, 16, 32, 40, 64]))
        else:
            c = int(rng.choice([32, 64, 64, 128, 192]))
            k = int(rng.choice([32, 64, 96, 128, 130, 192]))
        n = int(rng.integers(1, 6))
        if n * c * h * w * k * 9 > 6e8:                   # keeps the checker within a second or two per case
            continue
        out.append((n, c, h, w, k, 3, 3, 1, 1, 1, 1))
    return out


@pytest.mark.parametrize("geom", sweep(20240611, 48), ids=lambda g: "x".join(map(str, g[:5])))
def test_conv3x3_sweep_float(ctx, geom):
    rng = np.random.default_rng(abs(hash(geom)) % (2 ** 31))
    g, og = be.shape(*geom), oracle.shape(*geom)
    x = rng.standard_normal((g.n, g.c, g.h, g.w)).astype(np.float32)
    w = (rng.standard_normal((g.k, g.c, 3, 3)) * np.sqrt(2.0 / (g.c * 9))).astype(np.float32)
    b = rng.standard_normal(g.k).astype(np.float32)
    want_y = oracle.conv_fwd(og, x, w, b)
    announce("conv sweep float", geom, "fwd")
    assert_close(gpu_conv_fwd(ctx, g, x, w, b), want_y, TOL, "fwd")
    dy = rng.standard_normal(want_y.shape).astype(np.float32)
    announce("conv sweep float", geom, "bwd_data")
    assert_close(gpu_conv_bwd_data(ctx, g, dy, w), oracle.conv_bwd_data(og, dy, w), TOL, "bwd data")
    announce("conv sweep float", geom, "bwd_filter")
    zero = np.zeros_like(w)
    assert_close(gpu_conv_bwd_filter(ctx, g, x, dy, zero, np.float32(1.0)), oracle.conv_bwd_filter_sgd(og, x, dy, zero, 1.0), TOL, "bwd filter")


@pytest.mark.parametrize("geom", sweep(977, 48), ids=lambda g: "x".join(map(str, g[:5])))
def test_conv3x3_sweep_bfloat16(ctx, geom):
    rng = np.random.default_rng(abs(hash(geom)) % (2 ** 31) + 1)
    g, og = be.shape(*geom), oracle.shape(*geom)
    x = rnd(rng, (g.n, g.c, g.h, g.w))
    w = (rng.standard_normal((g.k, g.c, 3, 3)) * np.sqrt(2.0 / (g.c * 9))).astype(np.float32)
    b = rng.standard_normal(g.k).astype(np.float32)
    wr = oracle.round_bf16(w)  # forward and backward data multiply the filter rounded to bfloat16
    want_y = oracle.conv_fwd(og, x, wr, b)
    dy = rnd(rng, want_y.shape)
    check(lib.vdnn_ctx_set_activation_dtype(ctx.handle, 1))
    try:
        with Dev(ctx) as d:
            dx_, ddy, dw, db = d.act(x), d.act(dy), d.f32(w), d.f32(b)
            y, gx = d.empty_act(want_y.shape), d.empty_act(x.shape)
            announce("conv sweep bf16", geom, "fwd")
            check(lib.vdnn_conv_fwd(ctx.handle, None, g, 0, dx_.ptr, dw.ptr, db.ptr, y.ptr, None, 0))
            assert_close_bf16(get_act(y, want_y.shape), want_y, "fwd")
            announce("conv sweep bf16", geom, "bwd_data")
            check(lib.vdnn_conv_bwd_data(ctx.handle, None, g, 0, ddy.ptr, dw.ptr, gx.ptr, None, 0))
            assert_close_bf16(get_act(gx, x.shape), oracle.conv_bwd_data(og, dy, wr), "bwd data")
            announce("conv sweep bf16", geom, "bwd_filter")
            gw = d.f32(np.zeros_like(w))
            check(lib.vdnn_conv_bwd_filter(ctx.handle, None, g, 0, dx_.ptr, ddy.ptr, gw.ptr, None, 0))
            assert_close(gw.download(w.shape), oracle.conv_bwd_filter_sgd(og, x, dy, np.zeros_like(w), 1.0), 1e-4, "bwd filter")
    finally:
        check(lib.vdnn_ctx_set_activation_dtype(ctx.handle, 0))


# Layers of up to three input channels that leave the chip idle: backward data walks strips of two rows up, backward filter
# splits of one slice of 64 pixels up. Strips that do not divide the rows, a last strip of one row, several column blocks,
# reductions that are no whole slices, one and several tiles of filters.
@pytest.mark.parametrize("geom", [(4, 3, 20, 20, 8, 3, 3, 1, 1, 1, 1), (1, 3, 21, 20, 8, 3, 3, 1, 1, 1, 1), (1, 1, 5, 16, 4, 3, 3, 1, 1, 1, 1), (2, 2, 7, 64, 33, 3, 3, 1, 1, 1, 1),
                                  (3, 3, 33, 36, 70, 3, 3, 1, 1, 1, 1), (1, 3, 50, 224, 64, 3, 3, 1, 1, 1, 1), (8, 3, 101, 40, 16, 3, 3, 1, 1, 1, 1)],
                         ids=lambda g: "x".join(map(str, g[:5])))
def test_few_channels_on_an_idle_chip(ctx, geom):
    test_conv3x3_sweep_float(ctx, geom)
    test_conv3x3_sweep_bfloat16(ctx, geom)


# The 64x64 tile: one row or column short of a tile and one past it, reductions of one slice and of many splits, 260 and
# 516 tiles for 256 units (only the tiles behind whole rounds are split), taps shared by a tile's columns (channels in
# 64s and 32s) and not, planes that are no whole groups of pixels.
@pytest.mark.parametrize("geom", [
    (1, 16, 5, 13, 63, 3, 3, 1, 1, 1, 1), (1, 17, 9, 7, 65, 3, 3, 0, 0, 1, 1), (2, 64, 8, 8, 64, 1, 1, 0, 0, 1, 1), (3, 5, 1, 21, 7, 1, 1, 0, 0, 1, 1),
    (4, 32, 52, 80, 64, 3, 3, 1, 1, 1, 1), (2, 96, 129, 64, 64, 3, 3, 1, 1, 1, 1), (5, 33, 11, 11, 129, 5, 5, 2, 2, 1, 1), (2, 64, 12, 12, 66, 5, 5, 2, 2, 1, 1),
    (3, 32, 9, 12, 130, 4, 4, 1, 1, 1, 1), (2, 128, 13, 13, 192, 3, 3, 1, 1, 1, 1)], ids=lambda g: "x".join(map(str, g)))
def test_conv_small_tile(ctx, geom):
    rng = np.random.default_rng(sum((i + 1) * v for i, v in enumerate(geom)))
    g, og = be.shape(*geom), oracle.shape(*geom)
    x = rng.standard_normal((g.n, g.c, g.h, g.w)).astype(np.float32)
    w = (rng.standard_normal((g.k, g.c, g.r, g.s)) * np.sqrt(2.0 / (g.c * g.r * g.s))).astype(np.float32)
    b = rng.standard_normal(g.k).astype(np.float32)
    want_y = oracle.conv_fwd(og, x, w, b)
    announce("conv small tile", geom)
    assert_close(gpu_conv_fwd(ctx, g, x, w, b), want_y, TOL, "fwd")
    dy = rng.standard_normal(want_y.shape).astype(np.float32)
    assert_close(gpu_conv_bwd_data(ctx, g, dy, w), oracle.conv_bwd_data(og, dy, w), TOL, "bwd data")
    zero = np.zeros_like(w)
    assert_close(gpu_conv_bwd_filter(ctx, g, x, dy, zero, np.float32(1.0)), oracle.conv_bwd_filter_sgd(og, x, dy, zero, 1.0), TOL, "bwd filter")


@pytest.mark.parametrize("geom", [(4, 64, 16, 16, 64, 5, 5, 2, 2, 1, 1), (16, 64, 14, 14, 128, 1, 1, 0, 0, 1, 1), (8, 128, 12, 12, 192, 5, 5, 2, 2, 1, 1),
                                  (32, 96, 16, 16, 70, 1, 1, 0, 0, 1, 1), (2, 64, 28, 28, 256, 5, 5, 2, 2, 1, 1)], ids=lambda g: "x".join(map(str, g)))
def test_backward_filter_bits_do_not_depend_on_the_address(ctx, geom):
    """dy at a 16-byte boundary and one element past it: other loaders, the same tile and splits, so the same sums."""
    rng = np.random.default_rng(sum(geom))
    g = be.shape(*geom)
    x, dy = rng.standard_normal((g.n, g.c, g.h, g.w)).astype(np.float32), rng.standard_normal((g.n, g.k, g.h, g.w)).astype(np.float32)
    announce("backward filter, dy aligned and not", geom)
    with Dev(ctx) as d:
        xx, out = d.f32(x), [d.f32(np.zeros((g.k, g.c, g.r, g.s))) for _ in range(2)]
        for shift, dw in enumerate(out):
            b = d.f32(np.concatenate([np.zeros(shift, np.float32), dy.ravel()]))
            assert b.ptr % 16 == 0
            check(lib.vdnn_conv_bwd_filter(ctx.handle, None, g, 0, xx.ptr, b.ptr + 4 * shift, dw.ptr, None, 0))
        got = [dw.download((g.k, g.c, g.r, g.s)) for dw in out]
    assert np.array_equal(got[0], got[1])


@pytest.mark.parametrize("n,cin,cout", [(1, 64, 1), (63, 17, 65), (65, 192, 64), (3, 193, 129), (64, 1028, 260), (130, 5, 7)])
def test_fc_small_tile(ctx, n, cin, cout):
    rng = np.random.default_rng(n * 7 + cin * 3 + cout)
    x, w = rng.standard_normal((n, cin)).astype(np.float32), (rng.standard_normal((cout, cin)) / np.sqrt(cin)).astype(np.float32)
    b, dy = rng.standard_normal(cout).astype(np.float32), rng.standard_normal((n, cout)).astype(np.float32)
    announce("fc small tile", n, cin, cout)
    with Dev(ctx) as d:
        dx_, dw, db, ddy = d.f32(x), d.f32(w), d.f32(b), d.f32(dy)
        y, gx = d.f32(np.zeros((n, cout))), d.f32(np.zeros((n, cin)))
        check(lib.vdnn_fc_fwd(ctx.handle, None, n, cin, cout, dx_.ptr, dw.ptr, db.ptr, y.ptr))
        check(lib.vdnn_fc_bwd_data(ctx.handle, None, n, cin, cout, ddy.ptr, dw.ptr, gx.ptr))
        gw = d.f32(np.zeros_like(w))
        check(lib.vdnn_fc_bwd_weight(ctx.handle, None, n, cin, cout, dx_.ptr, ddy.ptr, gw.ptr))
        assert_close(y.download((n, cout)), oracle.fc_fwd(x, w, b), TOL, "fwd")
        assert_close(gx.download((n, cin)), oracle.fc_bwd_data(dy, w), TOL, "bwd data")
        assert_close(gw.download(w.shape), dy.astype(np.float64).T @ x.astype(np.float64), TOL, "bwd weight")


# Backward data of strided layers by residue classes: strides per axis up to four classes, windows smaller than the stride
# (classes that no tap reaches), padding up to the window, output channels that are no whole slices, planes smaller than
# the window plus stride, one tile and many, enough filters for split reductions.
STRIDED = [(2, 5, 9, 11, 7, 3, 3, 1, 1, 2, 2), (1, 17, 8, 8, 33, 1, 1, 0, 0, 2, 2), (3, 70, 13, 9, 130, 3, 3, 1, 1, 2, 2), (2, 6, 10, 7, 16, 4, 4, 3, 3, 2, 2),
           (2, 64, 7, 30, 48, 5, 5, 2, 2, 2, 2), (1, 9, 12, 12, 5, 3, 3, 0, 0, 1, 2), (2, 9, 12, 13, 20, 3, 2, 0, 1, 3, 1), (1, 8, 17, 5, 40, 5, 3, 2, 0, 4, 1),
           (1, 65, 3, 3, 600, 3, 3, 0, 0, 2, 2), (4, 40, 64, 66, 31, 3, 3, 1, 1, 2, 2), (1, 7, 20, 21, 18, 11, 11, 5, 5, 2, 2),
           # the small ones above again, large enough for the classes in both element types
           (20, 25, 39, 21, 27, 3, 3, 1, 1, 2, 2), (8, 67, 28, 28, 333, 1, 1, 0, 0, 2, 2), (8, 36, 30, 27, 40, 4, 4, 3, 3, 2, 2), (3, 49, 32, 42, 65, 3, 3, 0, 0, 1, 2),
           (4, 39, 32, 33, 130, 3, 2, 0, 1, 3, 1), (9, 28, 57, 15, 40, 5, 3, 2, 0, 4, 1), (6, 65, 7, 7, 600, 3, 3, 0, 0, 2, 2)]


@pytest.mark.parametrize("geom", STRIDED, ids=lambda g: "x".join(map(str, g)))
def test_strided_backward_data(ctx, geom):
    rng = np.random.default_rng(sum((i + 1) * v for i, v in enumerate(geom)))
    g, og = be.shape(*geom), oracle.shape(*geom)
    w = (rng.standard_normal((g.k, g.c, g.r, g.s)) * np.sqrt(2.0 / (g.c * g.r * g.s))).astype(np.float32)
    P, Q = lib.vdnn_out_dim(g.h, g.pad_h, g.r, g.stride_h), lib.vdnn_out_dim(g.w, g.pad_w, g.s, g.stride_w)
    dy = rnd(rng, (g.n, g.k, P, Q))  # bfloat16 values: both element types see the same gradient
    x = rnd(rng, (g.n, g.c, g.h, g.w))
    announce("strided bwd data", geom)
    want = oracle.conv_bwd_data(og, dy, w)
    assert_close(gpu_conv_bwd_data(ctx, g, dy, w), want, TOL, "float")
    with Dev(ctx) as d:
        ddy, dw, dxx, gx = d.f32(dy), d.f32(w), d.f32(x), d.f32(np.zeros_like(x))
        check(lib.vdnn_conv_bwd_data_relu(ctx.handle, None, g, 0, ddy.ptr, dw.ptr, dxx.ptr, gx.ptr, None, 0))
        assert_close(gx.download(x.shape), np.where(x > 0, want, 0), TOL, "float, gated")
        if g.n > 1:  # what one sample holds reaches no other one
            spoilt = dy.copy()
            spoilt[1] = np.inf
            b = d.f32(spoilt)
            check(lib.vdnn_conv_bwd_data(ctx.handle, None, g, 0, b.ptr, dw.ptr, gx.ptr, None, 0))
            assert_close(gx.download(x.shape)[0], want[0], TOL, "beside a sample of infinities")
    check(lib.vdnn_ctx_set_activation_dtype(ctx.handle, 1))
    try:
        with Dev(ctx) as d:
            ddy, dw, dxx, gx = d.act(dy), d.f32(w), d.act(x), d.empty_act(x.shape)
            check(lib.vdnn_conv_bwd_data_relu(ctx.handle, None, g, 0, ddy.ptr, dw.ptr, dxx.ptr, gx.ptr, None, 0))
            assert_close_bf16(get_act(gx, x.shape), np.where(x > 0, oracle.conv_bwd_data(og, dy, oracle.round_bf16(w)), 0), "bf16, gated")
    finally:
        check(lib.vdnn_ctx_set_activation_dtype(ctx.handle, 0))


def test_strided_backward_data_in_chunks_of_samples(ctx):
    """Results of five samples of 3.8 million elements do not fit the staging area of 16 million: four samples, then one, each
    with its own splits. Gated and not, both element types."""
    geom = (5, 24, 400, 400, 33, 3, 3, 1, 1, 2, 2)
    rng = np.random.default_rng(5)
    g, og = be.shape(*geom), oracle.shape(*geom)
    w = (rng.standard_normal((33, 24, 3, 3)) * 0.1).astype(np.float32)
    dy, x = rnd(rng, (5, 33, 200, 200)), rnd(rng, (5, 24, 400, 400))
    for bf16 in (0, 1):
        want = oracle.conv_bwd_data(og, dy, oracle.round_bf16(w) if bf16 else w)
        check(lib.vdnn_ctx_set_activation_dtype(ctx.handle, bf16))
        try:
            with Dev(ctx) as d:
                up = d.act if bf16 else d.f32
                ddy, dxx, dw, gx = up(dy), up(x), d.f32(w), up(np.zeros_like(x))
                for gate in (False, True):
                    announce("strided bwd data in chunks", bf16, gate)
                    be.profile_enable(ctx.handle, 1)
                    if gate:
                        check(lib.vdnn_conv_bwd_data_relu(ctx.handle, None, g, 0, ddy.ptr, dw.ptr, dxx.ptr, gx.ptr, None, 0))
                    else:
                        check(lib.vdnn_conv_bwd_data(ctx.handle, None, g, 0, ddy.ptr, dw.ptr, gx.ptr, None, 0))
                    assert be.profile_collect(ctx.handle)["conv_bwd_data_merge"]["launches"] == 2
                    got, ref = (get_act(gx, x.shape) if bf16 else gx.download(x.shape)), np.where(x > 0, want, 0) if gate else want
                    for n in range(5):
                        (assert_close_bf16(got[n], ref[n], "sample %d" % n) if bf16 else assert_close(got[n], ref[n], TOL, "sample %d" % n))
        finally:
            be.profile_enable(ctx.handle, 0)
            check(lib.vdnn_ctx_set_activation_dtype(ctx.handle, 0))


# Reduced channels (input channels forward, filters in backward data) that are no whole blocks of 16 or 32, through every
# bfloat16 kernel that pads them (windowed 3x3; pixel pairs; single pixels, odd rows or strides) and the float engine: one
# channel over and one short of a block, the smallest that pad. What a neighbouring sample holds must not reach a padded
# channel: a sample of infinities leaves the others' results alone.
@pytest.mark.parametrize("geom", [
    (2, 33, 8, 18, 31, 3, 3, 1, 1, 1, 1), (3, 12, 6, 64, 13, 3, 3, 1, 1, 1, 1), (2, 95, 14, 14, 65, 3, 3, 1, 1, 1, 1), (2, 40, 9, 12, 20, 5, 5, 2, 2, 1, 1),
    (2, 47, 7, 9, 49, 3, 3, 1, 1, 1, 1), (3, 15, 11, 13, 48, 3, 3, 0, 0, 1, 1), (2, 70, 13, 9, 130, 3, 3, 1, 1, 2, 2), (2, 129, 10, 16, 79, 1, 1, 0, 0, 1, 1),
    (5, 300, 5, 5, 200, 1, 1, 0, 0, 1, 1),
    # large enough for the bfloat16 engine in both directions
    (2, 33, 40, 58, 31, 3, 3, 1, 1, 1, 1), (6, 12, 52, 64, 13, 3, 3, 1, 1, 1, 1), (4, 95, 26, 14, 65, 3, 3, 1, 1, 1, 1), (4, 40, 40, 40, 20, 5, 5, 2, 2, 1, 1),
    (11, 47, 31, 29, 49, 3, 3, 1, 1, 1, 1), (18, 15, 43, 45, 48, 3, 3, 0, 0, 1, 1), (12, 129, 40, 46, 79, 1, 1, 0, 0, 1, 1),
    # large enough for the float engine's padded loaders forward
    (13, 47, 31, 29, 149, 3, 3, 1, 1, 1, 1), (18, 70, 53, 37, 130, 3, 3, 1, 1, 2, 2)], ids=lambda g: "x".join(map(str, g)))
def test_padded_channels(ctx, geom):
    rng = np.random.default_rng(sum((i + 1) * v for i, v in enumerate(geom)))
    g, og = be.shape(*geom), oracle.shape(*geom)
    x = rnd(rng, (g.n, g.c, g.h, g.w))
    w = oracle.round_bf16((rng.standard_normal((g.k, g.c, g.r, g.s)) * np.sqrt(2.0 / (g.c * g.r * g.s))).astype(np.float32))
    want_y = oracle.conv_fwd(og, x, w, np.zeros(g.k, np.float32))
    dy = rnd(rng, want_y.shape)
    want_dx = oracle.conv_bwd_data(og, dy, w)
    xi, dyi = x.copy(), dy.copy()
    xi[1], dyi[1] = np.inf, -np.inf
    announce("padded channels", geom)
    for bf16 in (0, 1):
        check(lib.vdnn_ctx_set_activation_dtype(ctx.handle, bf16))
        try:
            with Dev(ctx) as d:
                up = d.act if bf16 else d.f32
                get = (lambda b, s: get_act(b, s)) if bf16 else (lambda b, s: b.download(s))
                close = assert_close_bf16 if bf16 else (lambda a, b, what: assert_close(a, b, TOL, what))
                dw = d.f32(w)
                for a, b, rows in ((x, dy, slice(None)), (xi, dyi, slice(0, 1))):
                    y, dx = up(np.zeros_like(want_y)), up(np.zeros_like(x))
                    check(lib.vdnn_conv_fwd(ctx.handle, None, g, 0, up(a).ptr, dw.ptr, None, y.ptr, None, 0))
                    check(lib.vdnn_conv_bwd_data(ctx.handle, None, g, 0, up(b).ptr, dw.ptr, dx.ptr, None, 0))
                    close(get(y, want_y.shape)[rows], want_y[rows], "fwd")
                    close(get(dx, x.shape)[rows], want_dx[rows], "bwd data")
        finally:
            check(lib.vdnn_ctx_set_activation_dtype(ctx.handle, 0))


def kernels_of(ctx, g, which, bf16):
    """Names of the kernels of one call on zeros."""
    P, Q = lib.vdnn_out_dim(g.h, g.pad_h, g.r, g.stride_h), lib.vdnn_out_dim(g.w, g.pad_w, g.s, g.stride_w)
    x, y, w = (g.n, g.c, g.h, g.w), (g.n, g.k, P, Q), (g.k, g.c, g.r, g.s)
    check(lib.vdnn_ctx_set_activation_dtype(ctx.handle, int(bf16)))
    try:
        with Dev(ctx) as d:
            act = lambda shape: d.act(np.zeros(shape, np.float32)) if bf16 else d.f32(np.zeros(shape, np.float32))
            a, b, f = act(x), act(y), d.f32(np.zeros(w, np.float32))
            be.profile_enable(ctx.handle, 1)
            if which == "fwd":
                check(lib.vdnn_conv_fwd(ctx.handle, None, g, 0, a.ptr, f.ptr, None, b.ptr, None, 0))
            elif which == "bwd data":
                check(lib.vdnn_conv_bwd_data(ctx.handle, None, g, 0, b.ptr, f.ptr, a.ptr, None, 0))
            else:
                check(lib.vdnn_conv_bwd_filter(ctx.handle, None, g, 0, a.ptr, b.ptr, f.ptr, None, 0))
            return set(be.profile_collect(ctx.handle))
    finally:
        be.profile_enable(ctx.handle, 0)
        check(lib.vdnn_ctx_set_activation_dtype(ctx.handle, 0))


# Which route a layer takes is decided by its size: on a grid of a few tiles the routes made for large layers were up to
# 2.9 times slower than those they replaced. (pass, bfloat16, geometry, part of the kernel's name, taken or not; both sides of
# each rule, by a factor of two or more)
@pytest.mark.parametrize("which,bf16,geom,name,taken", [
    # padded channels on the bfloat16 engine: windowed, pairs, single pixels
    ("fwd", 1, (1, 18, 8, 8, 16, 3, 3, 1, 1, 1, 1), "bf16", False), ("fwd", 1, (4, 95, 40, 40, 65, 3, 3, 1, 1, 1, 1), "bf16win", True),
    ("fwd", 1, (8, 12, 4, 4, 64, 1, 1, 0, 0, 1, 1), "bf16", False), ("fwd", 1, (12, 129, 60, 60, 79, 1, 1, 0, 0, 1, 1), "bf16mfma", True),
    ("bwd data", 1, (11, 57, 5, 5, 45, 2, 2, 1, 1, 1, 1), "bf16", False), ("bwd data", 1, (22, 47, 31, 29, 49, 3, 3, 1, 1, 1, 1), "bf16mfma", True),
    ("bwd data", 1, (27, 73, 95, 95, 16, 1, 1, 0, 0, 1, 1), "bf16", False),  # a reduction of half a block, however large the layer
    # padded rows on the bfloat16 engine: groups of four pixels, single pixels (strided)
    ("bwd filter", 1, (2, 12, 13, 13, 65, 5, 5, 2, 2, 1, 1), "bf16", False), ("bwd filter", 1, (24, 22, 13, 13, 165, 5, 5, 2, 2, 1, 1), "bf16", True),
    ("bwd filter", 1, (5, 26, 32, 32, 5, 3, 3, 1, 1, 2, 2), "bf16", False), ("bwd filter", 1, (28, 70, 41, 19, 130, 3, 3, 1, 1, 2, 2), "bf16", True),
    # strided backward data by residue classes
    ("bwd data", 0, (8, 96, 55, 55, 8, 2, 2, 1, 1, 2, 2), "classes", False), ("bwd data", 0, (8, 40, 64, 66, 64, 3, 3, 1, 1, 2, 2), "classes", True),
    ("bwd data", 0, (1, 17, 8, 8, 33, 3, 3, 1, 1, 2, 2), "classes", False), ("bwd data", 1, (4, 358, 40, 19, 4, 2, 2, 0, 0, 1, 3), "classes", False),
    ("bwd data", 1, (2, 34, 16, 16, 66, 3, 3, 1, 1, 2, 2), "classes", True),
    # padded channels of float layers: the filter re-laid-out or read as it is
    ("fwd", 0, (1, 46, 29, 29, 48, 2, 2, 0, 0, 1, 1), "pack", False), ("fwd", 0, (12, 200, 28, 28, 300, 3, 3, 1, 1, 1, 1), "pack", True),
    ("bwd data", 0, (2, 30, 12, 5, 46, 2, 2, 0, 0, 1, 1), "pack", False), ("bwd data", 0, (18, 95, 26, 14, 65, 3, 3, 1, 1, 1, 1), "pack", True),
    # one product of a strided layer: short reductions on 64x64 tiles, up to a size
    ("bwd data", 0, (2, 128, 128, 128, 2, 7, 7, 3, 3, 2, 2), "64x64", True), ("bwd data", 0, (22, 128, 128, 128, 2, 7, 7, 3, 3, 2, 2), "64x64", False),
], ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_route_by_size(ctx, which, bf16, geom, name, taken):
    announce("route", which, bf16, geom)
    names = kernels_of(ctx, be.shape(*geom), which, bf16)
    assert any(name in n for n in names) == taken, names
