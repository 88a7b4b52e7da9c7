"""Forward and backward data of bfloat16 layers from a copy with a pixel's channels side by side (csrc/conv_staged.h), against the checker."""
import numpy as np
import pytest

import oracle
import vdnn_implementation_amd.backend as be
from gpu_util import Dev, announce
from util import assert_close_bf16, from_bf16_bits, to_bf16_bits
from vdnn_implementation_amd.backend import check, lib

pytestmark = pytest.mark.gpu

# n, c, h, w, k, r, s, pad_h, pad_w, stride; staged: forward, backward data
GEOMS = [
    ((12, 96, 27, 27, 130, 5, 5, 2, 2, 1), (True, True)),    # tiles past the rows and the pixels, split reduction
    ((20, 70, 19, 33, 200, 3, 3, 1, 1, 1), (True, True)),    # channels padded to 96, filters to 224
    ((14, 64, 40, 25, 192, 5, 3, 0, 2, 1), (True, True)),     # a window that is not square, more padding than half of it
    ((20, 128, 35, 33, 640, 5, 5, 2, 1, 2), (True, False)),  # strided: backward data goes by residue classes
    ((400, 33, 11, 9, 320, 3, 3, 1, 1, 1), (True, True)),    # tiles over three samples
]


@pytest.mark.parametrize("geom,staged", GEOMS, ids=lambda g: "x".join(map(str, g)) if len(g) > 2 else "")
def test_against_oracle(geom, staged):
    n, c, h, w, k, r, s, ph, pw, stride = geom
    rng = np.random.default_rng(n + c + k)
    full = (n, c, h, w, k, r, s, ph, pw, stride, stride)
    g, og = be.shape(*full), oracle.shape(*full)
    x = oracle.round_bf16(np.maximum(rng.standard_normal((n, c, h, w)), 0).astype(np.float32))
    f = (rng.standard_normal((k, c, r, s)) * np.sqrt(2.0 / (c * r * s))).astype(np.float32)
    b = rng.standard_normal(k).astype(np.float32)
    rounded = oracle.round_bf16(f)
    want_y = oracle.conv_fwd(og, x, rounded, b)
    dy = oracle.round_bf16(rng.standard_normal(want_y.shape).astype(np.float32))
    want_dx = oracle.conv_bwd_data(og, dy, rounded)
    with be.Context(pool_bytes=256 << 20) as ctx, Dev(ctx) as d:
        check(lib.vdnn_ctx_set_activation_dtype(ctx.handle, 1))
        dx_, df, db, ddy = d.up(to_bf16_bits(x), np.uint16), d.up(f), d.up(b), d.up(to_bf16_bits(dy), np.uint16)
        y, gx = d.empty(want_y.shape, np.uint16), d.empty(x.shape, np.uint16)
        be.profile_enable(ctx.handle, True)
        announce("staged", geom, "fwd")
        check(lib.vdnn_conv_fwd(ctx.handle, None, g, 0, dx_.ptr, df.ptr, db.ptr, y.ptr, None, 0))
        assert_close_bf16(from_bf16_bits(y.download(want_y.shape, np.uint16)), want_y, "forward")
        copies = lambda: be.profile_collect(ctx.handle).get("conv_stage_pixels", {"launches": 0})["launches"]
        assert copies() == int(staged[0])
        announce("staged", geom, "bwd data")
        check(lib.vdnn_conv_bwd_data(ctx.handle, None, g, 0, ddy.ptr, df.ptr, gx.ptr, None, 0))
        plain = from_bf16_bits(gx.download(x.shape, np.uint16))
        assert_close_bf16(plain, want_dx, "backward data")
        assert copies() == int(staged[0]) + int(staged[1])
        be.profile_enable(ctx.handle, False)
        check(lib.vdnn_conv_bwd_data_relu(ctx.handle, None, g, 0, ddy.ptr, df.ptr, dx_.ptr, gx.ptr, None, 0))
        assert np.array_equal(from_bf16_bits(gx.download(x.shape, np.uint16)), np.where(x > 0, plain, 0))
        if lib.vdnn_conv_bwd_data_in_place_ok(g):
            check(lib.vdnn_conv_bwd_data_relu(ctx.handle, None, g, 0, ddy.ptr, df.ptr, dx_.ptr, dx_.ptr, None, 0))
            assert np.array_equal(from_bf16_bits(dx_.download(x.shape, np.uint16)), np.where(x > 0, plain, 0))


# n, c, h, w, k, window, pad, stride; whether forward takes the copy
ROUTES = [((12, 96, 27, 27, 130, 5, 2, 1), True), ((24, 608, 45, 45, 80, 5, 2, 2), False),  # (one of five splits left)
          ((34, 111, 160, 45, 5, 5, 0, 2), True),    # two of seven splits left, whose rounds take as long
          ((2, 255, 120, 218, 3, 3, 0, 1), False),   # pairs of pixels, nine taps
          ((20, 96, 40, 40, 192, 5, 2, 1), True),    # pairs, twenty-five taps
          ((123, 16, 38, 38, 16, 5, 2, 1), True),    # pairs; sixteen channels are multiplied as a block of thirty-two
          ((5, 202, 143, 143, 112, 2, 1, 1), False)]  # four taps


@pytest.mark.parametrize("geom,staged", ROUTES, ids=lambda g: "x".join(map(str, g)) if isinstance(g, tuple) else "")
def test_copies_only_where_they_pay(geom, staged):
    n, c, h, w, k, r, pad, stride = geom
    p, q = (h + 2 * pad - r) // stride + 1, (w + 2 * pad - r) // stride + 1
    g = be.shape(n, c, h, w, k, r, r, pad, pad, stride, stride)
    with be.Context(pool_bytes=512 << 20) as ctx, Dev(ctx) as d:
        check(lib.vdnn_ctx_set_activation_dtype(ctx.handle, 1))
        x, f, b, y = d.empty((n, c, h, w), np.uint16), d.empty((k, c, r, r)), d.empty((k,)), d.empty((n, k, p, q), np.uint16)
        for buf, count in ((f, k * c * r * r), (b, k)):
            buf.upload(np.zeros(count, np.float32))
        x.upload(np.zeros((n, c, h, w), np.uint16))
        be.profile_enable(ctx.handle, True)
        announce("copy or not", geom)
        check(lib.vdnn_conv_fwd(ctx.handle, None, g, 0, x.ptr, f.ptr, b.ptr, y.ptr, None, 0))
        assert ("conv_stage_pixels" in be.profile_collect(ctx.handle)) == staged
