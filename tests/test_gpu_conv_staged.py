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
