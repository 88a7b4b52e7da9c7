"""Float convolutions computed on the bfloat16 matrix cores at float precision (csrc/conv_same_f32x3.h) against the checker, whose
sums are in double. A sum of K products meets a rounding of 2^-24 per eight products at most; random signs make that
2^-24 sqrt(K / 8) of the result, by 2-norm."""
import numpy as np
import pytest

import oracle
import vdnn_implementation_amd.backend as be
from gpu_util import Dev, announce
from vdnn_implementation_amd.backend import check, lib

pytestmark = pytest.mark.gpu

# n, c, h, w, k, window: both channel counts multiples of 16 where both directions take the kernel
GEOMS = [
    (5, 32, 58, 62, 256, 3),     # even rows, pixels no multiple of a tile
    (9, 48, 29, 31, 160, 5),     # odd rows, two and a half row tiles, split reduction
    (30, 96, 13, 13, 320, 3),    # planes smaller than a tile
    (4, 64, 72, 70, 48, 5),      # fewer rows than a tile, even rows under a 5x5 window
    (91, 112, 11, 9, 144, 3),    # odd rows, tiles over three samples
    (3, 528, 5, 256, 100, 3),    # rows as long as a tile; backward data stays on the float engine (100 reduced channels)
    (40, 32, 37, 37, 256, 3),    # whole rounds of tiles and a split rest
]


@pytest.fixture(scope="module")
def ctx():
    with be.Context(pool_bytes=256 << 20) as c:
        yield c


def norm_error(got, want):
    return np.linalg.norm(got.astype(np.float64) - want) / np.linalg.norm(want.astype(np.float64))


@pytest.mark.parametrize("geom", GEOMS, ids=lambda g: "x".join(map(str, g)))
def test_forward_and_backward_data_against_oracle(ctx, geom):
    n, c, h, w, k, r = geom
    rng = np.random.default_rng(n * 1000 + c)
    full = (n, c, h, w, k, r, r, r // 2, r // 2, 1, 1)
    g, og = be.shape(*full), oracle.shape(*full)
    x = np.maximum(rng.standard_normal((n, c, h, w)), 0).astype(np.float32)
    f = (rng.standard_normal((k, c, r, r)) * np.sqrt(2.0 / (c * r * r))).astype(np.float32)
    b = rng.standard_normal(k).astype(np.float32)
    want_y = oracle.conv_fwd(og, x, f, b)
    dy = rng.standard_normal(want_y.shape).astype(np.float32)
    want_dx = oracle.conv_bwd_data(og, dy, f)
    with Dev(ctx) as d:
        dx_, df, db, ddy = d.up(x), d.up(f), d.up(b), d.up(dy)
        y, gx = d.empty(want_y.shape), d.empty(x.shape)
        be.profile_enable(ctx.handle, True)
        announce("x3", geom, "fwd")
        check(lib.vdnn_conv_fwd(ctx.handle, None, g, 0, dx_.ptr, df.ptr, db.ptr, y.ptr, None, 0))
        first = y.download(want_y.shape)
        assert norm_error(first, want_y) <= 2.0 ** -24 * np.sqrt(c * r * r / 8)
        check(lib.vdnn_conv_fwd_relu(ctx.handle, None, g, 0, dx_.ptr, df.ptr, db.ptr, y.ptr, None, 0))
        assert np.array_equal(y.download(want_y.shape), np.maximum(first, 0))
        announce("x3", geom, "bwd data")
        check(lib.vdnn_conv_bwd_data(ctx.handle, None, g, 0, ddy.ptr, df.ptr, gx.ptr, None, 0))
        plain = gx.download(x.shape)
        # (one rounding per two products where the float engine computes it)
        assert norm_error(plain, want_dx) <= 2.0 ** -24 * np.sqrt(k * r * r / (8 if k % 16 == 0 else 2))
        check(lib.vdnn_conv_bwd_data_relu(ctx.handle, None, g, 0, ddy.ptr, df.ptr, dx_.ptr, dx_.ptr, None, 0))  # over the gating input
        assert np.array_equal(dx_.download(x.shape), np.where(x > 0, plain, 0))
        ran = be.profile_collect(ctx.handle)
        be.profile_enable(ctx.handle, False)
        assert ran["conv_fwd_x3_64x256"]["launches"] == 2
        assert ("conv_bwd_data_x3_64x256" in ran) == (k % 16 == 0)


@pytest.mark.parametrize("geom", [(5, 32, 58, 62, 256, 3), (9, 48, 29, 31, 160, 5)], ids=lambda g: "x".join(map(str, g)))
def test_values_without_three_parts(ctx, geom):
    """Infinities, NaN and floats that round to an infinite bfloat16 value reach the results that the checker's products reach, as
    they do on the float instruction, and no others."""
    n, c, h, w, k, r = geom
    rng = np.random.default_rng(3)
    full = (n, c, h, w, k, r, r, r // 2, r // 2, 1, 1)
    g, og = be.shape(*full), oracle.shape(*full)
    x = rng.standard_normal((n, c, h, w)).astype(np.float32)
    f = (rng.standard_normal((k, c, r, r)) * np.sqrt(2.0 / (c * r * r))).astype(np.float32)
    x[0, 1, 3, 0], x[0, 2, h - 1, w - 1], x[n - 1, 0, 0, 5], x[n - 1, 7, 9, 9] = np.inf, -np.inf, np.nan, 3.4e38
    f[5, :, 0, 0] = 0.0   # an infinity times zero is NaN
    want = oracle.conv_fwd(og, x, f, np.zeros(k, np.float32))
    with Dev(ctx) as d:
        dx_, df, y = d.up(x), d.up(f), d.empty(want.shape)
        announce("x3 special values", geom)
        check(lib.vdnn_conv_fwd(ctx.handle, None, g, 0, dx_.ptr, df.ptr, None, y.ptr, None, 0))
        got = y.download(want.shape)
    assert np.isnan(want).any() and np.isposinf(want).any() and np.isneginf(want).any()
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(np.isposinf(got), np.isposinf(want)) and np.array_equal(np.isneginf(got), np.isneginf(want))
    ordinary = np.isfinite(want) & (np.abs(want) < 1e6)
    assert norm_error(got[ordinary], want[ordinary]) <= 2.0 ** -24 * np.sqrt(c * r * r / 2)
    large = np.isfinite(want) & (np.abs(want) > 1e30)
    assert large.any() and np.allclose(got[large], want[large], rtol=1e-5, atol=0)
