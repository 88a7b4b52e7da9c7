"""Backward pooling of planes of any extents (2x2 cells behind the last window, 3x3 planes that do not fit LDS) and backward filter of up
to four channels in chunks down to four pixels a thread, against the checker: pooling moves values, so to the bit."""
import numpy as np
import pytest

import oracle
import vdnn_implementation_amd.backend as be
from gpu_util import Dev, announce, gpu_conv_bwd_filter
from util import from_bf16_bits, to_bf16_bits
from vdnn_implementation_amd.backend import check, lib

pytestmark = pytest.mark.gpu

# n, c, h, w, window
POOLS = [(2, 3, 7, 9, 2), (1, 5, 2, 2, 2), (3, 2, 2, 3, 2), (4, 7, 13, 12, 2), (1, 3, 221, 190, 2),
         (1, 3, 117, 118, 3), (2, 2, 130, 131, 3), (1, 2, 99, 254, 3), (1, 1, 3, 16001, 3), (1, 1, 9001, 4, 3), (1, 2, 120, 127, 3)]


@pytest.mark.parametrize("gated", [False, True], ids=["plain", "gated"])
@pytest.mark.parametrize("bf16", [False, True], ids=["float", "bfloat16"])
@pytest.mark.parametrize("geom", POOLS, ids=lambda g: "x".join(map(str, g)))
def test_maxpool_backward(geom, bf16, gated):
    n, c, h, w, win = geom
    rng = np.random.default_rng(h + w)
    full = (n, c, h, w, 0, win, win, 0, 0, 2, 2)
    g, og = be.shape(*full), oracle.shape(*full)
    x = oracle.round_bf16(rng.standard_normal((n, c, h, w)).astype(np.float32))  # (eight significant bits: windows with ties)
    if gated:
        x = np.maximum(x, 0)
    y = oracle.maxpool_fwd(og, x)
    # small whole numbers: sums of the windows that share a winner are exact in either element type
    dy = rng.integers(-8, 9, y.shape).astype(np.float32)
    want = oracle.maxpool_bwd(og, x, y, dy)
    if gated:
        want = np.where(x > 0, want, 0)
    with be.Context(pool_bytes=256 << 20) as ctx, Dev(ctx) as d:
        if bf16:
            check(lib.vdnn_ctx_set_activation_dtype(ctx.handle, 1))
        dtype, put, get = (np.uint16, to_bf16_bits, from_bf16_bits) if bf16 else (np.float32, lambda a: a, lambda a: a)
        dx_, dy_, ddy, gx = d.up(put(x), dtype), d.up(put(y), dtype), d.up(put(dy), dtype), d.up(put(np.full_like(x, 7)), dtype)
        announce("pool", geom, bf16, gated)
        check((lib.vdnn_maxpool_bwd_relu if gated else lib.vdnn_maxpool_bwd)(ctx.handle, None, g, dx_.ptr, dy_.ptr, ddy.ptr, gx.ptr))
        assert np.array_equal(get(gx.download(x.shape, dtype)), want)


SPECIAL = [(2, 3, 7, 9, 2), (1, 5, 40, 31, 2), (3, 2, 2, 3, 2), (1, 3, 221, 190, 2), (1, 3, 117, 118, 3), (1, 2, 99, 254, 3), (5, 3, 21, 30, 3)]


@pytest.mark.parametrize("gated", [False, True], ids=["plain", "gated"])
@pytest.mark.parametrize("bf16", [False, True], ids=["float", "bfloat16"])
@pytest.mark.parametrize("geom", SPECIAL, ids=lambda g: "x".join(map(str, g)))
def test_maxpool_backward_of_values_that_do_not_compare(geom, bf16, gated):
    """NaN, infinities, the lowest value and both zeros in x, negative zeros in dy and gradients whose sums round: the checker's bits,
    whose sums begin with +0 and run over the windows row by row."""
    n, c, h, w, win = geom
    rng = np.random.default_rng(h * w)
    full = (n, c, h, w, 0, win, win, 0, 0, 2, 2)
    g, og = be.shape(*full), oracle.shape(*full)
    x = oracle.round_bf16(rng.standard_normal((n, c, h, w)).astype(np.float32))
    lowest = np.uint32(0xFF7F0000).view(np.float32) if bf16 else np.finfo(np.float32).min
    for value in (np.nan, np.inf, -np.inf, lowest, -0.0, 0.0):
        x[rng.random(x.shape) < 0.12] = value
    x[:, :, :2, :2] = -np.inf     # windows in which nothing exceeds the lowest value
    y = oracle.maxpool_fwd(og, x)
    dy = rng.standard_normal(y.shape).astype(np.float32)
    if bf16:
        dy = oracle.round_bf16(dy)
    dy[rng.random(y.shape) < 0.3] = -0.0
    want = oracle.maxpool_bwd(og, x, y, dy)
    if gated:
        want = np.where(x > 0, want, np.float32(0))
    if bf16:
        want = oracle.round_bf16(want)
    with be.Context(pool_bytes=256 << 20) as ctx, Dev(ctx) as d:
        if bf16:
            check(lib.vdnn_ctx_set_activation_dtype(ctx.handle, 1))
        dtype, put, get = (np.uint16, to_bf16_bits, from_bf16_bits) if bf16 else (np.float32, lambda a: a, lambda a: a)
        dx_, dy_, ddy, gx = d.up(put(x), dtype), d.empty(y.shape, dtype), d.up(put(dy), dtype), d.up(put(np.full_like(x, 7)), dtype)
        announce("pool of special values", geom, bf16, gated)
        check((lib.vdnn_maxpool_bwd_relu if gated else lib.vdnn_maxpool_bwd)(ctx.handle, None, g, dx_.ptr, dy_.ptr, ddy.ptr, gx.ptr))
        assert np.array_equal(get(gx.download(x.shape, dtype)).view(np.uint32), want.view(np.uint32))


# n, c, h, w, k, pad, stride; the last is one chunk of fewer pixels than threads
FILTERS = [(3, 3, 25, 25, 24, 1, 1), (9, 4, 31, 29, 8, 0, 1), (2, 1, 40, 37, 4, 1, 2), (30, 2, 45, 45, 12, 0, 2), (1, 3, 9, 11, 16, 1, 1)]


@pytest.mark.parametrize("geom", FILTERS, ids=lambda g: "x".join(map(str, g)))
def test_backward_filter_of_few_channels(geom):
    n, c, h, w, k, pad, stride = geom
    rng = np.random.default_rng(n + h)
    full = (n, c, h, w, k, 3, 3, pad, pad, stride, stride)
    g, og = be.shape(*full), oracle.shape(*full)
    p, q = (h + 2 * pad - 3) // stride + 1, (w + 2 * pad - 3) // stride + 1
    x, dy = rng.standard_normal((n, c, h, w)).astype(np.float32), rng.standard_normal((n, k, p, q)).astype(np.float32)
    f = rng.standard_normal((k, c, 3, 3)).astype(np.float32)
    want = oracle.conv_bwd_filter_sgd(og, x, dy, f, -0.5).astype(np.float64)
    with be.Context(pool_bytes=256 << 20) as ctx:
        announce("filter of few channels", geom)
        got = gpu_conv_bwd_filter(ctx, g, x, dy, f, -0.5)
    # a rounding per product at most, random signs: 2^-24 sqrt(products) of the sum by 2-norm
    assert np.linalg.norm(got - want) <= 2.0 ** -24 * np.sqrt(n * p * q) * np.linalg.norm(want)
