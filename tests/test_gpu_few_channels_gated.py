"""Gated backward data of layers with up to four input channels (the products of all taps formed once, then gathered): against the
checker, whose sums are in double. Floats: a result is the sum of R*S partial sums of K products each, a rounding of 2^-24 per two products and
one per tap, with random signs 2^-24 sqrt(K R S / 2) of the result by 2-norm; bfloat16 results are rounded once, 2^-9."""
import numpy as np
import pytest

import oracle
import vdnn_implementation_amd.backend as be
from gpu_util import Dev, announce
from util import from_bf16_bits, to_bf16_bits
from vdnn_implementation_amd.backend import check, lib

pytestmark = pytest.mark.gpu

# n, c, h, w, k, window, pad, stride
GEOMS = [
    (3, 3, 37, 29, 20, 11, 0, 4),    # rows and columns no tap reaches behind the last output
    (2, 3, 15, 17, 33, 5, 2, 1),
    (5, 2, 19, 23, 48, 3, 1, 1),     # the row kernel of up to 64 filters
    (4, 4, 21, 18, 24, 3, 0, 2),
    (1, 1, 9, 9, 7, 5, 2, 2),
    (2, 3, 20, 21, 8, 2, 0, 3),      # pixels between the windows
    (40, 3, 64, 64, 70, 5, 2, 1),
    (75, 3, 64, 64, 70, 5, 2, 1),    # more products than the staging area holds at a time: 53 samples, then 22
    (47, 4, 150, 150, 33, 7, 3, 2),  # ... of a strided layer: 14 samples three times, then 5
    (2, 3, 12, 12, 9, 1, 0, 2),      # one tap
]


@pytest.mark.parametrize("bf16", [False, True], ids=["float", "bfloat16"])
@pytest.mark.parametrize("geom", GEOMS, ids=lambda g: "x".join(map(str, g)))
def test_gated_backward_data(geom, bf16):
    n, c, h, w, k, r, pad, stride = geom
    rng = np.random.default_rng(n + c + k + r)
    full = (n, c, h, w, k, r, r, pad, pad, stride, stride)
    g, og = be.shape(*full), oracle.shape(*full)
    rounded = oracle.round_bf16 if bf16 else (lambda a: a)
    x = rounded(rng.standard_normal((n, c, h, w)).astype(np.float32))
    f = rng.standard_normal((k, c, r, r)).astype(np.float32)
    p, q = (h + 2 * pad - r) // stride + 1, (w + 2 * pad - r) // stride + 1
    dy = rounded(rng.standard_normal((n, k, p, q)).astype(np.float32))
    want = np.where(x > 0, oracle.conv_bwd_data(og, dy, rounded(f)), 0).astype(np.float64)
    with be.Context(pool_bytes=256 << 20) as ctx, Dev(ctx) as d:
        if bf16:
            check(lib.vdnn_ctx_set_activation_dtype(ctx.handle, 1))
        dtype, put, get = (np.uint16, to_bf16_bits, from_bf16_bits) if bf16 else (np.float32, lambda a: a, lambda a: a)
        dx_, df, ddy, gx = d.up(put(x), dtype), d.up(f), d.up(put(dy), dtype), d.up(put(np.full_like(x, 7)), dtype)
        be.profile_enable(ctx.handle, True)
        announce("few channels, gated", geom, bf16)
        check(lib.vdnn_conv_bwd_data_relu(ctx.handle, None, g, 0, ddy.ptr, df.ptr, dx_.ptr, gx.ptr, None, 0))
        got = get(gx.download(x.shape, dtype)).astype(np.float64)
        gathers = be.profile_collect(ctx.handle).get("conv_bwd_data_gather", {"launches": 0})["launches"]
    if n > 40 and (stride > 1 or not bf16):
        assert gathers == -(-n // (66060288 // (c * r * r * p * q * 4)))  # chunks of what 63 MB hold
    assert np.all(got[x <= 0] == 0)
    error = np.linalg.norm(got - want) / np.linalg.norm(want)
    assert error <= (2.0 ** -9 if bf16 else 2.0 ** -24 * max(np.sqrt(k * r * r / 2), 2))


# n, c, h, w, k, window, pad, stride; whether the products are formed once (a float layer)
ROUTES = [(3, 3, 60, 60, 96, 11, 5, 1, True), (20, 4, 54, 54, 1, 11, 5, 1, False), (8, 3, 62, 62, 2, 7, 3, 1, False), (25, 4, 110, 110, 3, 2, 1, 1, False),
          (23, 3, 88, 88, 64, 11, 0, 4, True), (87, 3, 40, 40, 12, 3, 0, 2, True)]


@pytest.mark.parametrize("geom", ROUTES, ids=lambda g: "x".join(map(str, g)))
def test_products_only_where_they_pay(geom):
    """Few filters at stride 1 read little as one product of C rows: the products of all taps and the gather took up to eleven times as long."""
    n, c, h, w, k, r, pad, stride, products = geom
    p, q = (h + 2 * pad - r) // stride + 1, (w + 2 * pad - r) // stride + 1
    g = be.shape(n, c, h, w, k, r, r, pad, pad, stride, stride)
    with be.Context(pool_bytes=256 << 20) as ctx, Dev(ctx) as d:
        x, f, dy, dx = (d.up(np.ones(s, np.float32)) for s in ((n, c, h, w), (k, c, r, r), (n, k, p, q), (n, c, h, w)))
        be.profile_enable(ctx.handle, True)
        announce("products or not", geom)
        check(lib.vdnn_conv_bwd_data_relu(ctx.handle, None, g, 0, dy.ptr, f.ptr, x.ptr, dx.ptr, None, 0))
        assert ("conv_bwd_data_gather" in be.profile_collect(ctx.handle)) == products


@pytest.mark.parametrize("k,row_kernel", [(2, False), (64, True)])
def test_row_kernel_only_where_it_pays(k, row_kernel):
    g = be.shape(40, 3, 80, 80, k, 3, 3, 1, 1)
    with be.Context(pool_bytes=256 << 20) as ctx, Dev(ctx) as d:
        x, f, dy, dx = (d.up(np.ones(s, np.float32)) for s in ((40, 3, 80, 80), (k, 3, 3, 3), (40, k, 80, 80), (40, 3, 80, 80)))
        be.profile_enable(ctx.handle, True)
        check(lib.vdnn_conv_bwd_data_relu(ctx.handle, None, g, 0, dy.ptr, f.ptr, x.ptr, dx.ptr, None, 0))
        assert ("conv_bwd_data_smallc" in be.profile_collect(ctx.handle)) == row_kernel
