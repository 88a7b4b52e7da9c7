"""Streaming kernels of fully connected layers (csrc/fc_update.h, csrc/fc_stream.h) against the same sums in double: a sum of n products
rounds once per two, 2^-24 sqrt(n / 2) of it by 2-norm with random signs, and the update's multiply-add once more."""
import numpy as np
import pytest

import vdnn_implementation_amd.backend as be
from gpu_util import Dev, announce
from vdnn_implementation_amd.backend import check, lib

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    with be.Context(pool_bytes=256 << 20) as c:
        yield c


# rows, inputs, outputs: one row; rows that end within a slice; outputs and inputs that end within a tile; the largest batch
@pytest.mark.parametrize("n,c_in,c_out", [(1, 1024, 1024), (17, 1028, 1023), (33, 132, 8000), (64, 25088, 100), (128, 4100, 700)])
def test_filter_update(ctx, n, c_in, c_out):
    rng = np.random.default_rng(n)
    x = np.maximum(rng.standard_normal((n, c_in)), 0).astype(np.float32)
    dy = rng.standard_normal((n, c_out)).astype(np.float32)
    w = rng.standard_normal((c_out, c_in)).astype(np.float32)
    alpha = np.float32(-0.37)
    want = dy.T.astype(np.float64) @ x.astype(np.float64)
    guard = np.full(64, 7.0, np.float32)
    with Dev(ctx) as d:
        dx_, ddy = d.up(x), d.up(dy)
        out, upd = d.up(np.concatenate([np.zeros(w.size, np.float32), guard])), d.up(np.concatenate([w.ravel(), guard]))
        announce("fc update", n, c_in, c_out)
        check(lib.vdnn_fc_bwd_weight(ctx.handle, None, n, c_in, c_out, dx_.ptr, ddy.ptr, out.ptr))
        check(lib.vdnn_fc_bwd_weight_sgd(ctx.handle, None, n, c_in, c_out, dx_.ptr, ddy.ptr, upd.ptr, alpha))
        got, got_w = out.download((w.size + 64,)), upd.download((w.size + 64,))
    assert np.array_equal(got[w.size:], guard) and np.array_equal(got_w[w.size:], guard)
    got, got_w = got[:w.size].reshape(w.shape), got_w[:w.size].reshape(w.shape)
    assert np.linalg.norm(got - want) <= 2.0 ** -24 * np.sqrt(max(n, 2) / 2) * np.linalg.norm(want)
    # one multiply-add of the same sum
    assert np.allclose(got_w, w + np.float64(alpha) * got, rtol=2.0 ** -23, atol=2.0 ** -23)


# rows, inputs, outputs: one row; splits that end in half a fetch; outputs (inputs) that end within a wavefront's columns; the most rows
@pytest.mark.parametrize("n,c_in,c_out", [(1, 4096, 3072), (7, 4208, 3088), (31, 12592, 1008), (32, 1008, 12592)])
def test_forward_and_backward_data_of_few_rows(ctx, n, c_in, c_out):
    rng = np.random.default_rng(n + 10)
    x = np.maximum(rng.standard_normal((n, c_in)), 0).astype(np.float32)
    dy = rng.standard_normal((n, c_out)).astype(np.float32)
    w = (rng.standard_normal((c_out, c_in)) * np.sqrt(2.0 / c_in)).astype(np.float32)
    b = rng.standard_normal(c_out).astype(np.float32)
    want_y, want_dx = x.astype(np.float64) @ w.T.astype(np.float64) + b, dy.astype(np.float64) @ w.astype(np.float64)
    with Dev(ctx) as d:
        dx_, ddy, dw, db, y, gx = d.up(x), d.up(dy), d.up(w), d.up(b), d.empty((n, c_out)), d.empty((n, c_in))
        announce("fc stream", n, c_in, c_out)
        check(lib.vdnn_fc_fwd(ctx.handle, None, n, c_in, c_out, dx_.ptr, dw.ptr, db.ptr, y.ptr))
        plain_y = y.download((n, c_out))
        check(lib.vdnn_fc_fwd_relu(ctx.handle, None, n, c_in, c_out, dx_.ptr, dw.ptr, db.ptr, y.ptr))
        assert np.array_equal(y.download((n, c_out)), np.maximum(plain_y, 0))
        check(lib.vdnn_fc_bwd_data(ctx.handle, None, n, c_in, c_out, ddy.ptr, dw.ptr, gx.ptr))
        plain = gx.download((n, c_in))
        check(lib.vdnn_fc_bwd_data_relu(ctx.handle, None, n, c_in, c_out, ddy.ptr, dw.ptr, dx_.ptr, gx.ptr))
        gated = gx.download((n, c_in))
    assert np.linalg.norm(plain_y - want_y) <= 2.0 ** -24 * np.sqrt(c_in / 2) * np.linalg.norm(want_y)
    # (many splits of a small plain result are added up by another kernel than a gated one's)
    for got, want in ((plain, want_dx), (gated, np.where(x > 0, want_dx, 0))):
        assert np.linalg.norm(got - want) <= 2.0 ** -24 * np.sqrt(c_out / 2) * np.linalg.norm(want)
    assert not gated[x <= 0].any()
