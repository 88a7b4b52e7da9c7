"""State that outlives a launch: the counters with which a split product adds up its own sums (csrc/mfma_gemm.h, sum_splits) and the packing
kernels' cursors. One set per stream, so that calls on several streams, overlapping or captured, leave nothing behind that a later call meets."""
import numpy as np
import pytest
import torch

import oracle
import vdnn_implementation_amd.backend as be
from gpu_util import Dev, announce
from test_gpu_zvc import Pinned, decode, tensor
from vdnn_implementation_amd.backend import check, lib

pytestmark = pytest.mark.gpu
COUNTER_SETS = 8  # streams that have counters of their own; beyond them a second kernel adds the sums up

# n, c, h, w, k, window; splits; whether the product adds them up itself
PRODUCTS = [((1, 16, 43, 32, 285, 5), 2, True), ((7, 177, 9, 1, 317, 1), 3, True), ((4, 38, 7, 27, 201, 5), 5, True), ((2, 48, 41, 3, 211, 3), 6, True),
            ((9, 89, 6, 8, 296, 5), 7, False), ((1, 108, 50, 14, 116, 5), 11, False), ((21, 33, 40, 41, 140, 3), None, True)]


@pytest.fixture(scope="module")
def ctx():
    with be.Context(pool_bytes=512 << 20) as c:
        yield c


def arrays(geom, seed=0):
    n, c, h, w, k, r = geom
    rng = np.random.default_rng(n + c + k + seed)
    return (be.shape(n, c, h, w, k, r, r, r // 2, r // 2), rng.standard_normal((n, c, h, w)).astype(np.float32),
            rng.standard_normal((k, c, r, r)).astype(np.float32), rng.standard_normal(k).astype(np.float32))


def other_streams(count):
    """Streams of the default priority whose handles differ."""
    streams = {}
    while len(streams) < count:
        s = torch.cuda.Stream()
        streams[s.cuda_stream] = s
    return list(streams.values())


@pytest.mark.parametrize("geom,splits,fused", PRODUCTS, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else "")
def test_split_sums_take_their_route_and_have_one_result(geom, splits, fused):
    """The limits of the sum inside the product: two to six splits, tiles whose remainder alone is split (splits None), a stream beyond
    those that have counters; either way the same bits."""
    g, x, f, b = arrays(geom)
    n, c, h, w, k, r = geom
    results = {}
    with be.Context(pool_bytes=512 << 20) as ctx, Dev(ctx) as d:
        dx, df, db, y = d.up(x), d.up(f), d.up(b), d.empty((n, k, h, w))
        streams = other_streams(COUNTER_SETS + 1)

        def run(stream):
            be.profile_enable(ctx.handle, True)
            check(lib.vdnn_conv_fwd_relu(ctx.handle, stream, g, 0, dx.ptr, df.ptr, db.ptr, y.ptr, None, 0))
            ctx.synchronize()
            profile = be.profile_collect(ctx.handle)
            be.profile_enable(ctx.handle, False)
            return y.download((n, k, h, w)), profile

        announce("split sums", geom)
        for s in streams[:COUNTER_SETS]:
            got, profile = run(s.cuda_stream)
            results.setdefault(got.tobytes(), []).append(s)
            assert ("reduce_splits" not in profile) == fused and any(name.endswith("64x64") for name in profile), profile.keys()
        got, profile = run(streams[COUNTER_SETS].cuda_stream)
        results.setdefault(got.tobytes(), []).append(None)
        seen = profile["reduce_splits"]["bytes"] / (4.0 * n * k * h * w) - 1
        assert seen == splits if splits else seen != round(seen)
        assert len(results) == 1
        want = np.maximum(oracle.conv_fwd(oracle.shape(n, c, h, w, k, r, r, r // 2, r // 2, 1, 1), x, f, b), 0)
        # a rounding per two products of random signs
        assert np.linalg.norm(got.astype(np.float64) - want) <= 2.0 ** -24 * np.sqrt(c * r * r / 2) * np.linalg.norm(want)


def test_calls_of_other_tile_counts_in_turn(ctx):
    """Every call finds the counters of its stream at zero whatever ran before it there."""
    sets = [arrays(geom) for geom, _, fused in PRODUCTS if fused]
    with Dev(ctx) as d:
        calls = []
        for g, x, f, b in sets:
            y = d.empty((g.n, g.k, g.h, g.w))
            calls.append((g, d.up(x), d.up(f), d.up(b), y))
        first = {}
        for turn in range(6):
            for i in (range(len(calls)) if turn % 2 == 0 else reversed(range(len(calls)))):
                g, x, f, b, y = calls[i]
                check(lib.vdnn_fill(ctx.handle, None, g.n * g.k * g.h * g.w, 7.0, y.ptr))
                check(lib.vdnn_conv_fwd(ctx.handle, None, g, 0, x.ptr, f.ptr, b.ptr, y.ptr, None, 0))
                got = y.download((g.n, g.k, g.h, g.w)).tobytes()
                assert first.setdefault(i, got) == got


def test_overlapping_calls_spoil_no_later_one(ctx):
    """Two streams of one context with split products at the same time: their partial sums share the staging area, so those results are not
    looked at; the call after them is right."""
    geoms = [(7, 177, 9, 1, 317, 1), (2, 48, 41, 3, 211, 3)]
    (g, x, f, b), (g2, x2, f2, b2) = arrays(geoms[0]), arrays(geoms[1])
    s1, s2 = other_streams(2)
    with Dev(ctx) as d:
        first, second = (d.up(x), d.up(f), d.up(b)), (d.up(x2), d.up(f2), d.up(b2))
        y, y2 = d.empty((g.n, g.k, g.h, g.w)), d.empty((g2.n, g2.k, g2.h, g2.w))
        call = lambda s, g, t, y: check(lib.vdnn_conv_fwd(ctx.handle, s, g, 0, t[0].ptr, t[1].ptr, t[2].ptr, y.ptr, None, 0))
        count = g.n * g.k * g.h * g.w
        call(None, g, first, y)
        want = y.download((count,))
        announce("overlapping split products")
        for _ in range(20):
            for _ in range(10):
                call(s1.cuda_stream, g, first, y)
                call(s2.cuda_stream, g2, second, y2)
            ctx.synchronize()
            for s in (s1.cuda_stream, s2.cuda_stream, None):
                check(lib.vdnn_fill(ctx.handle, s, count, 7.0, y.ptr))
                call(s, g, first, y)
                ctx.synchronize()
                assert np.array_equal(y.download((count,)), want)


def test_captured_product_beside_calls_of_its_stream(ctx):
    """A product recorded into a graph, replayed several times on another stream than the one it was recorded on, with calls of that stream in
    between: the same bits every time."""
    g, x, f, b = arrays((2, 48, 41, 3, 211, 3))
    recording, other = other_streams(2)
    shape = (g.n, g.k, g.h, g.w)
    with Dev(ctx) as d:
        dx, df, db, y, y2 = d.up(x), d.up(f), d.up(b), d.empty(shape), d.empty(shape)
        call = lambda s, y: check(lib.vdnn_conv_fwd(ctx.handle, s, g, 0, dx.ptr, df.ptr, db.ptr, y.ptr, None, 0))
        call(recording.cuda_stream, y)
        ctx.synchronize()
        want = y.download(shape)
        announce("captured split product")
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=recording):
            call(recording.cuda_stream, y)
        for _ in range(4):
            check(lib.vdnn_fill(ctx.handle, None, want.size, 7.0, y.ptr))
            ctx.synchronize()
            with torch.cuda.stream(other):
                graph.replay()
            ctx.synchronize()
            assert np.array_equal(y.download(shape), want)
            call(recording.cuda_stream, y2)
            ctx.synchronize()
            assert np.array_equal(y2.download(shape), want)


@pytest.mark.parametrize("staged", [False, True], ids=["direct", "staged"])
def test_many_offloads_in_flight_on_two_streams(ctx, staged):
    """A hundred and forty packing kernels on two streams: one stream's long tensor packs while the other's short ones come and go."""
    rng = np.random.default_rng(5)
    big, small = tensor(rng, 3_000_000, np.uint32, 0.4), [tensor(rng, int(rng.integers(1, 20000)), np.uint16, 0.5) for _ in range(7)]
    s1, s2 = other_streams(2)
    with Dev(ctx) as d:
        sources = [d.up(t, t.dtype) for t in [big] + small]
        todo = []
        for i in range(140):
            which = 0 if i % 35 == 0 else 1 + i % 7
            a = big if which == 0 else small[which - 1]
            need = lib.vdnn_zvc_buffer_bytes(a.size, a.itemsize)
            stage = d.empty((need,), np.uint8) if staged else None
            todo.append((a, sources[which], Pinned(ctx, need), stage, need, (s1 if which == 0 else s2).cuda_stream, Pinned(ctx, 8)))
        announce("offloads on two streams", staged)
        for a, src, host, stage, need, s, word in todo:
            if staged:
                check(lib.vdnn_zvc_offload_staged_async(ctx.handle, host.ptr, stage.ptr, need, src.ptr, a.size, a.itemsize, word.ptr, None, s, None, 0))
            else:
                check(lib.vdnn_zvc_offload_async(ctx.handle, host.ptr, src.ptr, a.size, a.itemsize, s))
        ctx.synchronize()
        for a, _, host, stage, need, s, word in todo:
            got, length = decode(host.view, a.size, a.dtype)
            assert np.array_equal(got, a)
            if staged:
                assert int(word.view.view(np.uint64)[0]) == length
        for _, _, host, _, _, _, word in todo:
            host.free()
            word.free()


def test_captured_offloads_of_a_context_that_has_no_cursors_left():
    """A hundred packing kernels recorded into one graph, the context's first call among them: cursors come in blocks of 64, so memory is taken
    while a stream is captured. Replayed several times with calls outside the graph in between."""
    rng = np.random.default_rng(6)
    tensors = [tensor(rng, int(rng.integers(1, 20000)), np.uint32, 0.5) for _ in range(100)]
    recording, other = other_streams(2)
    with be.Context(pool_bytes=512 << 20) as ctx, Dev(ctx) as d:
        sources = [d.up(t, t.dtype) for t in tensors]
        hosts = [Pinned(ctx, lib.vdnn_zvc_buffer_bytes(t.size, t.itemsize)) for t in tensors]
        call = lambda i, s: check(lib.vdnn_zvc_offload_async(ctx.handle, hosts[i].ptr, sources[i].ptr, tensors[i].size, tensors[i].itemsize, s))
        ctx.synchronize()
        torch.cuda.synchronize()
        announce("captured offloads")
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=recording):
            for i in range(len(tensors)):
                call(i, recording.cuda_stream)
        for _ in range(4):
            for host in hosts:
                host.view[:] = 0xAB
            with torch.cuda.stream(other):
                graph.replay()
            torch.cuda.synchronize()
            for t, host in zip(tensors, hosts):
                assert np.array_equal(decode(host.view, t.size, t.dtype)[0], t)
            call(0, None)
            ctx.synchronize()
            assert np.array_equal(decode(hosts[0].view, tensors[0].size, tensors[0].dtype)[0], tensors[0])
        for host in hosts:
            host.free()
