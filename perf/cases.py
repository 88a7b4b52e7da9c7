"""The work that this framework is measured on: training steps through `Network`, and single layers through the C ABI.

A case is a dict of plain values. Four kinds:

  train  `steps` training steps of a network (forward and backward with the update inside backward), then every layer's
         trained parameters read into buffers that the program keeps: the unit between two checkpoints
  conv   one convolution layer on device tensors, `pass` "fwd" (bias and rectifier fused) or "bwd" (the gradients of
         input, filter and bias)
  block  what stands between two convolutions: rectifier, optional cross-channel normalisation, max-pooling, and the
         backward of each
  fc     one fully connected layer: forward with rectifier, gradients of the input, SGD update of weights and bias

Network tables, batch sizes, policies and options are those of this repository's configurations and benchmark; layer
sizes are those of the built-in networks and of the tests, odd ones among them.
"""
import ctypes as C
import math

import torch

from vdnn_implementation_amd import backend as be
from vdnn_implementation_amd import enums
from vdnn_implementation_amd.network import Network, layer_spec

lib, check = be.lib, be.check

NETS = {"alexnet": enums.ALEXNET, "alexnet_lrn": enums.ALEXNET_LRN, "overfeat": enums.OVERFEAT, "vgg16": enums.VGG16_128}
POLICIES = {"BASELINE": enums.BASELINE, "VDNN_NONE": enums.VDNN_NONE, "VDNN_CONV": enums.VDNN_CONV, "VDNN_ALL": enums.VDNN_ALL}
ALPHA = -1e-2  # the learning rate handed to the fully connected update, negated


def train(name, net, batch, steps, policy="BASELINE", perf=False, bf16=False, options=""):
    """options: words of the benchmark's rows: refined, fused, zvc, keep, inplace, recompute, ahead, budget (a third of
    BASELINE's memory)."""
    return {"name": name, "kind": "train", "net": net, "batch": batch, "steps": steps, "policy": policy, "perf": perf, "bf16": bf16, "options": options}


def small(name, batch, steps, hw, k1, k2, features, classes, bf16=False, options=""):
    """A small network of the tests' shape: 3x3 convolution, rectifier, normalisation, pooling, 5x5 convolution, rectifier,
    pooling, two fully connected layers, softmax."""
    c = train(name, "small", batch, steps, bf16=bf16, options=options)
    c.update(hw=hw, k1=k1, k2=k2, features=features, classes=classes)
    return c


def conv(name, way, n, c, h, w, k, r, pad, stride, bf16=False, perf=False):
    return {"name": name, "kind": "conv", "pass": way, "n": n, "c": c, "h": h, "w": w, "k": k, "r": r, "pad": pad, "stride": stride, "bf16": bf16, "perf": perf}


def block(name, n, c, h, w, window, lrn, bf16=False):
    return {"name": name, "kind": "block", "n": n, "c": c, "h": h, "w": w, "window": window, "lrn": lrn, "bf16": bf16}


def fc(name, n, c_in, c_out, bf16=False):
    return {"name": name, "kind": "fc", "n": n, "c_in": c_in, "c_out": c_out, "bf16": bf16}


def listed():
    return [
        # a network of a few thousand parameters (unit tests, first experiments): launches and host work are all of it
        small("train small f32", 4, 32, 20, 8, 12, 20, 10),
        # the smallest configured training job: AlexNet with LRN, batch 32, float, everything at its default
        train("train alexnet32 f32", "alexnet_lrn", 32, 8),
        # OverFeat, batch 128, float: the convolution inputs offloaded over the host link, the policy run literally
        train("train overfeat128 conv f32", "overfeat", 128, 4, policy="VDNN_CONV"),
        # VGG16, batch 64, perf-optimal kernels under VDNN_ALL with a third of BASELINE's memory as budget
        train("train vgg64 all perf", "vgg16", 64, 4, policy="VDNN_ALL", perf=True, options="refined fused zvc ahead budget"),
        # the headline: VGG16, batch 128, float, memory-optimal kernels, defaults
        train("train vgg128 f32", "vgg16", 128, 2),
        # VGG16, batch 128, bfloat16 activations under VDNN_ALL with the packed tensors kept on the device
        train("train vgg128 all bf16", "vgg16", 128, 6, policy="VDNN_ALL", bf16=True, options="refined fused zvc keep inplace recompute"),
        # one image through one convolution: scoring a single sample, where latency counts
        conv("conv fwd 1 image f32", "fwd", 1, 64, 56, 56, 128, 3, 1, 1),
        # forward of a middle layer in bfloat16 at an ordinary batch
        conv("conv fwd 256 bf16", "fwd", 32, 256, 28, 28, 512, 3, 1, 1, bf16=True),
        # backward of a float layer of no round sizes (an own network): strided 3x3, odd channels, odd planes
        conv("conv bwd ragged f32", "bwd", 21, 70, 53, 37, 130, 3, 1, 2),
        # backward of AlexNet's 5x5 layer in bfloat16: odd planes, a window that is not 3x3
        conv("conv bwd 5x5 bf16", "bwd", 64, 96, 27, 27, 256, 5, 2, 1, bf16=True),
        # AlexNet's first rectifier, normalisation and overlapping pooling, forward and backward
        block("block lrn pool f32", 64, 96, 55, 55, 3, True),
        # VGG16's first fully connected layer: a weight matrix far larger than the activations
        fc("fc 25088 f32", 64, 25088, 4096),
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _draw_train(rng):
    if rng.random() < 0.4:
        hw = rng.randint(12, 40)
        c = small("", _log(rng, 1, 64), 24, hw, _log(rng, 4, 48), _log(rng, 4, 64), _log(rng, 10, 200), _log(rng, 2, 100),
                  bf16=rng.random() < 0.3, options=rng.choice(["", "fused"]))
    else:
        net = rng.choice(["alexnet", "alexnet_lrn", "overfeat", "vgg16"])
        batch = _log(rng, 1, 128)
        how = rng.choice(["BASELINE", "BASELINE fused", "VDNN_NONE", "VDNN_CONV", "VDNN_ALL", "VDNN_ALL refined fused zvc keep",
                          "VDNN_ALL refined fused zvc ahead budget", "VDNN_ALL refined fused zvc keep inplace recompute"]).split(" ", 1)
        # the literal policies copy every tensor over the link: a batch of VGG16 that one would wait for
        if net == "vgg16" and how in (["VDNN_CONV"], ["VDNN_ALL"]):
            batch = min(batch, 32)
        steps = {"vgg16": 2}.get(net, 4) if batch > 32 else 6
        c = train("", net, batch, steps, policy=how[0], perf=rng.random() < 0.35, bf16=rng.random() < 0.4, options=how[1] if len(how) > 1 else "")
    return c


def _draw_conv(rng):
    r = rng.choice([1, 3, 3, 3, 3, 5, 11])
    stride = 4 if r == 11 else rng.choice([1, 1, 1, 1, 2])
    c = 3 if r == 11 else rng.choice([3, _log(rng, 8, 600), _log(rng, 8, 600), 16 * _log(rng, 1, 40), 64 * _log(rng, 1, 12)])
    k = rng.choice([_log(rng, 8, 600), 16 * _log(rng, 1, 40), 64 * _log(rng, 1, 12)])
    h = _log(rng, max(7, r), 224)
    w = rng.choice([h, h, h, _log(rng, max(7, r), 224)])
    pad = rng.choice([0, r // 2, r // 2]) if r < 11 else 0
    n = _log(rng, 1, 128)
    # no more than 4e11 multiply-adds and 2.5e8 elements a tensor
    while n > 1 and n * max(c * h * w, k * h * w // stride ** 2) > 2.5e8 or n * k * c * r * r * h * w / stride ** 2 > 4e11:
        n = (n + 1) // 2
    return conv("", rng.choice(["fwd", "bwd"]), n, c, h, w, k, r, pad, stride, bf16=rng.random() < 0.5, perf=rng.random() < 0.3)


def _draw_block(rng):
    h = _log(rng, 6, 224)
    w = rng.choice([h, h, _log(rng, 6, 224)])
    c = _log(rng, 8, 512)
    n = max(1, min(_log(rng, 1, 128), int(2e8 / (c * h * w))))
    return block("", n, c, h, w, rng.choice([2, 3]), rng.random() < 0.5, bf16=rng.random() < 0.5)


def _draw_fc(rng):
    return fc("", _log(rng, 1, 256), _log(rng, 64, 26000), _log(rng, 10, 4200), bf16=rng.random() < 0.5)


def draw(rng):
    p = rng.random()
    case = _draw_train(rng) if p < 0.4 else _draw_conv(rng) if p < 0.75 else _draw_block(rng) if p < 0.87 else _draw_fc(rng)
    case.pop("name")
    return case


# ---- networks ------------------------------------------------------------------------------------------------------

def _small_table(case):
    n, hw, k1, k2 = (case[k] for k in ("batch", "hw", "k1", "k2"))
    half = hw // 2
    quarter = (half - 3) // 2 + 1
    feat = k2 * quarter * quarter
    return [layer_spec(enums.FC_CONV, n, 3, hw, hw, 1, 1, k1, 3), layer_spec(enums.RELU, n, k1, hw, hw), layer_spec(enums.LRN, n, k1, hw, hw),
            layer_spec(enums.POOL, n, k1, hw, hw, 0, 2, 0, 2), layer_spec(enums.FC_CONV, n, k1, half, half, 2, 1, k2, 5), layer_spec(enums.RELU, n, k2, half, half),
            layer_spec(enums.POOL, n, k2, half, half, 0, 2, 0, 3), layer_spec(enums.FC_GEMM, n, feat, 1, 1, 0, 0, case["features"], 1),
            layer_spec(enums.RELU, n, case["features"], 1, 1), layer_spec(enums.FC_GEMM, n, case["features"], 1, 1, 0, 0, case["classes"], 1),
            layer_spec(enums.SOFTMAX, n, case["classes"], 1, 1)]


def _table_of(case):
    return {"layers": _small_table(case)} if case["net"] == "small" else {"cnn": NETS[case["net"]], "batch": case["batch"]}


def _network(case, seed):
    words = case["options"].split()
    assert set(words) <= {"refined", "fused", "zvc", "keep", "inplace", "recompute", "ahead", "budget"}
    kw = dict(refined="refined" in words, fuse="fused" in words, compress="zvc" in words, keep_packed="keep" in words, in_place="inplace" in words,
              recompute_first="recompute" in words, prefetch_within_peak="ahead" in words)
    if "budget" in words:
        with Network(policy=enums.BASELINE, plan_only=True, **_table_of(case)) as replay:
            assert replay.forwardPropagation() == 0 and replay.backwardPropagation() == 0
            peak = replay.stats()["peak_bytes_in_use"]
        kw.update(hbm_budget_bytes=peak // 3, plan_packed_fraction=0.63 if case["bf16"] else 0.60, offload_lag=-1)
    return Network(policy=POLICIES[case["policy"]], algo=enums.VDNN_PERF_OPT_ALGO if case["perf"] else enums.VDNN_MEMORY_OPT_ALGO, seed=seed, bf16=case["bf16"], **_table_of(case), **kw)


def _prepare_train(case, seed):
    net = _network(case, 1 + seed)  # input, labels and parameters are drawn from the seed by the constructor
    # one buffer per layer with parameters, the filter followed by the bias: what a checkpoint is written from
    fp = C.POINTER(C.c_float)
    out, reads = {}, []
    for l, s in enumerate(net.specs):
        if net.has_params(l):
            count = s.k * s.c * s.r * s.s
            buf = torch.empty(count + s.k, dtype=torch.float32, pin_memory=True)
            reads.append((l, C.cast(buf.data_ptr(), fp), C.cast(buf.data_ptr() + 4 * count, fp)))
            out["layer%d" % l] = buf
    return {"kind": "train", "net": net, "steps": case["steps"], "reads": reads, "out": out}


def _run_train(s):
    net = s["net"]
    for _ in range(s["steps"]):
        assert net.forwardPropagation() == 0
        assert net.backwardPropagation() == 0
    for l, filter_to, bias_to in s["reads"]:
        assert lib.vdnn_network_get_layer_params(net._h, l, filter_to, bias_to) == 0
    return s["out"]


def _work_train(case):
    macs = acts = params = 0
    with Network(plan_only=True, **_table_of(case)) as net:
        for l, s in enumerate(net.specs):
            y = math.prod(net.dst_shape(l))
            if net.has_params(l):
                macs += y * s.c * s.r * s.s
                params += s.k * (s.c * s.r * s.s + 1)
            if s.type != enums.RELU:  # a rectifier can be applied where its input is made
                acts += y
    elem = 2 if case["bf16"] else 4
    # an output is written and read in forward and read in backward, its gradient written and read; a parameter is read
    # in each direction and written once
    return {"flops": 6.0 * macs * case["steps"], "bytes": (5.0 * acts * elem + 3.0 * params * 4) * case["steps"] + 4.0 * params}


# ---- single layers -------------------------------------------------------------------------------------------------

_contexts = {}


def _context(bf16):
    """The program's device context for an element type of activations."""
    if bf16 not in _contexts:
        ctx = be.Context(pool_bytes=128 << 20)
        check(lib.vdnn_ctx_set_activation_dtype(ctx.handle, int(bf16)))
        _contexts[bf16] = ctx
    return _contexts[bf16].handle


def _block(shape, bf16=False):
    """A tensor that lies inside a larger allocation, as a block of the framework's own pool does."""
    dtype, head = (torch.bfloat16 if bf16 else torch.float32), 4096
    raw = torch.empty(head + math.prod(shape) * (2 if bf16 else 4), dtype=torch.uint8, device="cuda")
    return raw[head:].view(dtype).view(shape)


def _normal(shape, seed, which, scale=1.0, bf16=False):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 16 + which)
    return _block(shape, bf16).copy_(torch.randn(shape, generator=g, device="cuda").mul_(scale))


def _rectified(shape, seed, which, bf16):
    """An activation as it leaves a rectifier: half of its elements zero."""
    return _normal(shape, seed, which, bf16=bf16).clamp_(min=0)


def _gated(shape, seed, which, bf16, scale=1.0):
    """A gradient as it leaves a rectifier's backward: half of its elements zero."""
    return _normal(shape, seed, which, scale, bf16).mul_(_normal(shape, seed, which + 1) > 0)


def _conv_sizes(case):
    p = (case["h"] + 2 * case["pad"] - case["r"]) // case["stride"] + 1
    q = (case["w"] + 2 * case["pad"] - case["r"]) // case["stride"] + 1
    return (case["n"], case["c"], case["h"], case["w"]), (case["k"], case["c"], case["r"], case["r"]), (case["n"], case["k"], p, q)


def _prepare_conv(case, seed):
    xs, ws, ys = _conv_sizes(case)
    bf16, algo = case["bf16"], enums.VDNN_PERF_OPT_ALGO if case["perf"] else enums.VDNN_MEMORY_OPT_ALGO
    g = be.shape(case["n"], case["c"], case["h"], case["w"], case["k"], case["r"], case["r"], case["pad"], case["pad"], case["stride"], case["stride"])
    s = {"kind": "conv", "pass": case["pass"], "ctx": _context(bf16), "g": g, "algo": algo,
         "x": _rectified(xs, seed, 0, bf16), "w": _normal(ws, seed, 1, math.sqrt(2.0 / math.prod(ws[1:])))}
    passes = (0,) if case["pass"] == "fwd" else (1, 2)
    need = max(int(lib.vdnn_conv_workspace_bytes_dtype(g, algo, p, int(bf16))) for p in passes)
    s["workspace"] = torch.empty(need, dtype=torch.uint8, device="cuda") if need else None
    s["ws"] = (s["workspace"].data_ptr() if need else None, need)
    if case["pass"] == "fwd":
        s["b"], s["y"] = _normal((ys[1],), seed, 2), _block(ys, bf16)
    else:
        s["dy"] = _gated(ys, seed, 2, bf16)
        s["dx"], s["dw"], s["db"] = _block(xs, bf16), _block(ws), _block((ys[1],))
    return s


def _run_conv(s):
    ctx, g, algo, (ws, nws) = s["ctx"], s["g"], s["algo"], s["ws"]
    x, w = s["x"].data_ptr(), s["w"].data_ptr()
    if s["pass"] == "fwd":
        check(lib.vdnn_conv_fwd_relu(ctx, None, g, algo, x, w, s["b"].data_ptr(), s["y"].data_ptr(), ws, nws))
        return {"y": s["y"]}
    dy = s["dy"].data_ptr()
    check(lib.vdnn_conv_bwd_filter_bias(ctx, None, g, algo, x, dy, s["dw"].data_ptr(), s["db"].data_ptr(), ws, nws))
    check(lib.vdnn_conv_bwd_data_relu(ctx, None, g, algo, dy, w, x, s["dx"].data_ptr(), ws, nws))
    return {"dx": s["dx"], "dw": s["dw"], "db": s["db"]}


def _work_conv(case):
    xs, ws, ys = _conv_sizes(case)
    elem = 2 if case["bf16"] else 4
    flops = 2.0 * math.prod(ys) * math.prod(ws[1:])
    both = elem * (math.prod(xs) + math.prod(ys)) + 4 * (math.prod(ws) + ws[0])
    return {"flops": flops, "bytes": both} if case["pass"] == "fwd" else {"flops": 2 * flops, "bytes": both + elem * math.prod(xs) + 4 * math.prod(ws)}


def _pooled(case):
    return (case["n"], case["c"], (case["h"] - case["window"]) // 2 + 1, (case["w"] - case["window"]) // 2 + 1)


def _prepare_block(case, seed):
    xs, ys, bf16 = (case["n"], case["c"], case["h"], case["w"]), _pooled(case), case["bf16"]
    s = {"kind": "block", "lrn": case["lrn"], "ctx": _context(bf16), "dims": xs, "count": math.prod(xs),
         "g": be.shape(*xs, 0, case["window"], case["window"], 0, 0, 2, 2), "x": _normal(xs, seed, 0, 1.5, bf16), "dy": _normal(ys, seed, 1, 1.0, bf16)}
    for name in ("a", "da", "dx") + (("u", "du") if case["lrn"] else ()):
        s[name] = _block(xs, bf16)
    s["y"] = _block(ys, bf16)
    return s


def _run_block(s):
    ctx, g, count, (n, c, h, w) = s["ctx"], s["g"], s["count"], s["dims"]
    x, a, da, y, dy, dx = (s[k].data_ptr() for k in ("x", "a", "da", "y", "dy", "dx"))
    check(lib.vdnn_relu_fwd(ctx, None, count, x, a))
    if s["lrn"]:
        u, du = s["u"].data_ptr(), s["du"].data_ptr()
        check(lib.vdnn_lrn_fwd(ctx, None, n, c, h * w, a, u))
        check(lib.vdnn_maxpool_fwd(ctx, None, g, u, y))
        check(lib.vdnn_maxpool_bwd(ctx, None, g, u, y, dy, du))
        check(lib.vdnn_lrn_bwd(ctx, None, n, c, h * w, a, u, du, da))
    else:
        check(lib.vdnn_maxpool_fwd(ctx, None, g, a, y))
        check(lib.vdnn_maxpool_bwd(ctx, None, g, a, y, dy, da))
    check(lib.vdnn_relu_bwd(ctx, None, count, x, a, da, dx))
    return {"a": s["a"], "y": s["y"], "da": s["da"], "dx": s["dx"]}


def _work_block(case):
    x, y, elem = case["n"] * case["c"] * case["h"] * case["w"], math.prod(_pooled(case)), 2 if case["bf16"] else 4
    # through the entry points every layer's tensors are read and written: x, a (u), y forward; dy, da (du), dx and the
    # saved tensors backward
    passes = (2 + 1 + 2 + 3) if not case["lrn"] else (2 + 2 + 1 + 2 + 4 + 3)
    return {"bytes": float(elem * (passes * x + 2 * y)), "flops": 0.0 if not case["lrn"] else 30.0 * x}


def _prepare_fc(case, seed):
    n, ci, co, bf16 = case["n"], case["c_in"], case["c_out"], case["bf16"]
    return {"kind": "fc", "ctx": _context(bf16), "dims": (n, ci, co), "x": _rectified((n, ci), seed, 0, bf16), "w": _normal((co, ci), seed, 1, math.sqrt(2.0 / ci)),
            "b": _normal((co,), seed, 2), "dy": _gated((n, co), seed, 3, bf16, 1.0 / n), "y": _block((n, co), bf16), "dx": _block((n, ci), bf16)}


def _run_fc(s):
    ctx, (n, ci, co) = s["ctx"], s["dims"]
    x, w, b, dy = (s[k].data_ptr() for k in ("x", "w", "b", "dy"))
    check(lib.vdnn_fc_fwd_relu(ctx, None, n, ci, co, x, w, b, s["y"].data_ptr()))
    check(lib.vdnn_fc_bwd_data_relu(ctx, None, n, ci, co, dy, w, x, s["dx"].data_ptr()))
    check(lib.vdnn_fc_bwd_weight_sgd(ctx, None, n, ci, co, x, dy, w, ALPHA))
    check(lib.vdnn_fc_bwd_bias_sgd(ctx, None, n, co, dy, b, ALPHA))
    return {"y": s["y"], "dx": s["dx"], "w": s["w"], "b": s["b"]}


def _work_fc(case):
    n, ci, co, elem = case["n"], case["c_in"], case["c_out"], 2 if case["bf16"] else 4
    return {"flops": 6.0 * n * ci * co, "bytes": 4.0 * (3 * ci * co + 2 * co) + elem * n * (2 * ci + 2 * co)}


# ---- what perf calls -----------------------------------------------------------------------------------------------

def prepare(case, seed):
    return {"train": _prepare_train, "conv": _prepare_conv, "block": _prepare_block, "fc": _prepare_fc}[case["kind"]](case, seed)


def run(state):
    return {"train": _run_train, "conv": _run_conv, "block": _run_block, "fc": _run_fc}[state["kind"]](state)


def work(case):
    return {"train": _work_train, "conv": _work_conv, "block": _work_block, "fc": _work_fc}[case["kind"]](case)


def _tolerance_train(case):
    """What the trained parameters differ by when the initial ones are moved by one unit in their last place, or when the
    other algorithm mode computes the step (its sums run in another order), times four. A step moves the parameters
    by 1e-6 to 1e-3 of themselves. AlexNet and OverFeat at large batches saturate their softmax under this update rule, so
    rounding decides more there; with 8 significant bits it decides more everywhere."""
    large = case["batch"] > 32 and case["net"] != "small"
    if case["bf16"]:
        if case["net"] == "small":
            return {"rel": 1e-5, "max": 2e-4}
        if case["net"] == "vgg16":
            return {"rel": 1.6e-5, "max": 6e-4}
        return {"rel": 1e-3, "max": 0.1} if large else {"rel": 5e-5, "max": 4e-3}
    if case["net"] == "small":
        return {"rel": 5e-7, "max": 8e-6}
    if case["net"] == "vgg16":
        return {"rel": 1e-6, "max": 2.5e-5}
    return {"rel": 6e-6, "max": 2e-4} if large else {"rel": 1e-6, "max": 1e-4}


def tolerance(case):
    """Four times the difference from the same layer in 64 bits on the same inputs, as measured over the listed cases and
    ninety drawn ones."""
    if case["kind"] == "train":
        return _tolerance_train(case)
    if case["bf16"]:
        # one rounding to bfloat16 (2^-9 of a value at most, 1.7e-3 by norm); normalised values are rounded twice
        return {"rel": 7e-3, "max": 3e-2 if case["kind"] == "block" else 1.6e-2}
    if case["kind"] == "block":
        return {"rel": 4e-7, "max": 3e-6}
    if case["kind"] == "conv" and case["perf"]:
        return {"rel": 1.8e-5, "max": 1.9e-4}  # float operands as two bfloat16 parts: 4.5e-6 and 4.7e-5 seen
    return {"rel": 3e-6, "max": 1.5e-5}
