"""The work that a user of this backend has it do, as cases that can be timed and compared.

A case is a dict of plain values; `prepare` makes what a program holds before the call (device-resident inputs and
parameters, the compiled plan or the output buffers), `run` makes one pass through the public entry points and returns
its outputs as torch views of the buffers they lie in, `work` counts what a pass cannot do without.

Kinds:
  train   one training step of a network (forward, backward, update) through the plan and an optimizer
  predict the inference outputs of a network for one batch through a plan
  conv    a convolution and its two gradients, called as single operations
  matmul  a matrix product and its two gradients, called as single operations
  block   bias, batch norm, relu, max-pool and their gradients, called one by one (a plan without rewrites)
  tensor  pointwise, reduction and layout operations on one matrix, called one by one
  update  the multi-tensor optimizer on its own
"""
import math

import numpy as np
import torch

from dopt_amd import capi, configs, core, data, nnet, online, ops, workloads

F32 = np.float32


def listed():
    return [
        # the reference's softmax-regression example: 13 tiny dependent kernels, launch latency and nothing else
        {"name": "logit b100", "kind": "train", "net": "logit", "batch": 100, "rule": "sgd", "fused": False},
        # the 784-512-512-10 network at batch 256: dense layers that fill a fraction of the chip, fused ADAM
        {"name": "mlp b256", "kind": "train", "net": "mlp", "batch": 256, "width": 512, "rule": "adam", "fused": True},
        # the headline: VGG-16 with batch norm on 32 x 32 images at batch 128
        {"name": "vgg16 b128", "kind": "train", "net": "vgg", "batch": 128, "width": 64, "rule": "sgd", "fused": True},
        # the same network half as wide at batch 100, every batch from host memory through the augmenting feed
        {"name": "vgg half b100 host", "kind": "train", "net": "vgg", "batch": 100, "width": 32, "rule": "sgd",
         "fused": True, "feed": "host"},
        # the largest network the repository trains
        {"name": "wrn-28-10 b128", "kind": "train", "net": "wrn", "batch": 128, "depth": 28, "width": 10, "rule": "adam",
         "fused": True},
        # its small sibling with an update rule written as a graph, as the reference's own optimizers are
        {"name": "wrn-10-2 b64 graph", "kind": "train", "net": "wrn", "batch": 64, "depth": 10, "width": 2,
         "rule": "amsgrad", "fused": False},
        # a single image through the trained network: latency
        {"name": "vgg16 predict b1", "kind": "predict", "net": "vgg", "batch": 1, "width": 64},
        # a test-set batch of an odd size
        {"name": "wrn-28-10 predict b250", "kind": "predict", "net": "wrn", "batch": 250, "depth": 28, "width": 10},
        # filters and images no configuration has: 5 x 5, stride 2, odd sides and channel counts
        {"name": "conv 5x5 s2 ragged", "kind": "conv", "n": 50, "c": 48, "h": 45, "w": 39, "k": 100, "r": 5, "pad": 2,
         "stride": 2},
        # a large product and the two products of its gradient
        {"name": "matmul 4096", "kind": "matmul", "m": 4096, "n": 4096, "k": 4096},
        # the operations of one layer called singly, on the largest activation of the headline network
        {"name": "layer ops b128", "kind": "block", "n": 128, "c": 64, "h": 32, "w": 32},
        # AMSGrad over 16.8 M parameters in forty tensors of 4 K to 2.4 M values
        {"name": "amsgrad 16M", "kind": "update", "rule": "amsgrad", "total": 1 << 24, "tensors": 40},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _flops_limit():
    return 4.0e12


def draw(rng):
    while True:
        case = _draw(rng)
        w = work(case)
        # at most what the largest listed network costs, in arithmetic and in traffic
        if w["flops"] <= _flops_limit() and w["bytes"] <= 1.5e9:
            return case


def _draw(rng):
    kind = rng.choice(["train", "train", "train", "predict", "conv", "matmul", "block", "tensor", "update"])
    rule = rng.choice(["sgd", "adam", "amsgrad"])
    if kind in ("train", "predict"):
        net = rng.choice(["logit", "mlp", "vgg", "wrn"] if kind == "train" else ["mlp", "vgg", "wrn"])
        case = {"kind": kind, "net": net, "batch": _log_int(rng, 1, 512) if kind == "predict" else _log_int(rng, 8, 256)}
        if net == "logit":
            case["batch"] = _log_int(rng, 16, 512)
        elif net == "mlp":
            case["width"] = _log_int(rng, 64, 2048)
        elif net == "vgg":
            case["batch"] = max(case["batch"], 1 if kind == "predict" else 64)
            case["width"] = rng.choice([8, 16, 24, 32, 48, 64, 80])
        else:
            case["depth"], case["width"] = rng.choice([10, 16, 22]), rng.choice([1, 2, 4, 6, 10])
        if kind == "train":
            case["rule"], case["fused"] = rule, net != "logit" and rng.random() < 0.7
            if net in ("vgg", "wrn") and rng.random() < 0.3:
                case["feed"] = "host"
        return case
    if kind == "conv":
        r = rng.choice([1, 3, 3, 3, 5])
        return {"kind": kind, "n": _log_int(rng, 1, 256), "c": _log_int(rng, 3, 640), "h": _log_int(rng, 4, 64),
                "w": _log_int(rng, 4, 64), "k": _log_int(rng, 8, 640), "r": r, "pad": rng.choice([r // 2, r // 2, 0]),
                "stride": rng.choice([1, 1, 2])}
    if kind == "matmul":
        return {"kind": kind, "m": _log_int(rng, 16, 8192), "n": _log_int(rng, 10, 8192), "k": _log_int(rng, 16, 8192)}
    if kind == "block":
        return {"kind": kind, "n": _log_int(rng, 4, 256), "c": _log_int(rng, 8, 640), "h": 2 * _log_int(rng, 1, 32),
                "w": 2 * _log_int(rng, 1, 32)}
    if kind == "tensor":
        return {"kind": kind, "rows": _log_int(rng, 64, 65536), "cols": _log_int(rng, 10, 4096)}
    return {"kind": kind, "rule": rule, "total": _log_int(rng, 1 << 16, 1 << 25), "tensors": rng.randint(1, 130)}


# ------------------------------------------------------------------------------------------------ device memory

class _Raw:
    """A device buffer as torch takes it over without a copy."""

    def __init__(self, ptr, shape):
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f4", "data": (ptr, False), "version": 2}


def _view(ptr, shape):
    return torch.as_tensor(_Raw(ptr, shape), device="cuda")


def _ref(t):
    """A torch tensor as an operand of the entry points; it stays the tensor's memory."""
    return ops.Tensor(tuple(t.shape), np.int32 if t.dtype == torch.int32 else F32, _ptr=t.data_ptr(), _owner=t)


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(g, *shape, scale=1.0):
    return torch.randn(shape, generator=g, device="cuda") * scale


class _DeviceInit(nnet.Init):
    """He-scaled filters as nnet.Init draws them, made on the device."""

    def __init__(self, seed):
        super().__init__(0)
        self.gen, self.made = _gen(seed), []

    def he_gaussian(self, op):
        fan_in = int(np.prod(op.shape[1:]))
        self.made.append((op, _randn(self.gen, *op.shape, scale=math.sqrt(2.0 / fan_in))))

    def store(self):
        torch.cuda.synchronize()
        for op, t in self.made:
            ptr, nbytes = op.device_ptr()
            capi.check(capi.load().dopt_hip_copy_d2d(ptr, t.data_ptr(), nbytes))
        ops.sync()
        self.made = []


# ------------------------------------------------------------------------------------------------ networks

def _vgg_sizes(width):
    return [s if s < 0 else s * width // 64 for s in nnet.VGG16_SIZES]


def _classes(case):
    return 10


def _features(case):
    return [case["batch"], 784] if case["net"] in ("logit", "mlp") else [case["batch"], 3, 32, 32]


def _network(case, feats, init):
    net, n = case["net"], _classes(case)
    if net == "mlp":
        body = nnet.relu(nnet.dense(nnet.dataSource(feats), case["width"], init))
        body = nnet.relu(nnet.dense(body, case["width"], init))
    elif net == "vgg":
        d = 8 * case["width"]
        body = nnet.vgg(feats, _vgg_sizes(case["width"]), [d, d], init)
    else:
        body = nnet.wideResNet(feats, case["depth"], case["width"], init)
    return nnet.softmax(nnet.dense(body, n, init))


def _batch(case, g):
    shape = _features(case)
    x = torch.rand(shape, generator=g, device="cuda") if len(shape) == 2 else _randn(g, *shape)
    y = torch.zeros((case["batch"], _classes(case)), device="cuda")
    lab = torch.randint(0, _classes(case), (case["batch"], 1), generator=g, device="cuda")
    return x, y.scatter_(1, lab, 1.0)


def _prepare_train(case, seed):
    g = _gen(seed)
    shape = _features(case)
    feats, labels = core.float32(shape), core.float32([case["batch"], _classes(case)])
    x, y = _batch(case, g)
    state = {"case": case, "keep": [x, y]}
    if case["net"] == "logit":
        W, b = core.float32([784, 10]), core.float32([10])
        linear = core.matmul(feats, W) + core.repeat(b, case["batch"])
        numer = core.exp(linear - core.maxElement(linear))
        denom = core.repeat(core.sum(numer, [1]).reshape([case["batch"], 1]), [1, 10])
        preds = numer / denom
        loss = nnet.crossEntropy(preds, labels)
        wrt, proj, init = [W, b], None, None
        shown = [W, b]
    else:
        init = _DeviceInit(seed + 1000003)
        last = _network(case, feats, init)
        net = nnet.DAGNetwork([feats], [last])
        preds = last.trainOutput
        loss = nnet.crossEntropy(preds, labels) + net.paramLoss
        wrt, proj = net.params, net.paramProj
        shown = None
    # A rate so small that a second step on the same batch stays comparable between two correct summation orders: a relu
    # or max-pool decision within rounding of a tie moves a gradient by far more than rounding itself does, and a larger
    # rate carries that into every value of the next step.
    rate = 1e-6
    name = "learningRate" if case["rule"] == "sgd" else "alpha"
    make = getattr(online, ("fused_" if case["fused"] else "") + case["rule"])
    up = make([loss, preds], wrt, proj, flags=configs.REWRITES,
              **{name: rate if case["fused"] else core.float32([], [rate])})
    if init is not None:
        init.store()
    state["up"] = up
    # What a step returns: loss, predictions, and of the parameters the running statistics and the first optimizer
    # state - the gradient times a constant on the first step - of weights, scales and shifts.  The gradient of a bias
    # that batch norm follows is zero but for rounding, so those are left out, and beyond sixty tensors the smallest.
    outs = {"loss": _view(up._out_bufs[0].ptr, (1,)), "preds": _view(up._out_bufs[1].ptr, preds.shape)}
    if case["fused"]:
        first = {id(w): m.ptr for w, m in zip(wrt, up.state["m"])}
    else:
        held = up.momentum if case["rule"] == "sgd" else up.means
        first = {id(w): m.device_ptr()[0] for w, m in zip(wrt, held)}
    proj = proj or {}
    bn_bias = set()
    for i in range(1, len(wrt) - 1):
        if wrt[i].rank == 1 and wrt[i - 1].rank == 4 and wrt[i + 1].rank == 4 and wrt[i + 1].shape[0] == 1:
            bn_bias.add(id(wrt[i]))
    rows = []
    for i, w in enumerate(wrt):
        if id(w) in bn_bias:
            continue
        ptr = w.device_ptr()[0] if (w in proj or shown is not None) else first[id(w)]
        rows.append((0 if w.rank > 1 else 1, -w.volume, i, ptr, w.shape))
    for rank, _, i, ptr, shp in sorted(rows)[:60]:
        outs["p%03d" % i] = _view(ptr, shp)
    state["outs"] = outs
    if case.get("feed") == "host":
        hx = np.concatenate([x.cpu().numpy()] + [_batch(case, g)[0].cpu().numpy() for _ in range(3)])
        hy = np.tile(y.cpu().numpy(), (4, 1))
        it = data.SupervisedBatchIterator(hx, hy, [shape[1:], [_classes(case)]], shuffle=True, seed=seed)
        state["feed"] = data.DeviceFeed(it, case["batch"], 4, 4, True, False, seed=seed)
        state["vars"] = (feats, labels)
    else:
        state["args"] = {feats: _ref(x), labels: _ref(y)}
    return state


def _run_train(state):
    args = state.get("args")
    if args is None:
        feed = state["feed"]
        if feed.finished():
            feed.restart()
        f, l = feed.next()
        args = {state["vars"][0]: f, state["vars"][1]: l}
    state["up"].step_async(args)
    return state["outs"]


def _prepare_predict(case, seed):
    g = _gen(seed)
    feats = core.float32(_features(case))
    init = _DeviceInit(seed + 1000003)
    last = _network(case, feats, init)
    x, _ = _batch(case, g)
    net = nnet.DAGNetwork([feats], [last])
    # running statistics as a trained network has them
    for p in net.params:
        if p in net.paramProj:
            base = 1.0 if p.value[0] == 1.0 else 0.0
            init.made.append((p, base + 0.1 * torch.rand(p.shape, generator=g, device="cuda")))
    plan = core.compile([last.output], configs.REWRITES)
    init.store()
    out = torch.empty(last.output.shape, device="cuda")
    return {"case": case, "plan": plan, "args": {feats: _ref(x)}, "rets": [_ref(out)], "out": out, "keep": x}


def _run_predict(state):
    state["plan"].execute(state["args"], state["rets"])
    return state["out"]


# ------------------------------------------------------------------------------------------------ single operations

def _prepare_conv(case, seed):
    g, c = _gen(seed), case
    x = torch.relu(_randn(g, c["n"], c["c"], c["h"], c["w"]))
    w = _randn(g, c["k"], c["c"], c["r"], c["r"], scale=math.sqrt(2.0 / (c["c"] * c["r"] * c["r"])))
    p = [(s + 2 * c["pad"] - c["r"]) // c["stride"] + 1 for s in (c["h"], c["w"])]
    dy = _randn(g, c["n"], c["k"], p[0], p[1], scale=0.01)
    outs = [torch.empty_like(dy), torch.empty_like(x), torch.empty_like(w)]
    return {"case": case, "in": [x, w, dy], "t": [_ref(t) for t in (x, w, dy)], "outs": outs, "o": [_ref(t) for t in outs]}


def _run_conv(state):
    c, (x, w, dy), (y, dx, dw) = state["case"], state["t"], state["o"]
    pad, stride = (c["pad"],) * 2, (c["stride"],) * 2
    ops.convolution(x, w, pad, stride, out=y)
    ops.conv_bwd_data(dy, w, x.shape, pad, stride, out=dx)
    ops.conv_bwd_filter(dy, x, w.shape, pad, stride, out=dw)
    return state["outs"]


def _prepare_matmul(case, seed):
    g, c = _gen(seed), case
    a, b = _randn(g, c["m"], c["k"]), _randn(g, c["k"], c["n"], scale=math.sqrt(2.0 / c["k"]))
    dy = _randn(g, c["m"], c["n"], scale=0.01)
    outs = [torch.empty_like(dy), torch.empty_like(a), torch.empty_like(b)]
    return {"case": case, "in": [a, b, dy], "t": [_ref(t) for t in (a, b, dy)], "outs": outs, "o": [_ref(t) for t in outs]}


def _run_matmul(state):
    (a, b, dy), (y, da, db) = state["t"], state["o"]
    ops.matmul(a, b, out=y)
    ops.matmul_t(dy, b, trans_b=True, out=da)
    ops.matmul_t(a, dy, trans_a=True, out=db)
    return state["outs"]


def _prepare_block(case, seed):
    g, c = _gen(seed), case
    act, half, ch = (c["n"], c["c"], c["h"], c["w"]), (c["n"], c["c"], c["h"] // 2, c["w"] // 2), (c["c"],)
    ins = {"x": _randn(g, *act), "b": _randn(g, *ch), "gamma": 1.0 + 0.1 * _randn(g, *ch), "beta": 0.1 * _randn(g, *ch),
           "mean": torch.zeros(ch, device="cuda"), "var": torch.ones(ch, device="cuda"), "dp": _randn(g, *half, scale=0.01)}
    n = int(np.prod(act))
    shapes = {"y0": act, "bn": (n + 2 * c["c"],), "relu": act, "pool": half, "dpool": act, "drelu": act,
              "dbn": (n + 2 * c["c"],), "db": ch, "infer": act}
    outs = {k: torch.empty(s, device="cuda") for k, s in shapes.items()}
    return {"case": case, "in": ins, "t": {k: _ref(t) for k, t in ins.items()}, "outs": outs,
            "o": {k: _ref(t) for k, t in outs.items()}, "act": act}


def _run_block(state):
    t, o, act = state["t"], state["o"], state["act"]
    ops.add_bias(t["x"], t["b"], out=o["y0"])
    ops.bn_train(o["y0"], t["gamma"], t["beta"], t["mean"], t["var"], 0.9, out=o["bn"])
    y = o["bn"].view(0, act)
    ops.relu(y, out=o["relu"])
    ops.maxpool(o["relu"], (2, 2), out=o["pool"])
    # decisions taken from the input itself, so that rounding in batch norm cannot move them
    ops.maxpool_grad(t["dp"], t["x"], (2, 2), out=o["dpool"])
    ops.relu_grad(o["dpool"], t["x"], out=o["drelu"])
    ops.bn_grad(o["drelu"], o["y0"], t["gamma"], out=o["dbn"])
    ops.add_bias_grad(o["drelu"], out=o["db"])
    ops.bn_infer(o["y0"], t["gamma"], t["beta"], t["mean"], t["var"], out=o["infer"])
    return state["outs"]


def _prepare_tensor(case, seed):
    g, r, c = _gen(seed), case["rows"], case["cols"]
    ins = {"x": _randn(g, r, c), "u": torch.rand((r, c), generator=g, device="cuda") + 0.5,
           "i": torch.randint(-9, 9, (r, c), generator=g, device="cuda", dtype=torch.int32)}
    f, i32 = torch.float32, torch.int32
    shapes = {"exp": ((r, c), f), "pow": ((r, c), f), "sum": ((r,), f), "total": ((1,), f), "cols": ((c,), f), "max": ((r,), f),
              "soft": ((r, c), f), "argmin": ((r, 1), i32), "t": ((c, r), f), "slice": ((r - 2, c - 3), f),
              "pad": ((r + 1, c + 2), f), "twice": ((r, 2 * c), f), "isum": ((c,), i32), "imul": ((r, c), i32)}
    outs = {k: torch.empty(s, device="cuda", dtype=d) for k, (s, d) in shapes.items()}
    return {"case": case, "in": ins, "t": {k: _ref(v) for k, v in ins.items()}, "outs": outs,
            "o": {k: _ref(v) for k, v in outs.items()}}


def _run_tensor(state):
    t, o, (r, c) = state["t"], state["o"], state["t"]["x"].shape
    ops.pointwise("exp", t["x"], out=o["exp"])
    ops.pointwise("pow", t["u"], t["x"], out=o["pow"])
    ops.sum(o["exp"], [1], out=o["sum"])
    ops.sum(o["exp"], out=o["total"])
    ops.sum(t["u"], [0], out=o["cols"])
    ops.max_element(t["x"], [1], out=o["max"])
    ops.softmax(t["x"], out=o["soft"])
    ops.argmin(t["x"], 1, out=o["argmin"])
    ops.transpose(t["x"], out=o["t"])
    ops.slice(t["x"], [1, 2], [r - 1, c - 1], out=o["slice"])
    ops.pad(t["x"], [1, 0], [0, 2], out=o["pad"])
    ops.repeat(t["x"], [1, 2], out=o["twice"])
    ops.pointwise("mul", t["i"], t["i"], out=o["imul"])
    ops.sum(t["i"], [0], out=o["isum"])
    return state["outs"]


def _update_sizes(case):
    """`tensors` sizes spread over a factor of 586 as workloads.adam16m_sizes spreads them, `total` values in all."""
    n = min(case["tensors"], case["total"] // 16)
    raw = 586.0 ** (np.arange(n) / max(1, n - 1))
    sizes = [max(1, int(v)) for v in raw * case["total"] / raw.sum()]
    sizes[-1] += max(0, case["total"] - sum(sizes))
    return sizes


def _prepare_update(case, seed):
    g, sizes = _gen(seed), _update_sizes(case)
    if case["total"] == workloads.ADAM16M_TOTAL and case["tensors"] == 40:
        sizes = workloads.adam16m_sizes()
    names = {"sgd": "wgm", "adam": "wgmv", "amsgrad": "wgmvh"}[case["rule"]]
    scale = {"w": 1.0, "g": 0.1, "m": 0.1, "v": 0.01, "h": 0.01}
    flat = {k: _randn(g, sum(sizes), scale=scale[k]) for k in names}
    for k in "vh":
        if k in flat:
            flat[k] = flat[k].abs()
    # every tensor an allocation of its own, as a network's parameters are
    parts = {k: [p.clone() for p in torch.split(v, sizes)] for k, v in flat.items()}
    opt = ops.FusedOptimizer(*[[_ref(p) for p in parts[k]] for k in names])
    shown = [p for k in names if k != "g" for p in parts[k]]
    shown = sorted(shown, key=lambda p: -p.numel())[:60]
    return {"case": case, "opt": opt, "parts": parts, "outs": shown}


def _run_update(state):
    opt, rule = state["opt"], state["case"]["rule"]
    if rule == "sgd":
        opt.sgd(0.01, 0.9, False)
    else:
        getattr(opt, rule)(1e-3, 0.9, 0.999, 1e-8)
    return state["outs"]


_PREPARE = {"train": _prepare_train, "predict": _prepare_predict, "conv": _prepare_conv, "matmul": _prepare_matmul,
            "block": _prepare_block, "tensor": _prepare_tensor, "update": _prepare_update}
_RUN = {"train": _run_train, "predict": _run_predict, "conv": _run_conv, "matmul": _run_matmul, "block": _run_block,
        "tensor": _run_tensor, "update": _run_update}


def prepare(case, seed):
    capi.check(capi.load().dopt_hip_init(0))
    state = _PREPARE[case["kind"]](case, seed)
    torch.cuda.synchronize()
    return state


def run(state):
    return _RUN[state["case"]["kind"]](state)


# ------------------------------------------------------------------------------------------------ work and tolerance

def _layers(case):
    """(forward FLOPs, FLOPs of the gradient with respect to the layer's input, filter size) per contraction."""
    b, net, out = case["batch"], case["net"], []

    def conv(cin, cout, side, r, needs_dx=True):
        f = 2.0 * b * cin * cout * r * r * side * side
        out.append((f, f if needs_dx else 0.0, cin * cout * r * r))

    if net == "logit":
        dims, first = [784, 10], True
    elif net == "mlp":
        dims, first = [784, case["width"], case["width"], 10], True
    elif net == "vgg":
        c, side = 3, 32
        for s in _vgg_sizes(case["width"]):
            if s < 0:
                side //= 2
            else:
                conv(c, s, side, 3, bool(out))
                c = s
        d = 8 * case["width"]
        dims, first = [c * side * side, d, d, 10], False
    else:
        conv(3, 16, 32, 3, False)
        c, side = 16, 32
        for mult, s in ((1, 1), (2, 2), (4, 2)):
            u = 16 * mult * case["width"]
            for i in range((case["depth"] - 4) // 6):
                side //= s if i == 0 else 1
                conv(c, u, side, 3)
                conv(u, u, side, 3)
                if c != u:
                    conv(c, u, side, 1)
                c = u
        dims, first = [c, 10], False
    for i in range(len(dims) - 1):
        f = 2.0 * b * dims[i] * dims[i + 1]
        out.append((f, 0.0 if first and i == 0 else f, dims[i] * dims[i + 1]))
    return out


def work(case):
    k = case["kind"]
    if k in ("train", "predict"):
        rows = _layers(case)
        params = sum(r[2] for r in rows)
        io = int(np.prod(_features(case))) + case["batch"] * 10
        if k == "predict":
            return {"bytes": 4.0 * (params + io), "flops": sum(r[0] for r in rows)}
        # weights and optimizer state read and written once
        per = {"sgd": 4, "adam": 6, "amsgrad": 8}[case["rule"]]
        return {"bytes": 4.0 * (params * per + io), "flops": sum(2 * r[0] + r[1] for r in rows)}
    if k == "conv":
        p = [(s + 2 * case["pad"] - case["r"]) // case["stride"] + 1 for s in (case["h"], case["w"])]
        if min(p) < 1:
            return {"bytes": float("inf"), "flops": float("inf")}
        x, y = case["n"] * case["c"] * case["h"] * case["w"], case["n"] * case["k"] * p[0] * p[1]
        w = case["k"] * case["c"] * case["r"] * case["r"]
        return {"bytes": 8.0 * (x + y + w), "flops": 6.0 * y * case["c"] * case["r"] * case["r"]}
    if k == "matmul":
        m, n, kk = case["m"], case["n"], case["k"]
        return {"bytes": 8.0 * (m * n + m * kk + kk * n), "flops": 6.0 * m * n * kk}
    if k == "block":
        n = case["n"] * case["c"] * case["h"] * case["w"]
        # nine operations, each reading its operands and writing its result once
        return {"bytes": 4.0 * n * (2 + 2 + 2 + 1.25 + 2.25 + 3 + 3 + 1 + 2), "flops": 40.0 * n}
    if k == "tensor":
        n = case["rows"] * case["cols"]
        return {"bytes": 4.0 * n * (2 + 3 + 1 + 1 + 1 + 1 + 2 + 1 + 2 + 2 + 2 + 3 + 2 + 1), "flops": 20.0 * n}
    return {"bytes": float(case["total"]) * {"sgd": 20, "adam": 28, "amsgrad": 36}[case["rule"]], "flops": 10.0 * case["total"]}


def tolerance(case):
    """Four times what two correct fp32 evaluations were seen to differ by (other summation orders, filters moved by a
    rounding): sums of products reach 1e-6 and outputs behind a whole network 2e-6.  A training step shows more than its
    rounding: of its relu and max-pool decisions those within rounding of a tie differ, a share of about 1e-6, and each
    moves single gradient values by as much as they are large (5e-3 in the norm, up to 0.4 of the root mean square)."""
    if case["kind"] == "train":
        return {"rel": 0.02, "max": 0.99} if case["net"] in ("vgg", "wrn") else {"rel": 2e-3, "max": 0.1}
    if case["kind"] == "update":
        return {"rel": 1e-6}
    return {"rel": 1e-5, "max": 4e-4}
