"""dopt_hip_tiny_graph: runs of operations on tiny tensors as one launch.  Every node kind against the stand-alone
entry point it stands for, bit for bit (the contract that lets a plan run such a run as one step and still return
what the plan without rewrites returns), and a whole loss tail against the oracle."""
import ctypes as C

import numpy as np
import pytest

import oracle as O
from dopt_amd import capi, ops
from util import assert_close

pytestmark = pytest.mark.gpu

PW, RED, SMAX, SMAXG, REP, MATVEC = range(6)


def _node(kind, dst, a, b=-1, op=0, n=0, a_kind=0, b_kind=0, dims=(0, 0, 0, 0), reps=(0, 0, 0, 0), offs=(0, 0, 0)):
    nd = capi.TinyNode()
    nd.kind, nd.op, nd.dst, nd.a, nd.b, nd.a_kind, nd.b_kind, nd.n = kind, op, dst, a, b, a_kind, b_kind, n
    nd.dst_offset, nd.a_offset, nd.b_offset = offs
    nd.dims = (C.c_int * 4)(*dims)
    nd.reps = (C.c_int * 4)(*reps)
    return nd


def _run(slots, nodes):
    lib = capi.load()
    n = len(nodes)
    capi.check(lib.dopt_hip_tiny_graph(len(slots), (C.c_void_p * len(slots))(*[t.ptr for t in slots]), n,
                                       (capi.TinyNode * n)(*nodes)))


def test_every_pointwise_operation_as_a_node_equals_its_kernel():
    lib = capi.load()
    r = np.random.default_rng(1)
    names = ["add", "sub", "mul", "div", "lt", "lte", "gt", "gte", "eq", "neq", "max", "min", "pow", "atan2", "neg", "abs",
             "sgn", "exp", "log", "sqrt", "sin", "cos", "tan", "asin", "acos", "atan", "sinh", "cosh", "tanh", "asinh", "acosh",
             "atanh"]
    n = 1000
    a = (r.standard_normal(n) * 2).astype(np.float32)
    b = (r.standard_normal(n) * 2).astype(np.float32)
    a[::50] = b[::50]                                  # equal operands for the comparisons
    a[7], a[8], b[9] = np.nan, np.inf, -np.inf
    ta, tb = ops.tensor(a), ops.tensor(b)
    outs = [ops.Tensor([n]) for _ in names]
    nodes = []
    for k, name in enumerate(names):
        idx = lib.dopt_hip_pointwise_index(name.encode())
        assert idx >= 0
        binary = lib.dopt_hip_pointwise_arity(name.encode()) == 2
        nodes.append(_node(PW, 2 + k, 0, 1 if binary else -1, op=idx, n=n))
    _run([ta, tb] + outs, nodes)
    for name, out in zip(names, outs):
        binary = lib.dopt_hip_pointwise_arity(name.encode()) == 2
        want = ops.pointwise(name, ta, tb if binary else None).numpy()
        assert np.array_equal(out.numpy(), want, equal_nan=True), name
    # relu / reluGrad as nodes against their kernels, a one-element operand, and a column times a row
    relu, rgrad, scal, outer = ops.Tensor([n]), ops.Tensor([n]), ops.Tensor([n]), ops.Tensor([40 * 25])
    one = ops.tensor(np.array([1.25], np.float32))
    _run([ta, tb, relu, rgrad, scal, one, outer],
         [_node(PW, 2, 0, op=lib.dopt_hip_pointwise_index(b"relu"), n=n),
          _node(PW, 3, 0, 1, op=lib.dopt_hip_pointwise_index(b"reluGrad"), n=n),
          _node(PW, 4, 0, 5, op=lib.dopt_hip_pointwise_index(b"mul"), n=n, b_kind=1),
          _node(PW, 6, 0, 1, op=lib.dopt_hip_pointwise_index(b"mul"), n=1000, a_kind=2, b_kind=3, dims=(25, 0, 0, 0))])
    assert np.array_equal(relu.numpy(), ops.relu(ta).numpy(), equal_nan=True)
    assert np.array_equal(rgrad.numpy(), ops.relu_grad(ta, tb).numpy(), equal_nan=True)
    assert np.array_equal(scal.numpy(), a * np.float32(1.25), equal_nan=True)
    want = ops.matmul(ops.tensor(a[:40].reshape(40, 1)), ops.tensor(b[:25].reshape(1, 25))).numpy()
    assert np.array_equal(outer.numpy().reshape(40, 25), want, equal_nan=True)


@pytest.mark.parametrize("shape,axes", [((128, 10), [0, 1]),      # the loss: one contiguous row of 1280 values (quads)
                                        ((1283,), [0]),           # ... of a length that is no multiple of four
                                        ((3, 700), [1]),          # three such rows
                                        ((4095,), [0]),
                                        ((100, 10), [1]),         # short rows: one thread per row
                                        ((12, 30, 7), [1]),       # a strided reduction
                                        ((12, 30, 7), [0, 1]),
                                        ((5, 6, 7, 2), [1, 2]),
                                        ((64,), [0]), ((65,), [0]), ((1,), [0])])
@pytest.mark.parametrize("op", ["sum", "maxElement"])
def test_reductions_as_nodes_equal_dopt_hip_reduce(shape, axes, op):
    r = np.random.default_rng(2)
    x = r.standard_normal(shape).astype(np.float32)
    if op == "maxElement" and x.size > 3:
        x.reshape(-1)[[0, 3]] = np.nan
    tx = ops.tensor(x)
    want = (ops.sum(tx, axes) if op == "sum" else ops.max_element(tx, axes)).numpy()
    outer = int(np.prod(shape[:axes[0]], dtype=np.int64))
    R = int(np.prod([shape[a] for a in axes]))
    inner = int(np.prod(shape[axes[-1] + 1:], dtype=np.int64))
    out = ops.Tensor([max(outer * inner, 1)])
    _run([tx, out], [_node(RED, 1, 0, op=0 if op == "sum" else 1, n=outer * inner, dims=(outer, R, inner, 0))])
    assert np.array_equal(out.numpy().ravel(), want.ravel(), equal_nan=True)


@pytest.mark.parametrize("shape", [(5, 1), (300, 2), (100, 3), (70, 4), (64, 5), (9, 1, 7), (33, 15), (3, 16), (200, 17), (9, 31), (4, 32), (11, 33), (3, 16, 5), (2, 17, 3, 2)])
def test_softmax_of_few_classes(shape):
    """Kept in registers up to 16 and 32 classes: the bits of the node, which takes the classes in the reference's order."""
    r = np.random.default_rng(int(np.prod(shape)))
    x = (r.standard_normal(shape) * 5).astype(np.float32)
    x.ravel()[0] = np.inf
    x.ravel()[-1] = np.nan
    inner = int(np.prod(shape[2:], dtype=np.int64))
    tx, got = ops.tensor(x), ops.Tensor(shape)
    _run([tx, got], [_node(SMAX, 1, 0, n=x.size, dims=(shape[0], shape[1], inner, 0))])
    assert np.array_equal(ops.softmax(tx).numpy(), got.numpy(), equal_nan=True)


@pytest.mark.parametrize("shape", [(128, 10), (100, 10), (7, 63), (4, 5, 3, 3), (2, 70, 2, 2)])
def test_softmax_nodes_equal_their_kernels(shape):
    r = np.random.default_rng(3)
    x = (r.standard_normal(shape) * 3).astype(np.float32)
    dy = r.standard_normal(shape).astype(np.float32)
    tx, tdy = ops.tensor(x), ops.tensor(dy)
    y = ops.softmax(tx)
    dx = ops.softmax_grad(tdy, y)
    N, Cc = shape[0], shape[1]
    inner = int(np.prod(shape[2:], dtype=np.int64))
    gy, gdx = ops.Tensor(shape), ops.Tensor(shape)
    _run([tx, tdy, gy, gdx], [_node(SMAX, 2, 0, n=x.size, dims=(N, Cc, inner, 0)),
                              _node(SMAXG, 3, 1, 2, n=x.size, dims=(N, Cc, inner, 0))])
    assert np.array_equal(gy.numpy(), y.numpy()) and np.array_equal(gdx.numpy(), dx.numpy())
    assert_close(gy.numpy(), O.softmax(x), "softmax node")


@pytest.mark.parametrize("shape,reps", [((1,), (1000,)), ((3, 4), (2, 5)), ((2, 3, 4, 5), (2, 1, 3, 2)), ((7, 1), (1, 10))])
def test_repeat_node_equals_dopt_hip_repeat(shape, reps):
    r = np.random.default_rng(4)
    x = r.standard_normal(shape).astype(np.float32)
    tx = ops.tensor(x)
    want = ops.repeat(tx, list(reps)).numpy()
    out = ops.Tensor(want.shape)
    lead = 4 - len(shape)
    _run([tx, out], [_node(REP, 1, 0, n=want.size, dims=(1,) * lead + tuple(shape), reps=(1,) * lead + tuple(reps))])
    assert np.array_equal(out.numpy(), want)
    assert np.array_equal(want, np.tile(x, reps))


@pytest.mark.parametrize("rows,k", [(100, 10), (1, 2), (256, 16), (240, 17), (63, 65), (1, 4096), (31, 130), (2048, 2), (1024, 3)])
def test_matrix_vector_node_equals_the_product(rows, k):
    r = np.random.default_rng(rows + k)
    a, b = r.standard_normal((rows, k)).astype(np.float32), r.standard_normal((k, 1)).astype(np.float32)
    a[0] = -0.0
    ta, tb, out = ops.tensor(a), ops.tensor(b), ops.Tensor([rows, 1])
    _run([ta, tb, out], [_node(MATVEC, 2, 0, 1, n=rows, dims=(k, 0, 0, 0))])
    want = ops.matmul(ta, tb).numpy()
    assert np.array_equal(out.numpy().view(np.uint32), want.view(np.uint32))


def test_a_loss_tail_as_one_launch_matches_the_oracle():
    """softmax -> + eps -> log -> * labels -> sum -> * (-1/n), and back: d loss / d logits, as one launch with byte
    offsets into a shared buffer, against the oracle composed operation by operation."""
    lib = capi.load()
    r = np.random.default_rng(5)
    n, c = 128, 10
    logits = (r.standard_normal((n, c)) * 2).astype(np.float32)
    labels = np.eye(c, dtype=np.float32)[r.integers(0, c, n)]
    eps, scale = np.array([1e-6], np.float32), np.array([-1.0 / n], np.float32)
    idx = lambda name: lib.dopt_hip_pointwise_index(name.encode())
    work = ops.Tensor([6 * n * c])                     # y | y + eps | log | labels * log | d/dy | d/dlogits
    loss, total = ops.Tensor([1]), ops.Tensor([1])
    tl, tlab, teps, tsc = ops.tensor(logits), ops.tensor(labels), ops.tensor(eps), ops.tensor(scale)
    B = 4 * n * c
    slots = [tl, tlab, teps, tsc, work, total, loss]
    nodes = [_node(SMAX, 4, 0, n=n * c, dims=(n, c, 1, 0)),
             _node(PW, 4, 4, 2, op=idx("add"), n=n * c, b_kind=1, offs=(B, 0, 0)),
             _node(PW, 4, 4, op=idx("log"), n=n * c, offs=(2 * B, B, 0)),
             _node(PW, 4, 1, 4, op=idx("mul"), n=n * c, offs=(3 * B, 0, 2 * B)),
             _node(RED, 5, 4, op=0, n=1, dims=(1, n * c, 1, 0), offs=(0, 3 * B, 0)),
             _node(PW, 6, 5, 3, op=idx("mul"), n=1),
             # backward: d loss / d y = scale * labels / (y + eps), then through the softmax
             _node(PW, 4, 1, 4, op=idx("div"), n=n * c, offs=(4 * B, 0, B)),
             _node(PW, 4, 4, 3, op=idx("mul"), n=n * c, b_kind=1, offs=(4 * B, 4 * B, 0)),
             _node(SMAXG, 4, 4, 4, n=n * c, dims=(n, c, 1, 0), offs=(5 * B, 4 * B, 0))]
    _run(slots, nodes)
    y = O.softmax(logits)
    want_loss = O.sum(labels * np.log(y + eps[0]), [0, 1]) * scale[0]
    got = work.numpy().reshape(6, n, c)
    assert_close(got[0], y, "softmax")
    assert_close(loss.numpy(), np.asarray(want_loss).reshape(1), "loss")
    dy = (scale[0] * labels / (y + eps[0])).astype(np.float32)
    assert_close(got[5], O.softmax_grad(dy, y), "d loss / d logits")
    # limits are refused, not truncated
    bad = _node(PW, 1, 0, op=idx("neg"), n=5000)
    assert lib.dopt_hip_tiny_graph(2, (C.c_void_p * 2)(tl.ptr, work.ptr), 1, (capi.TinyNode * 1)(bad)) != 0
    assert b"at most" in lib.dopt_hip_last_error()
    ops.sync()


UNARY, BINARY = ["neg", "abs", "sgn", "exp", "sqrt", "tanh", "relu"], ["add", "sub", "mul", "div", "max", "min", "lt", "pow"]


def _random_run(seed, wide=False):
    """A graph of tiny operations of every kind a run may hold, over tensors of odd and even sizes, and its variables; `wide`: rows
    of 33 values and more, where a softmax is kept in memory and a fold of several rows is the work of a workgroup."""
    from dopt_amd import core, nnet
    r = np.random.default_rng(seed)
    rows, cols = int(r.choice([1, 2, 7, 33, 64, 100, 257, 400])), int(r.choice([1, 2, 3, 8, 10, 16, 40]))
    if wide:
        rows, cols = int(r.choice([1, 2, 3, 4, 5, 11, 40, 64])), int(r.choice([33, 48, 63, 64, 65, 68, 100, 129, 256, 1000, 1025]))
    if rows * cols > 4096:
        cols = 4096 // rows
    var = [core.float32([rows, cols]) for _ in range(3)] + [core.float32([1]), core.float32([rows, 1]), core.float32([1, cols])]
    full, single = list(var[:3]), [var[3]]
    outs = []
    for _ in range(int(r.integers(6, 22))):
        k, x = r.integers(0, 13 if wide else 11), full[r.integers(len(full))]
        y = full[r.integers(len(full))]
        if k < 3:
            op = BINARY[r.integers(len(BINARY))]
            full.append(core.Operation(op, [x, y], {}) if not hasattr(core, op) else getattr(core, op)(x, y))
        elif k == 3:
            op = UNARY[r.integers(len(UNARY) - 1)]
            full.append(core.Operation(op, [x], {}) if not hasattr(core, op) else getattr(core, op)(x))
        elif k == 4:
            full.append(core.softmax(x) if cols < 64 else x)
        elif k == 5:
            single.append(core.sum(x).reshape([1]) if r.random() < 0.5 else core.maxElement(x).reshape([1]))
        elif k == 6:
            full.append(core.repeat(core.sum(x, [0]).reshape([1, cols]), [rows, 1]))
        elif k == 7:
            full.append(core.repeat(core.maxElement(x, [1]).reshape([rows, 1]), [1, cols]))
        elif k == 8:
            full.append(core.matmul(core.matmul(x, core.float32([cols, 1], np.ones(cols, np.float32))), var[5]))
        elif k == 9:
            full.append(core.repeat(single[r.integers(len(single))], [rows * cols]).reshape([rows, cols]) * x)
        elif k == 10:
            single.append(single[r.integers(len(single))] * single[r.integers(len(single))] + var[3])
        elif k == 11:
            full.append(core.Operation("softmaxGrad", [x, y], {}) if cols < 64 else x * y)
        else:
            full.append(core.repeat((core.sum(x, [1]) if r.random() < 0.5 else core.maxElement(x, [1])).reshape([rows, 1]), [1, cols]) - y)
        if r.random() < 0.3:
            outs.append(full[-1])
    outs += [full[-1], single[-1], core.sum(full[-1] * full[0], [1])]
    return var, outs


@pytest.mark.parametrize("seed", range(40))
def test_runs_compiled_for_a_plan_equal_their_operations(seed):
    """The kernel that a plan compiles for a run against the plan that runs every operation by itself, bit for bit (NaNs by
    their place), with values that are not finite in every other case."""
    from dopt_amd import core
    var, outs = _random_run(seed)
    r = np.random.default_rng(1000 + seed)
    plain, fused = core.compile(outs, 0), core.compile(outs, core.PLAN_VIEWS | core.PLAN_FUSE)
    for case in range(2):
        args = {v: r.standard_normal(v.shape).astype(np.float32) for v in var}
        if case == 1 and seed % 2:
            a = args[var[0]].ravel()
            a[:: max(1, a.size // 3)] = np.nan
            a[a.size // 2] = np.inf
        for x, y in zip(plain.execute(args), fused.execute(args)):
            assert np.array_equal(x, y, equal_nan=True)


@pytest.mark.parametrize("wide", [False, True], ids=["narrow", "wide"])
@pytest.mark.parametrize("seed", range(30))
def test_runs_have_a_kernel_of_their_own(seed, wide):
    """The runs of a plan are compiled: none is left to the interpreter, and their bits are those of the plan that runs every
    operation by itself, on one and the other queue and replayed."""
    from dopt_amd import core
    var, outs = _random_run(2000 + seed, wide)
    r = np.random.default_rng(3000 + seed)
    base = core.PLAN_VIEWS | core.PLAN_FUSE
    plain = core.compile(outs, 0)
    plans = [core.compile(outs, base | f) for f in (core.PLAN_TIMING, core.PLAN_OVERLAP_LIGHT, core.PLAN_GRAPH)]
    dev = {v: ops.Tensor(v.shape) for v in var}
    for case in range(4):
        for v, t in dev.items():
            a = r.standard_normal(v.shape).astype(np.float32)
            if case == 1 and v is var[0]:
                a.ravel()[:: max(1, a.size // 3)] = np.nan
                a.ravel()[a.size // 2] = -np.inf
            t.set(a)
        want = plain.execute(dev)
        for p in plans:
            for x, y in zip(want, p.execute(dev)):
                assert np.array_equal(x, y, equal_nan=True)
    assert "tiny(interpreted)" not in plans[0].profile()
    assert any(label.startswith("tiny*") for label in plans[0].profile())


def test_a_run_with_an_argument_in_its_result_is_interpreted():
    from dopt_amd import core
    x, w = core.float32([10, 10]), core.float32([10, 10])
    a = x * w
    plan = core.compile([a, core.repeat(core.sum(a, [0]).reshape([1, 10]), [10, 1]) + a * x], core.PLAN_VIEWS | core.PLAN_FUSE | core.PLAN_TIMING)
    ones = np.ones((10, 10), np.float32)
    for given, interpreted in ((ones, 0), (ops.Tensor((10, 10), _ptr=plan.result_ptr(a)[0], _owner=plan), 1), (ones, 1)):
        plan.execute({x: given, w: ones})
        assert plan.profile().get("tiny(interpreted)", (0, 0))[1] == interpreted


def test_a_run_whose_argument_lies_in_its_own_result():
    """An argument at the address of a buffer that the run fills: what it reads is what was there before."""
    from dopt_amd import core
    x, w = core.float32([10, 10]), core.float32([10, 10])
    a = x * w
    b = core.sum(a, [0])
    c = core.repeat(b.reshape([1, 10]), [10, 1]) + a * x
    plan = core.compile([a, b, c], core.PLAN_VIEWS | core.PLAN_FUSE)
    r = np.random.default_rng(0)
    X, Wv = r.standard_normal((10, 10)).astype(np.float32), r.standard_normal((10, 10)).astype(np.float32)
    first = plan.execute({x: X, w: Wv})
    ptr, _ = plan.result_ptr(c)
    before = first[2]
    again = plan.execute({x: ops.Tensor((10, 10), _ptr=ptr, _owner=plan), w: Wv})
    A = before * Wv
    assert np.array_equal(again[0], A)
    plain = core.compile([a, b, c], 0).execute({x: before, w: Wv})
    for p, q in zip(plain, again):
        assert np.array_equal(p, q)
