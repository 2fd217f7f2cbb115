"""Pointwise chains: one generated kernel against the same nodes run one kernel at a time (which the
pointwise tests pin against the oracle), bit for bit; and plans that fuse such chains against plans
that do not."""
import ctypes as C

import numpy as np
import pytest

from dopt_amd import capi, core, nnet, online, ops

pytestmark = pytest.mark.gpu
T = ops.tensor


def _one_by_one(inputs, nodes):
    vals = list(inputs)
    n = max(t.size for t in inputs)
    full = next(t for t in inputs if t.size == n)
    for i, t in enumerate(vals):
        if t.size != n:
            vals[i] = T(np.full(full.shape, t.numpy().ravel()[0], t.dtype))
    for op, lhs, rhs in nodes:
        vals.append(ops.pointwise(op, vals[lhs], None if rhs is None else vals[rhs]))
    return vals[-1].numpy()


CHAINS = [
    # w - lr * g with lr a one-element tensor (the SGD update of online/sgd.d:58-63)
    ([(1000,), (1,), (1000,)], [("mul", 1, 2), ("sub", 0, 3)]),
    # beta2 * v + (1 - beta2) * g * g                       (online/adam.d:56)
    ([(4099,), (4099,), (1,), (1,)], [("mul", 2, 0), ("mul", 3, 1), ("mul", 5, 1), ("add", 4, 6)]),
    # w - eta * (m / (sqrt(v) + eps))                        (online/adam.d:58-60)
    ([(513,), (513,), (513,), (1,), (1,)], [("sqrt", 2, None), ("add", 5, 4), ("div", 1, 6), ("mul", 3, 7), ("sub", 0, 8)]),
    # a diamond: the same node read twice, comparisons and max in the mix
    ([(33, 65), (33, 65)], [("add", 0, 1), ("mul", 2, 2), ("exp", 0, None), ("max", 3, 4), ("gt", 5, 1), ("mul", 6, 5),
                            ("tanh", 7, None)]),
    ([(7,)], [("neg", 0, None), ("abs", 1, None)]),
    ([(1 << 20,), (1 << 20,), (1,)], [("div", 0, 2), ("log", 3, None), ("atan2", 4, 1), ("min", 5, 0)]),
]


@pytest.mark.parametrize("shapes,nodes", CHAINS)
def test_chain_equals_the_nodes_run_one_by_one(shapes, nodes):
    r = np.random.default_rng(len(nodes))
    inputs = [T((np.abs(r.standard_normal(s)) + 0.5).astype(np.float32)) for s in shapes]
    got = ops.pointwise_chain(inputs, nodes).numpy()
    want = _one_by_one(inputs, nodes)
    assert np.array_equal(got, want, equal_nan=True)


def test_chain_unaligned_operands_and_int32():
    r = np.random.default_rng(0)
    base = T(r.standard_normal(1003).astype(np.float32))
    a, b = base.view(1, [1001]), base.view(2, [1001])          # 4- and 8-byte offsets: the scalar kernel
    nodes = [("mul", 0, 1), ("add", 2, 0)]
    assert np.array_equal(ops.pointwise_chain([a, b], nodes).numpy(), _one_by_one([a, b], nodes))
    ia, ib = T(r.integers(-50, 50, 300).astype(np.int32)), T(r.integers(0, 5, 300).astype(np.int32))
    nodes = [("pow", 0, 1), ("mul", 2, 0), ("sub", 3, 1)]
    assert np.array_equal(ops.pointwise_chain([ia, ib], nodes).numpy(), _one_by_one([ia, ib], nodes))


@pytest.mark.parametrize("m,n", [(7, 12), (5, 10), (128, 512), (1, 8), (9, 1), (33, 20)])
def test_chain_row_and_column_operands_and_relu_nodes(m, n):
    """relu(x + ones[m,1] . b[1,n]) and reluGrad(dy * a[m,1] . ones[1,n], x): the outer products are read as
    a per-row and a per-column element; n % 4 != 0 takes the one-element-at-a-time kernel."""
    r = np.random.default_rng(m * 100 + n)
    x = r.standard_normal((m, n)).astype(np.float32)
    dy = r.standard_normal((m, n)).astype(np.float32)
    col = r.standard_normal((m, 1)).astype(np.float32)
    row = r.standard_normal((1, n)).astype(np.float32)
    # inputs: x (tensor), col (per row), row (per column); t0 = col*row, t1 = x + t0, t2 = relu(t1)
    got = ops.pointwise_chain([T(x), T(col), T(row)], [("mul", 1, 2), ("add", 0, 3), ("relu", 4, None)],
                              kinds=[0, 2, 3], inner=n).numpy()
    outer = ops.matmul(T(col), T(row))
    want = ops.relu(ops.pointwise("add", T(x), outer)).numpy()
    assert np.array_equal(got, want)
    got = ops.pointwise_chain([T(dy), T(x), T(col), T(row)], [("mul", 2, 3), ("mul", 0, 4), ("reluGrad", 5, 1)],
                              kinds=[0, 0, 2, 3], inner=n).numpy()
    want = ops.relu_grad(ops.pointwise("mul", T(dy), outer), T(x)).numpy()
    assert np.array_equal(got, want)


def test_chain_rejects_forward_references_and_unknown_ops():
    a = T(np.ones(8, np.float32))
    with pytest.raises(capi.HipError):
        ops.pointwise_chain([a], [("add", 0, 2), ("neg", 0, None)])
    with pytest.raises(capi.HipError):
        ops.pointwise_chain([a], [("frobnicate", 0, 0)])
    assert capi.load().dopt_hip_pointwise_arity(b"atan2") == 2
    assert capi.load().dopt_hip_pointwise_arity(b"sqrt") == 1
    assert capi.load().dopt_hip_pointwise_arity(b"matmul") == 0


def _mlp(seed):
    init = nnet.Init(seed)
    x, y = core.float32([32, 20]), core.float32([32, 5])
    top = nnet.softmax(nnet.dense(nnet.relu(nnet.dense(nnet.dataSource(x), 16, init, weight_decay=1e-3)), 5, init))
    net = nnet.DAGNetwork([x], [top])
    return x, y, net, nnet.crossEntropy(top.trainOutput, y) + net.paramLoss


@pytest.mark.parametrize("maker", [online.sgd, online.adam, online.amsgrad])
def test_op_graph_optimizers_fuse_their_update_rules_without_changing_a_bit(maker):
    r = np.random.default_rng(1)
    xs = r.standard_normal((32, 20)).astype(np.float32)
    ys = np.eye(5, dtype=np.float32)[r.integers(0, 5, 32)]
    runs, kernels = [], []
    for flags in (0, core.PLAN_VIEWS | core.PLAN_FUSE):
        x, y, net, loss = _mlp(3)
        up = maker([loss], net.params, net.paramProj, flags=flags)
        losses = [up({x: xs, y: ys})[0] for _ in range(4)]
        runs.append((losses, [p.value for p in net.params]))
        kernels.append(up.plan.stats()["kernels"])
    assert kernels[1] < kernels[0] * 0.7
    for a, b in zip(runs[0][0], runs[1][0]):
        assert a == b
    for a, b in zip(runs[0][1], runs[1][1]):
        assert np.array_equal(a, b)


def test_chain_keeps_values_that_something_else_reads():
    a = core.float32([64], np.arange(64, dtype=np.float32))
    b = core.float32([64], np.ones(64, np.float32))
    s = a + b                      # read by the chain AND returned
    t = core.exp(s * 0.5) - b
    u = core.sum(s)                # a reduction reads s too
    want = core.compile([t, s, u]).execute()
    got = core.compile([t, s, u], core.PLAN_VIEWS | core.PLAN_FUSE).execute()
    for g, w in zip(got, want):
        assert np.array_equal(g, w)


def test_scalar_arithmetic_joins_the_chain_it_is_broadcast_into():
    """`weightDecay * sum(...)` differentiated gives (one-element value) x (one-element value), broadcast over the filter
    by the product with a ones vector (core/ops/basic.d:370-381): the one-element product has no kernel of its own, the
    chain over the filter computes it; the same through a `repeat`.  Values as in the plan without rewrites."""
    r = np.random.default_rng(5)
    n = 6000                                     # above the tiny-run limit
    w = core.float32([n], r.standard_normal(n).astype(np.float32))
    g = core.float32([n], r.standard_normal(n).astype(np.float32))
    u = core.float32([1], np.float32([0.37]))
    s = core.sum(g)                              # a reduction: rank 0, not part of any chain
    t = (s * 0.5) * 1.25                         # two one-element nodes, read only through the broadcast
    out = w * t + g                              # rank 0 against rank 1: repeat(t, n) = ones[n,1] x t[1,1]
    v = core.exp(u * 0.3)                        # one-element nodes again
    out2 = core.repeat(v, [n]) * w - g           # ... broadcast by a repeat
    outs = [out, out2]
    plan = core.compile(outs, core.PLAN_VIEWS | core.PLAN_FUSE | core.PLAN_TIMING)
    got = plan.execute()
    prof = plan.profile()
    assert "mul" not in prof and "exp" not in prof, prof
    want = core.compile(outs).execute()
    for a, b in zip(got, want):
        assert np.array_equal(a, b)


def _random_graph(r, n_leaves=4, n_ops=18, size=96):
    """A random DAG over [size]-vectors and [8, size/8] matrices: pointwise nodes, scalar broadcasts,
    reshapes, contiguous slices padded back, reductions as side consumers, a few outputs in the middle."""
    shape2 = [8, size // 8]
    pool = [core.float32([size], (np.abs(r.standard_normal(size)) + 0.5).astype(np.float32)) for _ in range(n_leaves)]
    scalars = [core.float32([], [float(r.uniform(0.5, 1.5))]) for _ in range(2)]
    outputs = []
    for _ in range(n_ops):
        kind = r.integers(0, 10)
        a = pool[r.integers(0, len(pool))]
        b = pool[r.integers(0, len(pool))]
        if kind <= 3:
            node = [core.add, core.sub, core.mul, core.max][kind](a, b)
        elif kind == 4:
            node = core.abs(a) if r.integers(0, 2) else core.sqrt(core.abs(a))
        elif kind == 5:
            node = a * scalars[r.integers(0, 2)]                    # repeat(scalar) + reshape + mul
        elif kind == 6:
            node = core.reshape(core.reshape(a, shape2) * core.reshape(b, shape2), [size])
        elif kind == 7:
            half = size // 2
            lo = core.slice(a, [0], [half])                         # a view under PLAN_VIEWS
            node = core.pad(lo * lo, [0], [size - half])
        elif kind == 8:
            node = a + core.sum(b) * 0.01                           # a reduction reads b, its result is broadcast
        elif kind == 9 and r.integers(0, 2):
            # a dense layer's bias add and activation on the [8, size/8] view, and the activation's gradient
            bias = core.float32([shape2[1]], r.standard_normal(shape2[1]).astype(np.float32))
            pre = core.reshape(a, shape2) + core.repeat(bias, shape2[0])
            act = core.relu(pre)
            node = core.reshape(core.reluGrad(core.reshape(b, shape2), act) + act, [size])
        else:
            node = core.min(core.exp(a * 0.1), b)
        pool.append(node)
        if r.integers(0, 4) == 0:
            outputs.append(node)                                    # exposed in the middle of a would-be chain
    outputs.append(pool[-1])
    outputs.append(core.sum(pool[-2]))
    return outputs


@pytest.mark.parametrize("seed", range(20))
def test_random_graphs_give_the_same_values_with_every_rewrite(seed):
    outs = _random_graph(np.random.default_rng(100 + seed))
    want = core.compile(outs).execute()
    for flags in (core.PLAN_VIEWS, core.PLAN_VIEWS | core.PLAN_FUSE, core.PLAN_VIEWS | core.PLAN_FUSE | core.PLAN_GRAPH,
                  core.PLAN_OVERLAP_LIGHT, core.PLAN_VIEWS | core.PLAN_FUSE | core.PLAN_OVERLAP_LIGHT,
                  core.PLAN_VIEWS | core.PLAN_FUSE | core.PLAN_OVERLAP):
        plan = core.compile(outs, flags)
        bufs = [ops.Tensor(o.shape) for o in outs]
        for _ in range(3):                                           # direct, recorded, replayed
            plan.execute(None, bufs)
            for got, w in zip(bufs, want):
                assert np.array_equal(got.numpy(), w, equal_nan=True), flags


# sizes around a quad, a workgroup's 256 quads and its 1024 loose elements; more tensors than one launch's arguments hold
GROUPS = [[2, 3], [5, 64, 1023, 1024, 1025, 4099, 100003], list(range(2, 150, 2)), [7] * 3 + [4096, 4100]]


@pytest.mark.parametrize("sizes", GROUPS, ids=lambda s: "%d_tensors" % len(s))
@pytest.mark.parametrize("offset", [0, 1, 4])
def test_update_rules_of_many_tensors_as_one_step(sizes, offset):
    """Pointwise pieces that only feed outputs, one per tensor: one step for all that share a program.  Gradients arrive as
    views into a larger tensor (`offset` elements in: 1 is no quad), scalars as products with ones vectors, through `repeat`
    and as one-element arithmetic; a value is an output and read on, one is a view of an output.  Bits of the plan without
    rewrites, also at the second execution, which replays a recording."""
    r = np.random.default_rng(len(sizes) + offset)
    rate, decay, unit = core.float32([], [0.3]), core.float32([], [0.05]), core.float32([1], [0.7])
    outs = []
    for n in sizes:
        w, m = (core.float32([n], r.standard_normal(n).astype(np.float32)) for _ in range(2))
        packed = core.float32([n + offset + 3], r.standard_normal(n + offset + 3).astype(np.float32))
        g = core.slice(packed, [offset], [offset + n])
        nm = m * rate + (1.0 - rate) * g               # 1 - rate: arithmetic on one element, for every tensor anew
        nw = w - (decay * 2.0) * (nm / (core.sqrt(core.abs(nm)) + core.repeat(unit, [n])))
        outs += [nw, core.reshape(nm, [n, 1]), core.max(nm, g)]
    want = core.compile(outs).execute()
    for flags in (core.PLAN_VIEWS | core.PLAN_FUSE | core.PLAN_TIMING, core.PLAN_VIEWS | core.PLAN_FUSE | core.PLAN_GRAPH,
                  core.PLAN_VIEWS | core.PLAN_FUSE | core.PLAN_OVERLAP, core.PLAN_FUSE):
        plan = core.compile(outs, flags)
        bufs = [ops.Tensor(o.shape) for o in outs]
        for _ in range(3):
            plan.execute(None, bufs)
            for got, b in zip(bufs, want):
                assert np.array_equal(got.numpy(), b), flags
        if flags & core.PLAN_TIMING:
            assert any(k.startswith("pointwise*") and k.endswith("x%d" % len(sizes)) for k in plan.profile()), plan.profile()


def test_values_that_something_else_reads_stay_out_of_a_group():
    """A reduction and a narrower view end what may run last; a one-element value that leaves the plan is an operand.  (A value
    scaled by one of its own elements: below.)"""
    r = np.random.default_rng(9)
    a, b = (core.float32([300], r.standard_normal(300).astype(np.float32)) for _ in range(2))
    s = a * b
    outs = [s - a, core.sum(s + b), core.slice(s, [10], [20]) * core.slice(a, [0], [10]), core.exp(b) + a]
    one = core.sum(a * 0.5)
    outs += [(one * 0.25) * a, (one * 0.25) * b, one * 0.25]
    want = core.compile(outs).execute()
    got = core.compile(outs, core.PLAN_VIEWS | core.PLAN_FUSE).execute()
    for g, w in zip(got, want):
        assert np.array_equal(g, w)


@pytest.mark.parametrize("tensors", [1, 3])
@pytest.mark.parametrize("read_on", [True, False], ids=["an output as well", "only read by its product"])
def test_a_tensor_scaled_by_its_own_first_element(tensors, read_on):
    """A view of a value's first element starts where the value does, and a view of its first rows too: what reads one does not
    read the whole.  As a product with [1, 1] from either side, through the scalar broadcast and through `repeat`; 5000 elements
    are no run of tiny operations."""
    r = np.random.default_rng(11)
    n, outs = 5000, []
    first = lambda v: core.slice(v, [0], [1])
    forms = [lambda v: core.matmul(core.reshape(v, [n, 1]), core.reshape(first(v), [1, 1])), lambda v: v * core.reshape(first(v), []),
             lambda v: v - core.repeat(first(v), [n]), lambda v: core.matmul(core.reshape(first(v), [1, 1]), core.reshape(v, [1, n]))]
    for _ in range(tensors):
        a, b = (core.float32([n], r.standard_normal(n).astype(np.float32)) for _ in range(2))
        for k, form in enumerate(forms):
            y, z = a * b + (0.5 + k), a - b * (0.5 + k)   # values of their own for each form
            outs += ([y, z] if read_on else []) + [form(y), core.sum(form(z))]
        if not read_on:
            column, row = a * b, core.float32([1, 100], r.standard_normal(100).astype(np.float32))
            outs.append(core.matmul(core.reshape(core.slice(column, [0], [50]), [50, 1]), row) + core.reshape(column, [50, 100]))
    want = core.compile(outs).execute()
    for flags in (core.PLAN_VIEWS | core.PLAN_FUSE, core.PLAN_VIEWS | core.PLAN_FUSE | core.PLAN_GRAPH):
        plan = core.compile(outs, flags)
        bufs = [ops.Tensor(o.shape) for o in outs]
        for _ in range(3):
            plan.execute(None, bufs)
            for k, (got, w) in enumerate(zip(bufs, want)):
                assert np.array_equal(got.numpy(), w), (flags, k)


# more workgroups than one launch can have, 2^24 of them; and a tensor of more elements than go into a launch
@pytest.mark.parametrize("tensors, base, times", [(17, 2 ** 20, 1024), (1, 2 ** 20 + 1, 4097)])
def test_groups_of_more_than_a_launch(tensors, base, times):
    values, n = np.random.default_rng(2).standard_normal(base).astype(np.float32), base * times
    x = core.repeat(core.float32([base], values), [times])
    cs = [core.float32([1], [0.25 * (k + 1)]) for k in range(tensors)]
    outs = [(x + core.repeat(c, [n])) * x for c in cs]
    try:
        plan, ret = core.compile(outs, core.PLAN_VIEWS | core.PLAN_FUSE), ops.Tensor([n])
    except capi.HipError as e:
        if e.code != 4:
            raise
        pytest.skip("not enough device memory")
    for k in sorted({0, tensors - 1}):
        rets = [None] * tensors
        rets[k] = ret
        plan.execute(None, rets)
        want = (values + np.float32(0.25 * (k + 1))) * values
        for block in (0, times // 2, times - 2, times - 1):
            assert np.array_equal(ret.view(block * base, [base]).numpy(), want), (k, block)


def test_penalties_of_many_tensors_as_one_step():
    """sum(w * w) of three and more variables: the sums of dopt_hip_reduce_squares, bit for bit, whatever the size (one
    workgroup's chunk of 4096, several, no multiple of four)."""
    r = np.random.default_rng(2)
    ws = [core.float32([n], r.standard_normal(n).astype(np.float32)) for n in (65, 66, 4096, 4097, 50001, 1 << 20) + tuple(range(80, 160))]
    outs = [core.sum(w * w) for w in ws]
    want = core.compile(outs).execute()
    plan = core.compile(outs, core.PLAN_VIEWS | core.PLAN_FUSE | core.PLAN_TIMING)
    for g, w in zip(plan.execute(), want):
        assert np.array_equal(g, w)
    assert any(k.startswith("mul+sum*") for k in plan.profile()), plan.profile()


def test_batched_copies_of_every_length_and_alignment():
    lib = capi.load()
    r = np.random.default_rng(4)
    lengths = [1, 3, 4, 5, 1023, 1024, 1025, 4095, 4096, 4100, 16384, 70001] + [int(v) for v in r.integers(1, 9000, 140)]
    src = [ops.tensor(r.standard_normal(n + 8).astype(np.float32)) for n in lengths]
    dst = [ops.tensor(np.zeros(n + 8, np.float32)) for n in lengths]
    at = [(int(r.integers(0, 3)) * 2, int(r.integers(0, 5))) for _ in lengths]
    n = len(lengths)
    capi.check(lib.dopt_hip_copy_d2d_batch(n, (C.c_void_p * n)(*[d.ptr + 4 * j for d, (_, j) in zip(dst, at)]),
                                           (C.c_void_p * n)(*[s.ptr + 4 * i for s, (i, _) in zip(src, at)]),
                                           (C.c_size_t * n)(*[4 * k for k in lengths])))
    for s, d, (i, j), k in zip(src, dst, at, lengths):
        want = np.zeros(k + 8, np.float32)
        want[j:j + k] = s.numpy()[i:i + k]
        assert np.array_equal(d.numpy(), want)


def test_batched_copies_of_more_than_a_launch():
    """Nine copies of 2^31 - 1 words that are not on quads: more workgroups than one launch can have, 2^24 of them."""
    n, edge = 2 ** 31 - 1, 4096
    r = np.random.default_rng(6)
    try:
        src, dst = ops.Tensor([n + 8]), [ops.Tensor([n + 8]) for _ in range(9)]
    except capi.HipError as e:
        if e.code != 4:
            raise
        pytest.skip("not enough device memory")
    places = [0, n // 2, n + 8 - edge]
    values = [r.standard_normal(edge).astype(np.float32) for _ in places]
    for p, v in zip(places, values):
        src.view(p, [edge]).set(v)
    capi.check(capi.load().dopt_hip_copy_d2d_batch(9, (C.c_void_p * 9)(*[d.ptr + 4 * 3 for d in dst]), (C.c_void_p * 9)(*[src.ptr + 4 * 2] * 9),
                                                   (C.c_size_t * 9)(*[4 * n] * 9)))
    for k, d in enumerate(dst):   # words 2 .. 2 + n of the source at 3 .. 3 + n
        assert np.array_equal(d.view(0, [edge]).numpy(), np.concatenate([np.zeros(3, np.float32), values[0][2:-1]])), k
        assert np.array_equal(d.view(n // 2 + 1, [edge]).numpy(), values[1]), k
        assert np.array_equal(d.view(n + 8 - edge, [edge]).numpy(), np.concatenate([[0], values[2][:-6], np.zeros(5)]).astype(np.float32)), k
