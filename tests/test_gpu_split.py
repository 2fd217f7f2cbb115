"""fp32 products formed on the bf16 matrix instructions (three bf16 parts per value): the tile edges, the cuts of the
reduction and operands that are not finite, against float64."""
import time

import numpy as np
import pytest

from dopt_amd import capi, ops

pytestmark = pytest.mark.gpu
T = ops.tensor


def rng(seed):
    return np.random.default_rng(seed)


def walk(terms):
    """What the sum may be off by as a share of sum |a.b|: per 16 terms at most 12 roundings of 2^-24 of a partial sum that
    never exceeds sum |a.b|, as a random walk of that many steps, six standard deviations; plus one final rounding."""
    return (6 * np.sqrt(0.75 * terms) + 1) * 2.0 ** -24


def rounded_once_per_term(terms):
    """Relative error (2-norm) of a sum of `terms` products of zero mean that is rounded after each: a rounding is uniform over
    one unit in the last place, 0.43 * 2^-24 of the partial sum in the root mean square (the leading digits of the partial sum
    spread evenly over their logarithm), and the partial sums grow with the root of their length: 0.43 / sqrt(2) * sqrt(terms)."""
    return 0.30 * 2.0 ** -24 * np.sqrt(terms)


def check_norm(got, want, terms, what):
    """Against float64 in the 2-norm.  Not further off than one rounding per term, plus the roundings of the values themselves (four
    of a result: the Winograd transforms, the parts' sum and the last)."""
    got = got.astype(np.float64)
    assert np.all(np.isfinite(got)), what
    assert np.linalg.norm(got - want) <= (rounded_once_per_term(terms) + 4 * 2.0 ** -24) * np.linalg.norm(want), what


# one tile of every size and one value more; reductions of one slab, a part of one, several cuts; no multiple of four
@pytest.mark.parametrize("shape", [(65, 2048, 2100), (256, 256, 20000), (257, 1024, 4099), (130, 3001, 1030), (2049, 2047, 17),
                                   (1030, 4100, 1025), (4096, 4096, 64), (1537, 1538, 2050)])
@pytest.mark.parametrize("flags", [(False, False), (False, True), (True, False), (True, True)])
def test_large_products(shape, flags):
    M, N, K = shape
    r = rng(M + N + K)
    for positive in (False, True):
        a, b = r.standard_normal((M, K)).astype(np.float32), r.standard_normal((K, N)).astype(np.float32)
        if positive:
            a, b = np.maximum(a, 0), np.maximum(b, 0)
        sa, sb = (np.ascontiguousarray(a.T) if flags[0] else a), (np.ascontiguousarray(b.T) if flags[1] else b)
        got = ops.matmul_t(T(sa), T(sb), *flags).numpy()
        pick = r.integers(0, M, 64), r.integers(0, N, 64)
        rows, cols = np.append(pick[0], [0, M - 1, M - 1]), np.append(pick[1], [N - 1, 0, N - 1])
        want = np.einsum("ik,ki->i", a[rows].astype(np.float64), b[:, cols].astype(np.float64))
        mag = np.einsum("ik,ki->i", np.abs(a[rows]).astype(np.float64), np.abs(b[:, cols]).astype(np.float64))
        assert np.all(np.abs(got[rows, cols] - want) <= walk(K) * mag), (positive, np.max(np.abs(got[rows, cols] - want) / mag))


def fp32_sum(a, b, cuts):
    """a b, the reduction in `cuts` equal parts, each added term by term and rounded to fp32 after each, then the parts."""
    K = a.shape[1]
    depth = -(-K // cuts)
    pad = np.zeros((a.shape[0], depth * cuts - K))
    pa = np.hstack([a.astype(np.float64), pad]).reshape(a.shape[0], cuts, depth)
    pb = np.vstack([b.astype(np.float64), np.zeros((depth * cuts - K, b.shape[1]))]).reshape(cuts, depth, b.shape[1])
    acc = np.zeros((cuts, a.shape[0], b.shape[1]), np.float32)
    for k in range(depth):
        acc = (acc + pa[:, :, k].T[:, :, None] * pb[:, k][:, None, :]).astype(np.float32)
    total = acc[0]
    for c in range(1, cuts):
        total = total + acc[c]
    return total


# (M, N, K, cuts of the fp32 kernels): small outputs, which had eight; larger ones with three, two and none;
# a reduction too long for the cuts there may be, of non-negative terms
@pytest.mark.parametrize("shape", [(469, 5446, 173, 8), (2837, 897, 106, 8), (395, 5955, 588, 3), (1066, 2834, 79, 8), (3818, 1623, 2673, 2),
                                   (3000, 3000, 1400, 1), (3000, 3000, 200, 1), (300, 300, 500000, 32)])
def test_large_products_are_not_further_off_than_in_fp32(shape):
    M, N, K, cuts = shape
    r = rng(M + K)
    a, b = np.maximum(r.standard_normal((M, K), np.float32), 0), r.standard_normal((K, N), np.float32)
    if K > 100000:
        b = np.abs(b)
    side = 16 if K > 100000 else 48
    rows, cols = r.choice(M, side, replace=False), r.choice(N, side, replace=False)
    got = ops.matmul(T(a), T(b)).numpy()[np.ix_(rows, cols)]
    a, b = a[rows], b[:, cols]
    want, fp32 = a.astype(np.float64) @ b.astype(np.float64), fp32_sum(a, b, cuts)
    assert fp32.dtype == np.float32
    # (four standard deviations of a root mean square over side^2 values)
    assert np.linalg.norm(got - want) <= np.linalg.norm(fp32 - want) * (1 + 4 / np.sqrt(2 * side * side))


@pytest.mark.parametrize("shape", [(16384, 16384, 16384), (8192, 8192, 32768), (4096, 6000, 65536), (16384, 8192, 8208)])
def test_long_reductions_take_no_more_space_than_their_operands(shape):
    """A cut needs a copy of the output for each part: 4.3 GB for the first shape in four."""
    M, N, K = shape
    for ta in (0, 1):
        for tb in (0, 1):
            cuts = capi.load().dopt_hip_sgemm_order(ta, tb, M, N, K) >> 8 & 0xffff
            assert cuts == 1 or cuts * M * N <= M * K + K * N


def test_parts_below_the_bf16_rounding_count():
    """Operands that differ in their last bits only: a product of the leading bf16 parts alone would be the same for both."""
    M, N, K = 300, 2048, 2048
    a = np.full((M, K), 1.0 + 2.0 ** -23, np.float32)
    b = np.full((K, N), 1.0 - 2.0 ** -24, np.float32)
    got = ops.matmul(T(a), T(b)).numpy()
    want = K * (1.0 + 2.0 ** -23) * (1.0 - 2.0 ** -24)
    assert np.all(np.abs(got - want) <= want * 2.0 ** -23)


def test_operands_that_are_not_finite():
    M, N, K = 300, 2048, 2048
    r = rng(5)
    a, b = r.standard_normal((M, K)).astype(np.float32), r.standard_normal((K, N)).astype(np.float32)
    a[3, 5], a[200, 7], b[9, 1000], a[10, 0], b[11, 3] = np.inf, np.nan, -np.inf, 3.4e38, 1e-41
    got = ops.matmul(T(a), T(b)).numpy()
    with np.errstate(all="ignore"):
        want = a.astype(np.float64) @ b.astype(np.float64)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    inf = np.isinf(want)
    assert np.array_equal(got[inf], want[inf])
    with np.errstate(all="ignore"):
        over = np.abs(want) > 3.4e38
        mag = np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)
    fine = np.isfinite(want) & ~over & np.isfinite(got)
    assert fine.sum() > 0.9 * M * N
    assert np.all(np.abs(got[fine] - want[fine]) <= walk(K) * mag[fine])


@pytest.mark.parametrize("shape", [(2304, 2304, 1100), (2049, 2560, 1030), (300, 2048, 700)])
def test_finite_values_keep_their_bits_beside_others(shape):
    """An infinity or a NaN changes its own row or column: what dopt_hip_sgemm_order promises, equal bits whichever way the operands
    are stored and for the transposed product, holds for the values beside it, and they are what they are without it."""
    M, N, K = shape
    r = rng(M)
    a, b = r.standard_normal((M, K), np.float32), r.standard_normal((K, N), np.float32)
    plain = ops.matmul(T(a), T(b)).numpy()
    a[3, 5], a[200, 7], b[9, 1000], a[10, 0] = np.inf, np.nan, -np.inf, 1e36
    lib = capi.load()
    order = lib.dopt_hip_sgemm_order(0, 0, M, N, K)
    got = ops.matmul(T(a), T(b)).numpy()
    rows, cols = np.delete(np.arange(M), [3, 10, 200]), np.delete(np.arange(N), 1000)
    assert np.array_equal(got[np.ix_(rows, cols)], plain[np.ix_(rows, cols)])
    at, bt = np.ascontiguousarray(a.T), np.ascontiguousarray(b.T)
    seen = 0
    for ta, tb in ((False, True), (True, False), (True, True)):
        if lib.dopt_hip_sgemm_order(int(ta), int(tb), M, N, K) == order:
            again = ops.matmul_t(T(at if ta else a), T(bt if tb else b), ta, tb).numpy()
            assert np.array_equal(again, got, equal_nan=True), (ta, tb)
            seen += 1
        if lib.dopt_hip_sgemm_order(int(ta), int(tb), N, M, K) == order:
            again = ops.matmul_t(T(b if ta else bt), T(a if tb else at), ta, tb).numpy().T
            assert np.array_equal(again, got, equal_nan=True), ("transposed", ta, tb)
            seen += 1
    assert seen >= 3


ROUTES = {9: "rows", 10: "rows 256 x 256"}   # the kernels of the first byte of dopt_hip_sgemm_order that split their operands


def route(ta, tb, M, N, K):
    """(kernel, cuts, slabs of 16 steps per cut, slabs per pass)"""
    o = capi.load().dopt_hip_sgemm_order(int(ta), int(tb), M, N, K)
    return ROUTES.get(o & 0xff), o >> 8 & 0xffff, o >> 24 & 0xfffffff, o >> 52


# every tile, with the sum in one pass, in passes that wait in registers (128 x 128) and in C (the others), and cut: whole tiles and
# ragged ones, reductions of an odd number of slabs and no multiple of four
@pytest.mark.parametrize("shape,kernel,cuts,passes", [
    ((3072, 2816, 1104), "rows 256 x 256", 1, 2), ((3001, 2879, 1101), "rows 256 x 256", 1, 2), ((4096, 2304, 5000), "rows 256 x 256", 3, 1),
    ((1500, 1500, 2050), "rows", None, None), ((3000, 3000, 200), "rows", 1, 1), ((4100, 2050, 190), "rows", 1, 1),
    ((469, 5446, 173), "rows", 1, 6), ((130, 6001, 1030), "rows", None, None), ((2837, 897, 106), "rows", 1, 7),
    ((257, 300, 40000), "rows", None, None)])
def test_every_part_counts(shape, kernel, cuts, passes):
    """In the 2-norm: leaving out the l parts of one operand would be 2e-6 off, one of the six products of parts more than that."""
    M, N, K = shape
    r = rng(M + N)
    a, b = r.standard_normal((M, K), np.float32), r.standard_normal((K, N), np.float32)
    rows, cols = np.append(r.choice(M, 61, replace=False), [0, M - 1, M - 2]), np.append(r.choice(N, 61, replace=False), [0, N - 1, N - 2])
    want = a[rows].astype(np.float64) @ b[:, cols].astype(np.float64)
    at, bt = np.ascontiguousarray(a.T), np.ascontiguousarray(b.T)
    seen = {}
    for ta in (False, True):
        for tb in (False, True):
            name, c, depth, length = route(ta, tb, M, N, K)
            assert name == kernel and cuts in (None, c) and passes in (None, -(-depth // length)), (name, c, depth, length)
            got = ops.matmul_t(T(at if ta else a), T(bt if tb else b), ta, tb).numpy()
            assert np.linalg.norm(got[np.ix_(rows, cols)] - want) <= min(rounded_once_per_term(K), 1e-6) * np.linalg.norm(want)
            first = seen.setdefault((c, depth, length), got)
            assert np.array_equal(got, first), (ta, tb)


@pytest.mark.parametrize("shape", [(3072, 2816, 1104), (3001, 2879, 1101)])
def test_not_finite_in_either_pass(shape):
    M, N, K = shape
    assert route(0, 0, M, N, K)[:2] == ("rows 256 x 256", 1)
    r = rng(M)
    a, b = r.standard_normal((M, K), np.float32), r.standard_normal((K, N), np.float32)
    a[3, 5], a[700, K - 5], b[9, 1000], b[K - 3, 77], a[10, 0], a[11, K - 1] = np.inf, np.nan, -np.inf, np.nan, 1e36, 3.4e38
    got = ops.matmul(T(a), T(b)).numpy()
    rows, cols = np.append(r.choice(M, 50, replace=False), [3, 700, 10, 11]), np.append(r.choice(N, 50, replace=False), [1000, 77])
    with np.errstate(all="ignore"):
        want = a[rows].astype(np.float64) @ b[:, cols].astype(np.float64)
        mag = np.abs(a[rows]).astype(np.float64) @ np.abs(b[:, cols]).astype(np.float64)
    got = got[np.ix_(rows, cols)]
    assert np.array_equal(np.isnan(got), np.isnan(want))
    inf = np.isinf(want)
    assert np.array_equal(got[inf], want[inf])
    fine = np.isfinite(want) & (mag < 3.4e38)
    assert np.all(np.isfinite(got[fine])) and np.all(np.abs(got[fine] - want[fine]) <= walk(K) * mag[fine])


# ---- the Winograd convolution kernel

BT = np.array([[1, 0, -1, 0], [0, 1, 1, 0], [0, -1, 1, 0], [0, 1, 0, -1]], np.float64)
G = np.array([[1, 0, 0], [.5, .5, .5], [.5, -.5, .5], [0, 0, 1]], np.float64)
AT = np.array([[1, 1, 1, 0], [0, 1, -1, -1]], np.float64)


def sandwich(m, x):
    """m x m^T over the last two axes, where a zero of m takes nothing from an infinity."""
    def left(m, x):
        out = []
        for row in m:
            out.append(sum(c * x[..., i, :] for i, c in enumerate(row) if c != 0))
        return np.stack(out, axis=-2)
    with np.errstate(all="ignore"):
        return np.swapaxes(left(m, np.swapaxes(left(m, x), -1, -2)), -1, -2)


def winograd(x, w, mag=False):
    """F(2x2, 3x3) of a true convolution with pad 1 in float64, or the same with every term's absolute value."""
    f = np.abs if mag else (lambda v: v)
    N, C, H, W = x.shape
    g = f(w[:, :, ::-1, ::-1].astype(np.float64))
    xp = np.pad(f(x.astype(np.float64)), ((0, 0), (0, 0), (1, 1), (1, 1)))
    d = np.stack([np.stack([xp[:, :, r:r + H:2, q:q + W:2] for q in range(4)], -1) for r in range(4)], -2)
    u, v = sandwich(f(G), g), sandwich(f(BT), d)
    with np.errstate(all="ignore"):
        m = np.stack([np.stack([np.einsum("kc,nchw->nkhw", u[..., i, j], v[..., i, j]) for j in range(4)], -1) for i in range(4)], -2)
    y = sandwich(f(AT), m)
    return y.transpose(0, 1, 2, 4, 3, 5).reshape(N, w.shape[0], H, W)


def winograd_share(terms):
    """Of the sum of absolute terms: the sum over the channels, and at most six roundings each in the two transforms before
    it and the one after."""
    return walk(terms) + 12 * 2.0 ** -24


# 128-row and 64-row tiles; rows of 64 to 4 pixels; the last pixel tile a part of one; one chunk to spare, split reductions
@pytest.mark.parametrize("shape", [(3, 64, 32, 32, 64), (2, 64, 64, 64, 64), (1, 80, 16, 16, 160), (5, 96, 8, 8, 320),
                                   (5, 64, 16, 16, 128), (3, 208, 8, 8, 128), (9, 128, 4, 4, 256), (1, 64, 4, 4, 128),
                                   (2, 640, 8, 8, 128)])
@pytest.mark.parametrize("backward", [False, True])
def test_winograd(shape, backward):
    N, C, H, W, K = shape
    r = rng(N + C + H)
    x = np.maximum(r.standard_normal((N, C, H, W)), 0).astype(np.float32)
    w = r.standard_normal((K, C, 3, 3)).astype(np.float32)
    if backward:   # the data gradient is the convolution with the filter's transposed and reversed copy
        got = ops.conv_bwd_data(T(x), T(np.ascontiguousarray(w.transpose(1, 0, 2, 3)[:, :, ::-1, ::-1])), (N, K, H, W), (1, 1), (1, 1)).numpy()
    else:
        got = ops.convolution(T(x), T(w), (1, 1), (1, 1)).numpy()
    want, mag = winograd(x, w), winograd(x, w, True)
    assert np.all(np.abs(got - want) <= winograd_share(C) * mag), np.max(np.abs(got - want) / mag)
    check_norm(got, want, 9 * C, shape)   # (every part counts: without the l parts of one operand it would be 2e-6 off)


@pytest.mark.parametrize("shape", [(2, 64, 16, 16, 64), (2, 64, 16, 16, 128)])
def test_winograd_operands_that_are_not_finite(shape):
    N, C, H, W, K = shape
    r = rng(K)
    x = np.maximum(r.standard_normal((N, C, H, W)), 0).astype(np.float32)
    w = (0.1 * r.standard_normal((K, C, 3, 3))).astype(np.float32)
    x[0, 3, 0, 0], x[0, 5, 9, 9], x[1, 7, 4, 5], x[1, 8, 12, 12] = np.inf, np.nan, -np.inf, 3.4e38
    w[5, 2, 0, 0], w[6, 9, 1, 1] = np.inf, 3.4e38
    got = ops.convolution(T(x), T(w), (1, 1), (1, 1)).numpy()
    want, mag = winograd(x, w), winograd(x, w, True)
    huge = ~(mag < 3e38)               # where fp32 may overflow on the way, only what float64 says is not finite is known
    assert np.all(np.isfinite(got[~huge]))
    bad = ~np.isfinite(want)
    assert np.array_equal(np.isnan(got[bad]), np.isnan(want[bad]))
    inf = np.isinf(want)
    assert np.array_equal(got[inf], want[inf])
    assert np.all(np.abs(got[~huge] - want[~huge]) <= winograd_share(C) * mag[~huge])
    # a value that rounds to infinity in 16 bits but is none
    fits = huge & np.isfinite(want) & (mag < 3.4e38)
    assert np.all(np.isfinite(got[fits]))


def winograd_fp32(x, w, cuts):
    """`winograd` in fp32, the channels of each of `cuts` parts added one after the other and rounded after each, then the parts."""
    N, C, H, W = x.shape
    g = w[:, :, ::-1, ::-1]
    xp = np.pad(x, ((0, 0), (0, 0), (1, 1), (1, 1)))
    d = np.stack([np.stack([xp[:, :, r:r + H:2, q:q + W:2] for q in range(4)], -1) for r in range(4)], -2)
    u = sandwich(G.astype(np.float32), g)
    v = sandwich(BT.astype(np.float32), d).transpose(1, 4, 5, 0, 2, 3).reshape(C, 4, 4, -1)
    y = 0.0
    for part in np.array_split(np.arange(C), cuts):
        m = np.zeros((w.shape[0], 4, 4, v.shape[-1]), np.float32)
        for c in part:
            m = (m + u[:, c, :, :, None].astype(np.float64) * v[c]).astype(np.float32)
        t = sandwich(AT.astype(np.float32), m.transpose(0, 3, 1, 2))
        y = y + t.reshape(-1, N, H // 2, W // 2, 2, 2).transpose(1, 0, 2, 4, 3, 5).reshape(N, -1, H, W)
    return y


# (images, channels, rows, columns, filters, cuts of the reduction): layers whose tiles fill less than half of the chip, and a few
# tiles, whose reduction is cut into single chunks
@pytest.mark.parametrize("shape", [(32, 64, 32, 32, 64, 2), (32, 320, 16, 16, 320, 2), (32, 160, 32, 32, 160, 2), (1, 640, 8, 8, 640, 40),
                                   (18, 432, 4, 4, 128, 27), (2, 512, 4, 4, 512, 32)])
def test_winograd_is_not_further_off_than_fp32_with_the_same_cuts(shape):
    N, C, H, W, K, cuts = shape
    r = rng(C)
    x = np.maximum(r.standard_normal((N, C, H, W)), 0).astype(np.float32)
    w = (r.standard_normal((K, C, 3, 3)) * np.sqrt(2 / (9 * C))).astype(np.float32)
    rows = np.arange(0, K, K // 32 if H < 16 else K // 8)
    got = ops.convolution(T(x), T(w), (1, 1), (1, 1)).numpy()[:4, rows]
    x, w = x[:4], w[rows]
    want, fp32 = winograd(x, w), winograd_fp32(x, w, cuts)
    assert fp32.dtype == np.float32
    assert np.linalg.norm(got - want) <= np.linalg.norm(fp32 - want)


# ---- the filter gradient of 3 x 3 layers

def filter_gradient(dy, x, f=lambda v: v):
    """dw[k][c][r][s] = sum dy[n][k][p][q] x[n][c][p + 1 - r][q + 1 - s] in float64 (a true convolution, pad 1)."""
    H, W = x.shape[2:]
    xp = np.pad(f(x.astype(np.float64)), ((0, 0), (0, 0), (1, 1), (1, 1)))
    g = f(dy.astype(np.float64)).transpose(1, 0, 2, 3).reshape(dy.shape[1], -1)
    with np.errstate(all="ignore"):
        taps = [g @ xp[:, :, 2 - r:2 - r + H, 2 - s:2 - s + W].transpose(0, 2, 3, 1).reshape(-1, x.shape[1])
                for r in range(3) for s in range(3)]
    return np.stack(taps, -1).reshape(dy.shape[1], x.shape[1], 3, 3)


# 128-, 160- and 64-row tiles; rows of 64 to 8 pixels, whole images of 4 x 4; channels past a tile's edge; one chunk, split sums
@pytest.mark.parametrize("shape", [(2, 32, 64, 64, 128), (3, 48, 32, 32, 160), (1, 70, 8, 8, 64), (5, 64, 16, 16, 128),
                                   (3, 33, 8, 8, 320), (8, 64, 4, 4, 64), (4, 160, 4, 4, 160), (20, 128, 4, 4, 128), (2, 16, 32, 32, 20)])
def test_filter_gradient(shape):
    N, C, H, W, K = shape
    r = rng(N + C + H)
    x = np.maximum(r.standard_normal((N, C, H, W)), 0).astype(np.float32)
    dy = r.standard_normal((N, K, H, W)).astype(np.float32)
    got = ops.conv_bwd_filter(T(dy), T(x), (K, C, 3, 3), (1, 1), (1, 1)).numpy()
    want, mag = filter_gradient(dy, x), filter_gradient(dy, x, np.abs)
    assert np.all(np.abs(got - want) <= walk(N * H * W) * mag), np.max(np.abs(got - want) / mag)
    check_norm(got, want, N * H * W / 2, shape)


# 4 x 4 images, either side of the lines between the kernels
@pytest.mark.parametrize("shape", [(252, 64, 4, 4, 64), (256, 64, 4, 4, 64), (256, 62, 4, 4, 27), (8, 192, 4, 4, 192), (12, 191, 4, 4, 65)])
def test_filter_gradient_of_small_images(shape):
    test_filter_gradient(shape)


@pytest.mark.parametrize("shape", [(8, 64, 4, 4, 128), (256, 64, 4, 4, 64)])
def test_filter_gradient_of_small_images_that_are_not_finite(shape):
    test_filter_gradient_operands_that_are_not_finite(shape)


def test_filter_gradient_without_a_split_takes_no_longer_than_with_one():
    """4 x 4 images, an odd and an even number of quads of filter values: one workgroup added the 35 chunks of the odd one, seven
    times as long."""
    def best(N, C, H, W, K):
        dy, x, dw = T(np.ones((N, K, H, W), np.float32)), T(np.ones((N, C, H, W), np.float32)), ops.Tensor([K, C, 3, 3])
        times = []
        for _ in range(12):
            ops.sync()
            start = time.perf_counter()
            for _ in range(10):
                ops.conv_bwd_filter(dy, x, dw.shape, (1, 1), (1, 1), out=dw)
            ops.sync()
            times.append(time.perf_counter() - start)
        return min(times)
    assert best(140, 62, 4, 4, 27) < 3 * best(140, 64, 4, 4, 28)


@pytest.mark.parametrize("shape", [(4, 64, 16, 16, 128), (8, 64, 4, 4, 64), (3, 32, 32, 32, 160)])
def test_filter_gradient_operands_that_are_not_finite(shape):
    N, C, H, W, K = shape
    r = rng(K + H)
    x = r.standard_normal((N, C, H, W)).astype(np.float32)
    dy = (0.01 * r.standard_normal((N, K, H, W))).astype(np.float32)
    x[0, 3, 1, 1], x[1, 5, 2, 0], x[2, 9, 3, 3], dy[1, 7, 2, 2], dy[0, 11, 0, 0] = np.inf, np.nan, 3.4e38, -np.inf, 1e-41
    got = ops.conv_bwd_filter(T(dy), T(x), (K, C, 3, 3), (1, 1), (1, 1)).numpy()
    want, mag = filter_gradient(dy, x), filter_gradient(dy, x, np.abs)
    fine = mag < 3e38
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(got[np.isinf(want)], want[np.isinf(want)])
    assert np.all(np.abs(got[fine] - want[fine]) <= walk(N * H * W) * mag[fine])


# an odd number of filter values, so one block adds all the pixels: 64-, 128- and 160-row tiles, every pixel geometry (64-row tiles on
# 4 x 4 images: the general kernel, whose result can be split)
@pytest.mark.parametrize("shape", [(32, 33, 16, 16, 65), (8, 33, 32, 32, 65), (128, 33, 8, 8, 65), (512, 17, 4, 4, 65), (32, 17, 16, 16, 255),
                                   (2, 17, 64, 64, 255), (512, 17, 4, 4, 255), (8, 17, 32, 32, 159), (128, 17, 8, 8, 159),
                                   (512, 17, 4, 4, 159)])
def test_filter_gradient_is_not_further_off_than_one_rounding_per_term(shape):
    N, C, H, W, K = shape
    r = rng(N + H + K)
    x = np.maximum(r.standard_normal((N, C, H, W)), 0).astype(np.float32)
    dy = r.standard_normal((N, K, H, W)).astype(np.float32)
    got = ops.conv_bwd_filter(T(dy), T(x), (K, C, 3, 3), (1, 1), (1, 1)).numpy()
    want = filter_gradient(dy, x)
    # half of the terms are zero, and a sum is not rounded by adding one
    assert np.linalg.norm(got - want) <= rounded_once_per_term(N * H * W / 2) * np.linalg.norm(want)


# 65536 pixels and more in one block, every product non-negative
@pytest.mark.parametrize("shape", [(128, 33, 32, 32, 65), (16, 17, 64, 64, 255), (64, 17, 32, 32, 159)])
def test_long_filter_gradient_of_one_sign(shape):
    """Rounded after each term, the partial sums grow with their length: 0.43 * 2^-24 * sqrt(terms / 3) of the sum."""
    N, C, H, W, K = shape
    r = rng(K)
    x = np.maximum(r.standard_normal((N, C, H, W), np.float32), 0)
    dy = np.abs(r.standard_normal((N, K, H, W), np.float32))
    got = ops.conv_bwd_filter(T(dy), T(x), (K, C, 3, 3), (1, 1), (1, 1)).numpy()
    want = filter_gradient(dy, x)
    assert np.linalg.norm(got - want) <= 0.25 * 2.0 ** -24 * np.sqrt(N * H * W / 2) * np.linalg.norm(want)


# ---- the general kernels: any filter size, stride and padding

def general(x, w, pad, stride, f=lambda v: v):
    """A true convolution in float64, tap by tap; a zero of the padding times an infinity is not formed."""
    N, C, H, W = x.shape
    K, _, R, S = w.shape
    P, Q = (H + 2 * pad - R) // stride + 1, (W + 2 * pad - S) // stride + 1
    xp = np.pad(f(x.astype(np.float64)), ((0, 0), (0, 0), (pad, pad), (pad, pad)))
    g = f(w.astype(np.float64))
    y = np.zeros((N, K, P, Q))
    with np.errstate(all="ignore"):
        for r in range(R):
            for s in range(S):
                a, b = R - 1 - r, S - 1 - s
                y += np.einsum("kc,nchw->nkhw", g[:, :, r, s], xp[:, :, a:a + stride * P:stride, b:b + stride * Q:stride])
    return y


def general_gradients(x, w, dy, pad, stride, f=lambda v: v):
    N, C, H, W = x.shape
    K, _, R, S = w.shape
    P, Q = dy.shape[2:]
    xp = np.pad(f(x.astype(np.float64)), ((0, 0), (0, 0), (pad, pad), (pad, pad)))
    g, d, dx, dw = f(w.astype(np.float64)), f(dy.astype(np.float64)), np.zeros(xp.shape), np.zeros(w.shape)
    for r in range(R):
        for s in range(S):
            at = np.s_[:, :, R - 1 - r:R - 1 - r + stride * P:stride, S - 1 - s:S - 1 - s + stride * Q:stride]
            dx[at] += np.einsum("kc,nkhw->nchw", g[:, :, r, s], d)
            dw[:, :, r, s] = np.einsum("nkhw,nchw->kc", d, xp[at])
    return dx[:, :, pad:pad + H, pad:pad + W], dw


# 64-row and 128-row tiles; 1 x 1 and 5 x 5 filters, strides 1 to 3; channel counts off the slab and one past a tile's rows
@pytest.mark.parametrize("shape", [(2, 48, 13, 11, 100, 5, 2, 2), (3, 20, 9, 9, 64, 5, 2, 1), (4, 160, 16, 16, 320, 3, 1, 2),
                                   (5, 33, 8, 8, 129, 1, 0, 1), (2, 64, 16, 16, 128, 1, 0, 2), (1, 17, 10, 7, 40, 3, 0, 3)])
def test_general_convolution(shape):
    N, C, H, W, K, R, pad, stride = shape
    r = rng(C + K)
    x = np.maximum(r.standard_normal((N, C, H, W)), 0).astype(np.float32)
    w = r.standard_normal((K, C, R, R)).astype(np.float32)
    got = ops.convolution(T(x), T(w), (pad, pad), (stride, stride)).numpy()
    dy = r.standard_normal(got.shape).astype(np.float32)
    want, mag = general(x, w, pad, stride), general(x, w, pad, stride, np.abs)
    assert np.all(np.abs(got - want) <= walk(C * R * R) * mag)
    check_norm(got, want, C * R * R / 2, shape)
    wants, mags = general_gradients(x, w, dy, pad, stride), general_gradients(x, w, dy, pad, stride, np.abs)
    dx = ops.conv_bwd_data(T(dy), T(w), x.shape, (pad, pad), (stride, stride)).numpy()
    dw = ops.conv_bwd_filter(T(dy), T(x), w.shape, (pad, pad), (stride, stride)).numpy()
    assert np.all(np.abs(dx - wants[0]) <= walk(K * R * R) * mags[0])
    assert np.all(np.abs(dw - wants[1]) <= walk(dy[:, 0].size) * mags[1])
    check_norm(dx, wants[0], K * R * R / stride ** 2, shape)
    check_norm(dw, wants[1], dy[:, 0].size / 2, shape)


# either side of the lines between stages of one slab and of two: 411 tiles of one slab, 578 of nine, 1024 of ten and of thirty-two; 256 of one,
# 411 of four, 578 of ten, 1024 of thirty-three, a few
@pytest.mark.parametrize("shape", [(145, 7, 29, 25, 15, 1, 0, 1), (145, 16, 30, 34, 40, 3, 1, 1), (64, 145, 32, 32, 250, 1, 0, 1), (64, 500, 33, 31, 250, 1, 0, 1),
                                   (64, 16, 32, 32, 32, 1, 0, 1), (145, 60, 29, 25, 50, 1, 0, 1), (145, 150, 30, 34, 150, 1, 0, 1), (64, 520, 33, 31, 250, 1, 0, 1),
                                   (5, 16, 31, 9, 70, 1, 0, 1), (2, 3, 17, 15, 130, 3, 1, 1)])
def test_general_convolution_of_short_reductions(shape):
    N, C, H, W, K, R, pad, stride = shape
    r = rng(C + K)
    x, w = r.standard_normal((N, C, H, W), np.float32), r.standard_normal((K, C, R, R), np.float32)
    got = ops.convolution(T(x), T(w), (pad, pad), (stride, stride)).numpy()
    dy = r.standard_normal(got.shape, np.float32)
    dx = ops.conv_bwd_data(T(dy), T(w), x.shape, (pad, pad), (stride, stride)).numpy()
    for part in (slice(0, 1), slice(N - 1, N)):
        check_norm(got[part], general(x[part], w, pad, stride), C * R * R, shape)
        check_norm(dx[part], general_gradients(x[part], w, dy[part], pad, stride)[0], K * R * R, shape)
    x[N - 1, C - 1, 0, 0], dy[0, 0, 1, 1] = np.inf, np.nan   # the pass that forms a tile again, in stages of one slab too
    for again, plain in ((ops.convolution(T(x), T(w), (pad, pad), (stride, stride)).numpy(), got),
                         (ops.conv_bwd_data(T(dy), T(w), x.shape, (pad, pad), (stride, stride)).numpy(), dx)):
        fine = np.isfinite(again)
        assert not fine.all() and fine.mean() > 0.9 and np.array_equal(again[fine], plain[fine])


# results of odd counts whose reductions are cut: forward, backward-data, both; the classes of a stride (with classes that no tap reaches);
# filter gradients of K C 9 values (128 x 32 and 64 x 64 tiles, rows of 8, 16 and 32 pixels)
@pytest.mark.parametrize("shape", [(3, 116, 21, 11, 9, 5, 2, 1), (1, 507, 9, 13, 215, 3, 0, 1), (3, 51, 23, 7, 617, 3, 1, 1), (1, 66, 23, 7, 13, 3, 1, 1), (5, 459, 5, 11, 407, 1, 0, 1),
                                   (47, 5, 4, 11, 300, 3, 0, 2), (1, 123, 5, 7, 366, 3, 0, 2), (3, 7, 9, 7, 385, 5, 2, 3), (2, 9, 11, 7, 333, 1, 0, 2), (1, 86, 5, 8, 128, 3, 1, 2),
                                   (100, 33, 16, 16, 43, 3, 1, 1), (64, 35, 8, 8, 131, 3, 1, 1), (12, 17, 32, 32, 21, 3, 1, 1)])
def test_results_of_odd_counts_are_cut_too(shape):
    N, C, H, W, K, R, pad, stride = shape
    r = rng(C + K + R)
    x, w = r.standard_normal((N, C, H, W), np.float32), r.standard_normal((K, C, R, R), np.float32)
    ps = ((pad, pad), (stride, stride))
    got = ops.convolution(T(x), T(w), *ps).numpy()
    dy = r.standard_normal(got.shape, np.float32)
    dx, dw = ops.conv_bwd_data(T(dy), T(w), x.shape, *ps).numpy(), ops.conv_bwd_filter(T(dy), T(x), w.shape, *ps).numpy()
    wants = general_gradients(x, w, dy, pad, stride)
    check_norm(got, general(x, w, pad, stride), C * R * R, shape)
    check_norm(dx, wants[0], K * R * R / stride ** 2, shape)
    check_norm(dw, wants[1], dy[:, 0].size, shape)
    # into results off the 16-byte grid: nothing around them is touched
    for want, run in ((got, lambda o: ops.convolution(T(x), T(w), *ps, out=o)), (dx, lambda o: ops.conv_bwd_data(T(dy), T(w), x.shape, *ps, out=o)),
                      (dw, lambda o: ops.conv_bwd_filter(T(dy), T(x), w.shape, *ps, out=o))):
        whole = T(np.full(want.size + 8, 7.0, np.float32))
        run(whole.view(1, want.shape))
        flat = whole.numpy()
        assert (flat[:1] == 7.0).all() and (flat[1 + want.size:] == 7.0).all()
        assert np.allclose(flat[1:1 + want.size], want.ravel(), rtol=1e-4, atol=1e-5 * np.sqrt(C * R * R + K * R * R))


# forward of up to 64 output pixels: 1, 25, 31, 32, 33, 64 of them and 65; rows of 32 and of one more; reductions of 256 steps, of no whole
# quads, of one part and of many; strides, no padding, several images; a count of results that is no multiple of four
@pytest.mark.parametrize("shape", [(1, 400, 1, 1, 300, 1, 0, 1), (1, 257, 5, 5, 33, 5, 2, 1), (31, 29, 3, 3, 45, 3, 0, 1), (1, 64, 4, 8, 32, 3, 1, 1), (3, 131, 1, 11, 65, 3, 1, 1),
                                   (1, 256, 1, 1, 31, 1, 0, 1), (1, 256, 8, 8, 32, 1, 0, 1), (1, 640, 8, 8, 640, 3, 1, 1), (1, 99, 16, 16, 70, 3, 1, 2), (2, 37, 17, 13, 34, 7, 0, 3),
                                   (4, 512, 2, 2, 64, 3, 1, 1), (1, 1024, 4, 4, 32, 1, 0, 1), (1, 2049, 7, 7, 36, 1, 0, 1), (5, 61, 13, 1, 40, 3, 1, 1), (1, 5000, 2, 3, 32, 3, 1, 1)])
def test_convolution_of_few_pixels(shape):
    import ctypes as C_
    N, C, H, W, K, R, pad, stride = shape
    r = rng(C + K + R)
    x, w, b = r.standard_normal((N, C, H, W), np.float32), r.standard_normal((K, C, R, R), np.float32), r.standard_normal(K, np.float32)
    ps = ((pad, pad), (stride, stride))
    want = general(x, w, pad, stride)
    got = ops.convolution(T(x), T(w), *ps).numpy()
    check_norm(got, want, C * R * R, shape)
    whole = T(np.full(want.size + 8, 7.0, np.float32))   # into results off the 16-byte grid, from operands off it
    off = lambda v: T(np.append(np.zeros(1, np.float32), v.ravel())).view(1, v.shape)
    ops.convolution(off(x), off(w), *ps, out=whole.view(1, want.shape))
    flat = whole.numpy()
    assert (flat[:1] == 7.0).all() and (flat[1 + want.size:] == 7.0).all()
    check_norm(flat[1:1 + want.size].reshape(want.shape), want, C * R * R, shape)
    assert np.array_equal(flat[1:1 + want.size].reshape(want.shape), got)   # the same sums wherever the result lies
    lib, d = capi.load(), ops.conv_desc(x.shape, w.shape, *ps)
    if lib.dopt_hip_conv_packed_layout(C_.byref(d), 0) == 3:   # left open and closed: the same bits
        tx, tw, tb, o = T(x), T(w), T(b), capi.SplitSum()
        closed, opened = ops.Tensor(want.shape), ops.Tensor(want.shape)
        capi.check(lib.dopt_hip_conv_fwd_bias_packed(C_.byref(d), tx.ptr, tw.ptr, tb.ptr, closed.ptr))
        capi.check(lib.dopt_hip_conv_fwd_bias_packed_open(C_.byref(d), tx.ptr, tw.ptr, tb.ptr, opened.ptr, C_.byref(o)))
        capi.check(lib.dopt_hip_split_sum_close(C_.byref(o)))
        assert np.array_equal(opened.numpy(), closed.numpy())
        check_norm(closed.numpy(), want + b.astype(np.float64)[:, None, None], C * R * R, shape)


# filter gradients from many copies: either side of 2^17 values; rows of values that are no whole block, one block, several
@pytest.mark.parametrize("shape", [(64, 128, 16, 16, 113, 3, 1, 1), (64, 128, 16, 16, 114, 3, 1, 1), (100, 48, 31, 29, 25, 5, 2, 2), (64, 64, 32, 32, 7, 1, 0, 1),
                                   (130, 65, 28, 28, 3, 1, 0, 1), (64, 16, 32, 32, 32, 3, 1, 1), (40, 3, 33, 31, 17, 7, 3, 2)])
def test_filter_gradients_of_few_values(shape):
    N, C, H, W, K, R, pad, stride = shape
    r = rng(C + K + R)
    x, P = r.standard_normal((N, C, H, W), np.float32), [(n + 2 * pad - R) // stride + 1 for n in (H, W)]
    dy, w = r.standard_normal((N, K, *P), np.float32), np.zeros((K, C, R, R), np.float32)
    whole = T(np.full(w.size + 8, 7.0, np.float32))
    ops.conv_bwd_filter(T(dy), T(x), w.shape, (pad, pad), (stride, stride), out=whole.view(4, w.shape))
    flat = whole.numpy()
    assert (flat[:4] == 7.0).all() and (flat[4 + w.size:] == 7.0).all()
    check_norm(flat[4:4 + w.size].reshape(w.shape), general_gradients(x, w, dy, pad, stride)[1], dy[:, 0].size, shape)


def test_odd_filter_gradients_in_a_plan():
    """A backward pair whose filter gradient has an odd count beside the batch norm that adds riding sums: it adds its own."""
    from dopt_amd import core, nnet
    x, y = core.float32([64, 65, 8, 8]), core.float32([64, 10])
    init = nnet.Init(3)
    h = nnet.relu(nnet.batchNorm(nnet.conv2D(nnet.dataSource(x), 33, (3, 3), init, padding=(1, 1))))
    h = nnet.relu(nnet.batchNorm(nnet.conv2D(h, 143, (3, 3), init, padding=(1, 1))))
    h = nnet.relu(nnet.batchNorm(nnet.conv2D(h, 145, (3, 3), init, padding=(1, 1))))
    net = nnet.DAGNetwork([x], [nnet.softmax(nnet.dense(h, 10, init))])
    loss = nnet.crossEntropy(net.outputs[0].trainOutput, y)
    outs = [loss] + core.grad(loss, net.params)
    r = rng(4)
    args = {x: r.standard_normal((64, 65, 8, 8), np.float32), y: np.eye(10, dtype=np.float32)[r.integers(0, 10, 64)]}
    a, b = (core.compile(outs, f).execute(args) for f in (core.PLAN_VIEWS, core.PLAN_VIEWS | core.PLAN_FUSE))
    for p, q, o in zip(a, b, outs):
        assert np.allclose(p, q, rtol=1e-4, atol=1e-5 * max(1.0, float(np.abs(p).max()))), o.shape


def test_general_convolution_operands_that_are_not_finite():
    """A value far from every bad one is what it is without them; an infinity stays one and a NaN stays one."""
    r = rng(3)
    x = np.abs(r.standard_normal((2, 48, 13, 11))).astype(np.float32) + np.float32(0.1)
    w = np.abs(r.standard_normal((100, 48, 5, 5))).astype(np.float32) + np.float32(0.1)
    dy = np.abs(r.standard_normal((2, 100, 7, 6))).astype(np.float32) + np.float32(0.1)
    x[0, 3, 0, 0], x[0, 5, 12, 10], x[1, 7, 6, 5], dy[0, 1, 3, 3], dy[1, 9, 3, 2] = np.inf, np.nan, np.inf, np.inf, np.nan
    pad = stride = (2, 2)
    y = ops.convolution(T(x), T(w), pad, stride).numpy()
    dx = ops.conv_bwd_data(T(dy), T(w), x.shape, pad, stride).numpy()
    dw = ops.conv_bwd_filter(T(dy), T(x), w.shape, pad, stride).numpy()
    fx, fdy = np.nan_to_num(x, nan=1.0, posinf=1.0), np.nan_to_num(dy, nan=1.0, posinf=1.0)
    reach = lambda bad: bad.astype(np.float32)   # how many bad terms an output takes in
    one_x, one_w, one_dy = np.ones_like(x), np.ones_like(w), np.ones_like(dy)
    for got, nans, infs, want in (
            (y, general(reach(np.isnan(x)), one_w, 2, 2), general(reach(np.isinf(x)), one_w, 2, 2), general(fx, w, 2, 2)),
            (dx, general_gradients(x, one_w, reach(np.isnan(dy)), 2, 2)[0], general_gradients(x, one_w, reach(np.isinf(dy)), 2, 2)[0],
             general_gradients(fx, w, fdy, 2, 2)[0]),
            (dw, general_gradients(reach(np.isnan(x)), w, one_dy, 2, 2)[1] + general_gradients(one_x, w, reach(np.isnan(dy)), 2, 2)[1],
             general_gradients(reach(np.isinf(x)), w, one_dy, 2, 2)[1] + general_gradients(one_x, w, reach(np.isinf(dy)), 2, 2)[1],
             general_gradients(fx, w, fdy, 2, 2)[1])):
        assert np.array_equal(np.isnan(got), nans > 0)
        assert np.array_equal(np.isposinf(got), (infs > 0) & ~(nans > 0))
        fine = np.isfinite(got)
        assert np.all(np.abs(got[fine] - want[fine]) <= walk(2500) * want[fine])   # (every term is positive)


def test_general_convolution_error_grows_with_chains_not_with_the_reduction():
    """Reductions that are not cut (256 tiles and more): a sum is added up in chains of at most 16 slabs of 16 terms, and the chains
    one after the other, each rounded once.  So it is not further off float64 than a reduction of nine slabs whose roundings are as many
    as a chain's, and the roundings of the chains (0.43 / sqrt(2) of 2^-24 each, see rounded_once_per_term)."""
    r = rng(12)
    N, C, H, W, K = 64, 256, 17, 15, 256
    off = lambda got, want: np.linalg.norm(got - want) / np.linalg.norm(want)
    x, w = r.standard_normal((N, C, H, W), np.float32), r.standard_normal((K, C, 3, 3), np.float32)
    y = ops.convolution(T(x), T(w), (1, 1), (1, 1)).numpy()
    dy = r.standard_normal(y.shape, np.float32)
    dx = ops.conv_bwd_data(T(dy), T(w), x.shape, (1, 1), (1, 1)).numpy()
    dw = ops.conv_bwd_filter(T(dy), T(x), w.shape, (1, 1), (1, 1)).numpy()
    x9, w9 = np.ascontiguousarray(x[:, :16]), np.ascontiguousarray(w[:, :16])
    nine = off(ops.convolution(T(x9), T(w9), (1, 1), (1, 1)).numpy()[:4], general(x9[:4], w9, 1, 1))
    bound = lambda slabs, chain: 1.1 * np.hypot(nine * np.sqrt(chain / 9), 0.30 * 2.0 ** -24 * np.sqrt(slabs / chain))
    assert off(y[:4], general(x[:4], w, 1, 1)) <= bound(144, 8)
    few = np.zeros((4, C, H, W), np.float32)
    assert off(dx[:4], general_gradients(few, w, dy[:4], 1, 1)[0]) <= bound(144, 8)
    want = general_gradients(x, w[:32], np.ascontiguousarray(dy[:, :32]), 1, 1)[1]
    assert off(dw[:32], want) <= bound(N * H * W / 16, 16)


# channel counts off the slab, of x and of dy; images of one 256-pixel tile each, and several in a tile
@pytest.mark.parametrize("shape", [(3, 17, 16, 16, 23, 5, 2, 1), (3, 33, 16, 16, 20, 1, 0, 1), (4, 40, 8, 8, 130, 5, 2, 1), (3, 17, 32, 32, 24, 3, 1, 2),
                                   (2, 150, 7, 9, 70, 3, 0, 2)])
def test_general_convolution_finite_values_keep_their_bits_beside_others(shape):
    N, C, H, W, K, R, pad, stride = shape
    r = rng(K)
    x, w = (np.abs(r.standard_normal(s)).astype(np.float32) + np.float32(0.1) for s in ((N, C, H, W), (K, C, R, R)))
    y = ops.convolution(T(x), T(w), (pad, pad), (stride, stride)).numpy()
    dy = np.abs(r.standard_normal(y.shape)).astype(np.float32) + np.float32(0.1)
    gradient = lambda: ops.conv_bwd_data(T(dy), T(w), x.shape, (pad, pad), (stride, stride)).numpy()
    plain = y, gradient()
    x[1, 0, 3, 3], x[N - 1, C - 1, 0, 0], dy[1, 0, 1, 1], dy[N - 1, K - 1, 0, 2] = np.inf, np.nan, np.nan, np.inf
    for got, want in zip((ops.convolution(T(x), T(w), (pad, pad), (stride, stride)).numpy(), gradient()), plain):
        fine = np.isfinite(got)
        assert fine[0].all() and not fine.all() and np.array_equal(got[fine], want[fine])


# ---- operands and sums at the ends of the range of fp32, where bf16 parts would be lost or overflow

def scaled_pairs(p, q, least_q=-149):
    """The two operands of a product at very different scales: (p, q) with finite products between 1e-12 and 1e+35."""
    for ep, eq in ((-112, 100), (-120, 100), (-130, 100), (-140, 100), (60, 40), (-20, 110), (-80, 120)):
        for swap in (False, True):
            if swap and ep < least_q:
                continue
            with np.errstate(under="ignore"):
                yield (ep, eq, swap), np.ldexp(p, eq if swap else ep), np.ldexp(q, ep if swap else eq)


def test_products_of_operands_at_the_ends_of_the_range():
    r = rng(17)
    for M, N, K in ((300, 2048, 700), (2304, 2304, 1100)):   # the smaller tiles, 256 x 256
        p, q = r.standard_normal((M, K), np.float32), r.standard_normal((K, N), np.float32)
        for what, a, b in scaled_pairs(p, q):
            got = ops.matmul(T(a), T(b)).numpy()[:256:5]
            check_norm(got, a[:256:5].astype(np.float64) @ b.astype(np.float64), K, (M, what))


@pytest.mark.parametrize("shape", [(2, 64, 16, 16, 64), (2, 64, 8, 8, 128)])
def test_winograd_operands_at_the_ends_of_the_range(shape):
    N, C, H, W, K = shape
    r = rng(K)
    # (the filter's transform is in fp32: of subnormal values it is rounded to steps of 2^-149, with every instruction)
    for what, x, w in scaled_pairs(r.standard_normal((N, C, H, W), np.float32), r.standard_normal((K, C, 3, 3), np.float32), -122):
        check_norm(ops.convolution(T(x), T(w), (1, 1), (1, 1)).numpy(), winograd(x, w), 9 * C, what)


# 64-, 128- and 160-row tiles
@pytest.mark.parametrize("shape", [(4, 33, 16, 16, 65), (8, 32, 4, 4, 128), (4, 32, 32, 32, 160)])
def test_filter_gradient_operands_at_the_ends_of_the_range(shape):
    N, C, H, W, K = shape
    r = rng(K)
    for what, x, dy in scaled_pairs(r.standard_normal((N, C, H, W), np.float32), r.standard_normal((N, K, H, W), np.float32)):
        check_norm(ops.conv_bwd_filter(T(dy), T(x), (K, C, 3, 3), (1, 1), (1, 1)).numpy(), filter_gradient(dy, x), N * H * W, what)


def test_general_convolution_operands_at_the_ends_of_the_range():
    r = rng(23)
    x, w = r.standard_normal((2, 48, 13, 11), np.float32), r.standard_normal((100, 48, 5, 5), np.float32)
    dy, pad = r.standard_normal((2, 100, 7, 6), np.float32), (2, 2)
    for what, p, q in scaled_pairs(x, w):
        check_norm(ops.convolution(T(p), T(q), pad, pad).numpy(), general(p, q, 2, 2), 48 * 25, what)
    for what, p, q in scaled_pairs(dy, w):
        check_norm(ops.conv_bwd_data(T(p), T(q), x.shape, pad, pad).numpy(), general_gradients(x, q, p, 2, 2)[0], 100 * 9, what)
    for what, p, q in scaled_pairs(x, dy):
        check_norm(ops.conv_bwd_filter(T(q), T(p), w.shape, pad, pad).numpy(), general_gradients(p, w, q, 2, 2)[1], 84, what)


# ---- the direct 3 x 3 kernel: tiles of 32, 64, 128 and 160 rows, forward and (channels swapped) backward-data

# one and several chunks of channels, ragged and whole; rows one past a tile; whole images and rows of an image; every padding
DIRECT = [(2, 16, 16, 16, 16, 1), (3, 33, 32, 32, 17, 1), (1, 160, 16, 16, 32, 1), (2, 20, 16, 16, 48, 1), (1, 33, 64, 64, 64, 1),
          (3, 40, 8, 8, 100, 1), (1, 48, 16, 16, 256, 1), (2, 24, 10, 10, 80, 0), (5, 24, 6, 6, 20, 2), (33, 24, 32, 32, 160, 1),
          (9, 96, 4, 4, 30, 1)]


@pytest.mark.parametrize("shape", DIRECT)
def test_direct_convolution(shape):
    N, C, H, W, K, pad = shape
    r = rng(C + K)
    x = np.maximum(r.standard_normal((N, C, H, W)), 0).astype(np.float32)
    w = r.standard_normal((K, C, 3, 3)).astype(np.float32)
    got = ops.convolution(T(x), T(w), (pad, pad), (1, 1)).numpy()
    dy = r.standard_normal(got.shape).astype(np.float32)
    dx = ops.conv_bwd_data(T(dy), T(w), x.shape, (pad, pad), (1, 1)).numpy()
    want, mag = general(x, w, pad, 1), general(x, w, pad, 1, np.abs)
    assert np.all(np.abs(got - want) <= walk(C * 9) * mag)
    check_norm(got, want, C * 9 / 2, shape)
    want, mag = general_gradients(x, w, dy, pad, 1)[0], general_gradients(x, w, dy, pad, 1, np.abs)[0]
    assert np.all(np.abs(dx - want) <= walk(K * 9) * mag)
    check_norm(dx, want, K * 9, shape)


# a tile of every height; every term is positive
@pytest.mark.parametrize("shape", [(2, 20, 16, 16, 17, 1), (2, 20, 16, 16, 48, 1), (4, 40, 8, 8, 100, 1), (33, 17, 32, 32, 160, 1)])
def test_direct_convolution_operands_that_are_not_finite(shape):
    N, C, H, W, K, pad = shape
    r = rng(K)
    x, w = (np.abs(r.standard_normal(s)).astype(np.float32) + np.float32(0.1) for s in ((N, C, H, W), (K, C, 3, 3)))
    x[0, 3, 0, 0], x[N - 1, C - 1, H - 1, 2], w[K - 1, 2, 1, 1], w[1, C - 1, 0, 2], w[2, 5, 1, 0] = np.inf, np.nan, np.inf, np.nan, 2.0 ** 120
    got = ops.convolution(T(x), T(w), (pad, pad), (1, 1)).numpy()
    want = general(x, w, pad, 1)   # (zeros of the padding times an infinity are NaNs in both)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isposinf(got), np.isposinf(want))
    fine = np.isfinite(got)
    assert np.all(np.abs(got[fine] - want[fine]) <= walk(C * 9) * want[fine])


# a tile of every height with whole and ragged channels, and one reduction that is cut
@pytest.mark.parametrize("shape", [(2, 20, 16, 16, 17), (2, 16, 16, 16, 32), (2, 20, 16, 16, 48), (4, 72, 8, 8, 100), (4, 200, 8, 8, 100),
                                   (33, 17, 32, 32, 160)])
def test_direct_convolution_finite_values_keep_their_bits_beside_others(shape):
    N, C, H, W, K = shape
    r = rng(K)
    x, w, dy = (np.abs(r.standard_normal(s)).astype(np.float32) + np.float32(0.1) for s in ((N, C, H, W), (K, C, 3, 3), (N, K, H, W)))
    both = lambda: (ops.convolution(T(x), T(w), (1, 1), (1, 1)).numpy(), ops.conv_bwd_data(T(dy), T(w), x.shape, (1, 1), (1, 1)).numpy())
    plain = both()
    x[0, 3, 0, 0], x[N - 1, C - 1, H - 1, 2], dy[0, 1, 3, 3], dy[1, K - 1, 3, 2] = np.inf, np.nan, np.inf, np.nan
    for got, want in zip(both(), plain):
        fine = np.isfinite(got)
        assert 0.8 < fine.mean() < 1.0 and np.array_equal(got[fine], want[fine])
    w[K - 1, 2, 1, 1], w[1, C - 1, 0, 2] = np.inf, np.nan
    for got, want in zip(both(), plain):
        fine = np.isfinite(got)
        assert 0.7 < fine.mean() < 1.0 and np.array_equal(got[fine], want[fine])


@pytest.mark.parametrize("shape", [(2, 20, 16, 16, 17), (2, 20, 16, 16, 48), (2, 40, 8, 8, 100)])
def test_direct_convolution_operands_at_the_ends_of_the_range(shape):
    N, C, H, W, K = shape
    r = rng(K)
    for what, x, w in scaled_pairs(r.standard_normal((N, C, H, W), np.float32), r.standard_normal((K, C, 3, 3), np.float32)):
        check_norm(ops.convolution(T(x), T(w), (1, 1), (1, 1)).numpy(), general(x, w, 1, 1), 9 * C, what)


# ---- packed filters beyond 2 GiB

def cheap(r, *shape):
    """Values of mean zero that are made faster than normal ones."""
    out = r.random(shape, np.float32)
    out -= np.float32(0.5)
    return out


def test_winograd_filter_of_more_than_2_gib():
    N, C, K = 2, 5120, 5120   # 2.5 GB in three 16-bit parts
    r = rng(1)
    d = capi.ConvDesc(N, C, 4, 4, K, 3, 3, 1, 1, 1, 1)
    assert capi.load().dopt_hip_conv_packed_bytes(d, 0) == capi.load().dopt_hip_conv_packed_bytes(d, 1) == 96 * C * K > 2 ** 31
    x, dy, w = cheap(r, N, C, 4, 4), cheap(r, N, K, 4, 4), cheap(r, K, C, 3, 3)
    dw = T(w)
    rows = np.array([0, 77, 2600, K - 1])
    got = ops.convolution(T(x), dw, (1, 1), (1, 1)).numpy()[:, rows]
    want, mag = winograd(x, w[rows]), winograd(x, w[rows], True)
    assert np.all(np.abs(got - want) <= winograd_share(C) * mag)
    got = ops.conv_bwd_data(T(dy), dw, x.shape, (1, 1), (1, 1)).numpy()[:, rows]
    flipped = np.ascontiguousarray(w[:, rows].transpose(1, 0, 2, 3)[:, :, ::-1, ::-1])
    want, mag = winograd(dy, flipped), winograd(dy, flipped, True)
    assert np.all(np.abs(got - want) <= winograd_share(K) * mag)


def test_general_filter_of_more_than_2_gib():
    M = 1400000   # 25 taps x 16 (padded) x M values: 2.2 GB
    r = rng(2)
    w, x = cheap(r, M, 1, 5, 5), cheap(r, 1, 1, 6, 6)
    y = ops.convolution(T(x), T(w), (2, 2), (1, 1)).numpy()
    for rows in (np.arange(100), np.arange(M - 100, M)):
        want, mag = general(x, w[rows], 2, 1), general(x, w[rows], 2, 1, np.abs)
        assert np.all(np.abs(y[:, rows] - want) <= walk(25) * mag)
    del y
    w = w.reshape(1, M, 5, 5)
    dx = ops.conv_bwd_data(T(x), T(w), (1, M, 6, 6), (2, 2), (1, 1)).numpy()
    for rows in (np.arange(100), np.arange(M - 100, M)):
        part, zero = np.ascontiguousarray(w[:, rows]), np.zeros((1, 100, 6, 6), np.float32)
        want, mag = general_gradients(zero, part, x, 2, 1)[0], general_gradients(zero, part, x, 2, 1, np.abs)[0]
        assert np.all(np.abs(dx[:, rows] - want) <= walk(25) * mag)


def test_general_filter_of_2_27_channels():
    """Its packing takes as many workgroups as one launch cannot have, 2^24 of 256 threads."""
    N, C = 4, 2 ** 27 - 1
    r = rng(4)
    w, x, edge = np.zeros((1, C, 1, 1), np.float32), np.zeros((N, C, 1, 1), np.float32), 200
    for at in (0, C // 2, C - edge):
        w[:, at:at + edge], x[:, at:at + edge] = cheap(r, 1, edge, 1, 1), cheap(r, N, edge, 1, 1)
    y = ops.convolution(T(x), T(w), (0, 0), (1, 1)).numpy()
    used = np.flatnonzero(w[0, :, 0, 0])
    a, b = x[:, used, 0, 0].astype(np.float64), w[0, used, 0, 0].astype(np.float64)
    assert np.all(np.abs(y[:, 0, 0, 0] - a @ b) <= walk(3 * edge) * (np.abs(a) @ np.abs(b)))


def test_direct_filter_of_more_than_2_gib():
    """One output channel, padded to a tile of 64 rows: the direct kernel's copy would be 2.2 GB, its last channels out of reach."""
    C = 940000
    r = rng(3)
    assert capi.load().dopt_hip_conv_packed_bytes(capi.ConvDesc(1, C, 16, 16, 1, 3, 3, 1, 1, 1, 1), 0) == 0
    w, x = cheap(r, 1, C, 3, 3), np.zeros((1, C, 16, 16), np.float32)
    x[:, -64:] = cheap(r, 1, 64, 16, 16)
    y = ops.convolution(T(x), T(w), (1, 1), (1, 1)).numpy()
    want, mag = general(x[:, -64:], w[:, -64:], 1, 1), general(x[:, -64:], w[:, -64:], 1, 1, np.abs)
    assert np.all(np.abs(y - want) <= walk(9 * 64) * mag)
