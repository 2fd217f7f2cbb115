"""fp32 products formed on the bf16 matrix instructions (three bf16 parts per value): the tile edges, the cuts of the
reduction and operands that are not finite, against float64."""
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
