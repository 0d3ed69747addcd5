"""Exact kNN of float rows over pool slices (rows split into three bf16 parts,
one selection over all slices' candidates) against the merging fp32 kernels
(knn_collect off) and 64 bits.  Rows whose sums are exact in both give the same
ids and distance bits; few distinct rows: more ties than a selection holds,
decided by the ids; on other float rows the error against 64 bits is no larger
than the fp32 kernels'."""
import numpy as np
import pytest

from helpers import debug_opts

pytestmark = pytest.mark.gpu


def _both(ctx, X, k, q, metric):
    got = ctx.knn_exact(X, k, queries=q, metric=metric)
    with debug_opts(ctx, knn_collect=False):
        ref = ctx.knn_exact(X, k, queries=q, metric=metric)
    return got, ref


def _same(ctx, X, k, q, metric):
    (ids, dist), (rid, rd) = _both(ctx, X, k, q, metric)
    np.testing.assert_array_equal(ids, rid)
    np.testing.assert_array_equal(dist.view(np.uint32), rd.view(np.uint32))


@pytest.mark.parametrize("n,d,nq,k,distinct", [
    (4096, 33, 256, 5, 0), (5001, 100, 300, 100, 0), (20011, 128, 257, 128, 0), (9000, 7, 9000, 64, 0),
    (70001, 20, 511, 33, 0), (4100, 300, 512, 17, 0), (30000, 16, 400, 100, 3), (6000, 96, 333, 128, 1),
    (300000, 4, 256, 10, 5),
    # blocks of 256 queries: a batch that fills the chip, an odd last block; and more than one batch
    (30011, 100, 5003, 64, 0), (131073, 9, 131073, 8, 0), (4099, 260, 140001, 6, 0),
])
def test_slices_match_the_fp32_kernels(ctx, n, d, nq, k, distinct):
    rng = np.random.default_rng(n + k)
    if distinct:
        X = rng.integers(0, 9, size=(distinct, d))[rng.integers(0, distinct, size=n)].astype(np.float32) + 0.5
    else:
        X = rng.integers(-30, 30, size=(n, d)).astype(np.float32) + 0.5
    q = None if nq == n else rng.permutation(n)[:nq] if nq < n else rng.integers(0, n, size=nq)
    print(f"exact slices n={n} d={d} nq={nq} k={k} distinct={distinct}", flush=True)
    for metric in ("l2", "ip"):
        _same(ctx, X, k, q, metric)


@pytest.mark.parametrize("metric", ["l2", "ip"])
@pytest.mark.parametrize("d", [33, 128, 300])
def test_lists_do_not_depend_on_the_batch(ctx, d, metric):
    # (5,003 queries: blocks of 256 queries and 8 waves; the smaller calls: 128 and 4)
    rng = np.random.default_rng(d)
    X = rng.standard_normal((30011, d)).astype(np.float32)
    q = rng.permutation(30011)[:5003]
    ids, dist = ctx.knn_exact(X, 20, queries=q, metric=metric)
    for nq in (1, 2, 33, 128, 255, 256, 700):
        i, v = ctx.knn_exact(X, 20, queries=q[:nq], metric=metric)
        np.testing.assert_array_equal(i, ids[:nq])
        np.testing.assert_array_equal(v.view(np.uint32), dist[:nq].view(np.uint32))


@pytest.mark.parametrize("d", [1, 100, 300])
def test_whole_numbers_beyond_two_parts(ctx, d):
    """One element of 2049..2895 per row: every sum is a whole number below
    2^24, so exact in fp32; two rows of a kind lie at distance 0."""
    rng = np.random.default_rng(d)
    n = 6000
    X = np.zeros((n, d), np.float32)
    X[np.arange(n), rng.integers(0, min(d, 5), size=n)] = rng.integers(2049, 2896, size=n)
    X[n // 2:] = X[:n - n // 2]
    q = rng.permutation(n)[:400]
    for metric in ("l2", "ip"):
        _same(ctx, X, 8, q, metric)
    assert (ctx.knn_exact(X, 8, queries=q)[1][:, 0] == 0.0).all()


def _rows(kind, rng, n, d):
    if kind == "sparse":
        X = np.zeros((n, d), np.float32)
        X[np.arange(n)[:, None], np.argsort(rng.random((n, min(d, 12))), axis=1)[:, :3]] = rng.standard_normal((n, min(d, 3)))
        return X
    if kind == "mixture":
        return (rng.uniform(-10, 10, (8, d))[rng.integers(0, 8, n)] + rng.standard_normal((n, d))).astype(np.float32)
    return rng.standard_normal((n, d)).astype(np.float32)


def _errors(X, q, out, metric):
    """Errors of the distances of `out` against 64 bits, in 2^-24 of the operands' magnitude."""
    X64 = X.astype(np.float64)
    ids, dist = out
    Q, P = X64[q][:, None], X64[ids]
    dot, qq, pp = (Q * P).sum(-1), (Q * Q).sum(-1), (P * P).sum(-1)
    e = dist - dot if metric == "ip" else dist - (qq + pp - 2 * dot)
    return e / (np.sqrt(qq * pp) if metric == "ip" else qq + pp) * 2.0 ** 24


@pytest.mark.parametrize("metric", ["l2", "ip"])
@pytest.mark.parametrize("kind,d", [("normal", 2), ("normal", 4), ("normal", 33), ("normal", 100), ("normal", 128),
                                    ("mixture", 100), ("mixture", 128), ("sparse", 64), ("sparse", 288), ("normal", 300),
                                    ("sparse", 960)])
def test_error_against_64_bits(ctx, kind, d, metric):
    rng = np.random.default_rng(d)
    n, k = 8192, 32
    X = _rows(kind, rng, n, d)
    q = rng.permutation(n)[:1024]
    e, f = (_errors(X, q, out, metric) for out in _both(ctx, X, k, q, metric))
    rms = [float(np.sqrt((x * x).mean())) for x in (e, f)]
    print(f"exact d={d} {kind} {metric}: rms error {rms[0]:.3f} ulps, fp32 kernels {rms[1]:.3f}; "
          f"largest {np.abs(e).max():.2f}, {np.abs(f).max():.2f}", flush=True)
    # the same sums in another order: 5 % for the sample (32,768 distances); a
    # single distance may round the other way once more at each end of its sum
    assert rms[0] <= 1.05 * rms[1]
    assert np.abs(e).max() <= np.abs(f).max() + 2.0


@pytest.mark.parametrize("metric", ["l2", "ip"])
@pytest.mark.parametrize("big,small", [(20, 0), (40, 0), (60, -50)])
def test_rows_of_two_magnitudes(ctx, big, small, metric):
    """Some rows with one huge coordinate, zero in all others: their inner
    products are the small ones' alone, with all of their bits.  (2^110 apart:
    more than the split rows hold, the fp32 kernels' launch.)"""
    rng = np.random.default_rng(7)
    n, d, rows = 5000, 96, 50
    X = rng.integers(-20, 20, size=(n, d)).astype(np.float32) * np.float32(2.0 ** small)
    X[:, :rows] = 0.0
    X[np.arange(rows), np.arange(rows)] = 2.0 ** big
    q = np.concatenate([np.arange(rows), rng.permutation(n - rows)[:250] + rows])
    _same(ctx, X, 20, q, metric)


@pytest.mark.parametrize("metric", ["l2", "ip"])
def test_rows_that_are_not_finite(ctx, metric):
    rng = np.random.default_rng(9)
    X = rng.integers(-20, 20, size=(5000, 60)).astype(np.float32) + 0.5
    X[10, 3] = np.inf
    X[410, 5] = -np.inf
    X[420, 7] = np.nan
    X[430] = 1e30                                # the norm is not finite
    q = np.concatenate([[10, 410, 420, 430], rng.permutation(5000)[:300]])
    _same(ctx, X, 16, q, metric)
