"""Bucketed kNN of float rows longer than 256: the collect kernel on rows
split into three bf16 parts, against the merging fp32 kernels (knn_collect off)
and 64 bits.  Integer-valued rows have exact sums, so there both paths give
the same tables bit for bit; on float rows the split path's error against 64
bits is no larger."""
import numpy as np
import pytest

from helpers import debug_opts

pytestmark = pytest.mark.gpu


def _buckets(rng, n, nb, probe):
    assign = rng.integers(0, nb, size=n)
    assign[assign == nb - 1] = 0                     # the last bucket is empty
    members = np.argsort(assign, kind="stable").astype(np.int32)
    off = np.searchsorted(assign[members], np.arange(nb + 1)).astype(np.int64)
    pr = np.stack([rng.permutation(np.delete(np.arange(nb), b))[:probe] for b in range(nb)]).astype(np.int32)
    return off, members, pr.reshape(nb, probe)


def _both(ctx, X, off, members, pr, M, metric="l2", running=None):
    with debug_opts(ctx, knn_collect=2):               # buckets of any size
        got = ctx.knn_bucketed(X, off, members, pr, M, metric=metric, running=running)
    with debug_opts(ctx, knn_collect=False):
        ref = ctx.knn_bucketed(X, off, members, pr, M, metric=metric, running=running)
    return got, ref


@pytest.mark.parametrize("n,d,nb,probe,M", [
    (3000, 257, 5, 1, 64), (2500, 320, 3, 0, 65), (4100, 288, 9, 2, 96), (1500, 500, 4, 1, 128),
    (700, 1024, 3, 1, 5), (40, 300, 2, 0, 33), (1, 270, 1, 0, 8), (193, 960, 1, 0, 128), (2000, 992, 300, 3, 16),
    (32769, 288, 20, 1, 16),   # blocks of 256 queries, odd last ones
])
def test_integer_rows_match_the_fp32_kernels(ctx, n, d, nb, probe, M):
    rng = np.random.default_rng(n + d)
    X = rng.integers(-60, 60, size=(n, d)).astype(np.float32)
    if n > 100:
        X[50:60] = X[40]                             # ties
    off, members, pr = _buckets(rng, n, nb, probe) if nb > 1 else (np.array([0, n]), np.arange(n, dtype=np.int32),
                                                                 np.zeros((1, 0), np.int32))
    print(f"wide split n={n} d={d} M={M}", flush=True)
    for metric in ("l2", "ip"):
        got, ref = _both(ctx, X, off, members, pr, M, metric)
        np.testing.assert_array_equal(got[0], ref[0])
        np.testing.assert_array_equal(got[1], ref[1])
        # merged into the table of another bucketing
        o2, m2, p2 = _buckets(np.random.default_rng(5), n, max(2, nb), 0)
        run = ctx.knn_bucketed(X, o2, m2, p2, M, metric=metric)
        got, ref = _both(ctx, X, off, members, pr, M, metric, running=run)
        np.testing.assert_array_equal(got[0], ref[0])
        np.testing.assert_array_equal(got[1], ref[1])


@pytest.mark.parametrize("metric", ["l2", "ip"])
def test_whole_numbers_beyond_two_parts(ctx, metric):
    """One element of 2049..2895 per row: every sum is a whole number below
    2^24, so exact in fp32; two rows of a kind lie at distance 0."""
    rng = np.random.default_rng(4)
    n, d = 4000, 300
    X = np.zeros((n, d), np.float32)
    X[np.arange(n), rng.integers(0, 5, size=n)] = rng.integers(2049, 2896, size=n)
    X[n // 2:] = X[:n // 2]
    got, ref = _both(ctx, X, np.array([0, n]), np.arange(n, dtype=np.int32), np.zeros((1, 0), np.int32), 8, metric)
    np.testing.assert_array_equal(got[0], ref[0])
    np.testing.assert_array_equal(got[1], ref[1])
    assert metric == "ip" or (got[1][:, 0] == 0.0).all()


@pytest.mark.parametrize("metric", ["l2", "ip"])
@pytest.mark.parametrize("big,small", [(20, 0), (40, 0), (60, -50)])
def test_rows_of_two_magnitudes(ctx, big, small, metric):
    """Some rows with one huge coordinate, zero in all others: their inner
    products are the small ones' alone, with all of their bits.  (2^110 apart:
    more than the split rows hold, the fp32 kernel's launch.)"""
    rng = np.random.default_rng(7)
    n, d, rows = 1500, 300, 50
    X = rng.integers(-20, 20, size=(n, d)).astype(np.float32) * np.float32(2.0 ** small)
    X[:, :rows] = 0.0
    X[np.arange(rows), np.arange(rows)] = 2.0 ** big
    off, members, pr = _buckets(rng, n, 3, 1)
    got, ref = _both(ctx, X, off, members, pr, 20, metric)
    np.testing.assert_array_equal(got[0], ref[0])
    np.testing.assert_array_equal(got[1], ref[1])


def _rows(kind, rng, n, d):
    if kind == "sparse":
        X = np.zeros((n, d), np.float32)
        X[np.arange(n)[:, None], np.argsort(rng.random((n, 12)), axis=1)[:, :3]] = rng.standard_normal((n, 3))
        return X
    if kind == "mixture":
        return (rng.uniform(0, 1, (8, d))[rng.integers(0, 8, n)] + 0.1 * rng.standard_normal((n, d))).astype(np.float32)
    if kind == "latent":
        return (rng.standard_normal((n, 24)) @ rng.standard_normal((24, d)) * 0.2
                + 0.02 * rng.standard_normal((n, d))).astype(np.float32)
    x = rng.standard_normal((n, d))
    return (x / np.linalg.norm(x, axis=1, keepdims=True)).astype(np.float32)


@pytest.mark.parametrize("d", [257, 288, 512, 960, 1024])
@pytest.mark.parametrize("kind,metric", [("mixture", "l2"), ("latent", "l2"), ("unit", "ip"), ("sparse", "l2"), ("sparse", "ip")])
def test_error_against_64_bits(ctx, kind, metric, d):
    rng = np.random.default_rng(d)
    n, M = 2000, 64
    X = _rows(kind, rng, n, d)
    X64 = X.astype(np.float64)
    dot = X64 @ X64.T
    sq = np.diag(dot)
    full = dot if metric == "ip" else sq[:, None] + sq[None] - 2 * dot
    scale = np.sqrt(sq[:, None] * sq[None]) if metric == "ip" else sq[:, None] + sq[None]
    rms = []
    for ids, dist in _both(ctx, X, np.array([0, n]), np.arange(n, dtype=np.int32), np.zeros((1, 0), np.int32), M, metric):
        e = (dist - np.take_along_axis(full, ids.astype(np.int64), 1)) / np.take_along_axis(scale, ids.astype(np.int64), 1)
        assert np.isfinite(e).all()
        rms.append(float(np.sqrt((e * e).mean())) * 2 ** 24)
    print(f"wide split d={d} {kind} {metric}: rms error {rms[0]:.3f} ulps, fp32 kernel {rms[1]:.3f}", flush=True)
    # the same sums in another order: 5 % for the sample (128,000 distances)
    assert rms[0] <= 1.05 * rms[1]


@pytest.mark.parametrize("metric", ["l2", "ip"])
def test_rows_that_are_not_finite_and_scales(ctx, metric):
    rng = np.random.default_rng(9)
    n, d, M = 600, 320, 32
    X = rng.integers(-20, 20, size=(n, d)).astype(np.float32)
    X[:200] *= np.float32(2.0 ** 40)
    X[200:400] *= np.float32(2.0 ** -40)
    X[401] = 0.0
    off, members, pr = _buckets(rng, n, 3, 1)
    got, ref = _both(ctx, X, off, members, pr, M, metric)
    np.testing.assert_array_equal(got[0], ref[0])
    np.testing.assert_array_equal(got[1], ref[1])
    X[10, 3] = np.inf
    X[410, 5] = -np.inf
    X[420, 7] = np.nan
    got, ref = _both(ctx, X, off, members, pr, M, metric)
    np.testing.assert_array_equal(got[0], ref[0])
    np.testing.assert_array_equal(got[1], ref[1])


@pytest.mark.parametrize("metric", ["l2", "ip"])
def test_small_scales(ctx, metric):
    """Rows around 2^-60 (the product of two rows' scales underflows, the dot
    products do not) and 2^-130 (the rows are not normal floats) among rows of
    ordinary size: sums exact in both kernels."""
    rng = np.random.default_rng(11)
    n, d, M = 600, 288, 32
    X = rng.integers(-20, 20, size=(n, d)).astype(np.float32)
    scale = -60 if metric == "l2" else -130
    X[:300] *= np.float32(2.0 ** scale)
    off, members, pr = _buckets(rng, n, 3, 1)
    got, ref = _both(ctx, X, off, members, pr, M, metric)
    np.testing.assert_array_equal(got[0], ref[0])
    np.testing.assert_array_equal(got[1], ref[1])


@pytest.mark.parametrize("size", [40, 200, 350, 500, 1000])
def test_small_buckets_stay_on_the_fp32_kernel(ctx, size):
    """Buckets below 400 rows: the fp32 kernel's table; from there on the one over split rows."""
    X = _rows("mixture", np.random.default_rng(size), 3000, 300)
    nb = 3000 // size
    off = np.linspace(0, 3000, nb + 1).astype(np.int64)
    args = (X, off, np.arange(3000, dtype=np.int32), np.zeros((nb, 0), np.int32), 32)
    split, fp32 = _both(ctx, *args)
    got = ctx.knn_bucketed(*args)
    assert (split[1].view(np.uint32) != fp32[1].view(np.uint32)).any()
    want = fp32 if 3000 / nb < 400 else split
    np.testing.assert_array_equal(got[0], want[0])
    np.testing.assert_array_equal(got[1].view(np.uint32), want[1].view(np.uint32))


def test_out_of_core_build(ctx):
    """Chunks of buckets against rows split in the member order of all: the
    resident build's table and graph."""
    X = _rows("mixture", np.random.default_rng(3), 20011, 300)
    kw = dict(n_buckets=16, M=32, K=16, rounds=2, nprobe=1)
    res = ctx.build_graph(X, **kw)
    ooc = ctx.build_graph(X, device_budget_mb=12, **kw)
    assert res.stats["ooc_chunks"] == 0 and ooc.stats["ooc_chunks"] > 3
    np.testing.assert_array_equal(ooc.knn_ids, res.knn_ids)
    np.testing.assert_array_equal(ooc.knn_dists.view(np.uint32), res.knn_dists.view(np.uint32))
    np.testing.assert_array_equal(ooc.graph, res.graph)
