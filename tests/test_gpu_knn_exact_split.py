"""Exact kNN of float rows over pool slices (rows split into two fp16 parts,
one selection over all slices' candidates) against the merging fp32 kernels
(knn_collect off).  Half-integer rows: sums exact in both, so ids and distance
bits agree; few distinct rows: more ties than a selection holds, decided by
the ids."""
import numpy as np
import pytest

from helpers import debug_opts

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,d,nq,k,distinct", [
    (4096, 33, 256, 5, 0), (5001, 100, 300, 100, 0), (20011, 128, 257, 128, 0), (9000, 7, 9000, 64, 0),
    (70001, 20, 511, 33, 0), (4100, 300, 512, 17, 0), (30000, 16, 400, 100, 3), (6000, 160, 333, 128, 1),
    (300000, 4, 256, 10, 5),
])
def test_slices_match_the_fp32_kernels(ctx, n, d, nq, k, distinct):
    rng = np.random.default_rng(n + k)
    if distinct:
        X = rng.integers(0, 9, size=(distinct, d))[rng.integers(0, distinct, size=n)].astype(np.float32) + 0.5
    else:
        X = rng.integers(-30, 30, size=(n, d)).astype(np.float32) + 0.5
    q = None if nq == n else rng.permutation(n)[:nq]
    print(f"exact slices n={n} d={d} nq={nq} k={k} distinct={distinct}", flush=True)
    for metric in ("l2", "ip"):
        ids, dist = ctx.knn_exact(X, k, queries=q, metric=metric)
        with debug_opts(ctx, knn_collect=False):
            rid, rd = ctx.knn_exact(X, k, queries=q, metric=metric)
        np.testing.assert_array_equal(ids, rid)
        np.testing.assert_array_equal(dist.view(np.uint32), rd.view(np.uint32))
