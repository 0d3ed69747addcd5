"""Pageable inputs of 32 MiB and more and results of 2 MiB and more go through
two pinned halves of 4 MiB: the same results as device tensors, whatever the
last chunk's length."""
import numpy as np
import pytest

import gt_oracle as O

pytestmark = pytest.mark.gpu


# rows of 4 bytes x d and results of 4 bytes x k: below the limits, at them, one element past them and past a chunk,
# odd chunk counts
@pytest.mark.parametrize("n,d,k", [(16383, 128, 5), (16384, 128, 128), (16391, 131, 127), (24577, 128, 86), (70001, 61, 33),
                                   (65535, 128, 8), (65536, 128, 8), (65543, 131, 9), (98305, 129, 5), (8192, 64, 64),
                                   (8191, 64, 64)])
def test_host_arrays_match_device_tensors(ctx, n, d, k):
    import torch
    X = np.random.default_rng(n).integers(0, 50, size=(n, d)).astype(np.float32)
    print(f"staging n={n} d={d} k={k}", flush=True)
    ids, dist = ctx.knn_exact(torch.from_numpy(X).cuda(), k)
    for host in (X, torch.from_numpy(X).pin_memory()):
        hi, hd = ctx.knn_exact(host, k)
        np.testing.assert_array_equal(np.asarray(hi), ids.cpu().numpy())
        np.testing.assert_array_equal(np.asarray(hd), dist.cpu().numpy())
    table = np.sort(np.random.default_rng(k).integers(0, n, size=(n, k)), axis=1).astype(np.int32)
    np.testing.assert_array_equal(ctx.sanitize(table).view(np.int32), np.asarray(O.sanitize(table)).view(np.int32))
