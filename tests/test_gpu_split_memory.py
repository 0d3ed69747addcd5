"""Device memory and the rows kept for the split (bucketed kNN beyond 256
dimensions): what a call returns does not depend on how much is free, a call
whose copy does not fit still runs, and the copy is given back where another
call needs its room.  The memory is taken by tensors, never to the last: every
case leaves half a GiB or more."""
import numpy as np
import pytest

from helpers import debug_opts

pytestmark = pytest.mark.gpu

N, D, NB, M = 800_000, 320, 200, 16      # the copy: 1.0 GB, the candidates: 1.6 GB


@pytest.fixture(scope="module")
def rows():
    import torch
    g = torch.Generator(device="cuda").manual_seed(3)
    X = torch.randn(N, D, generator=g, device="cuda")
    members = np.arange(N, dtype=np.int32)
    off = np.linspace(0, N, NB + 1).astype(np.int64)
    yield X, off, members, np.zeros((NB, 0), np.int32)
    del X
    torch.cuda.empty_cache()


@pytest.fixture
def fresh():
    import gtann
    c = gtann.Context(0)
    yield c
    c.close()


def _take(leave):
    """Tensors over all of the free memory but `leave` bytes."""
    import torch
    torch.cuda.empty_cache()
    free, _ = torch.cuda.mem_get_info()
    print(f"free {free >> 20} MiB, leaving {leave >> 20}", flush=True)
    sizes = [32 << 30] * ((free - leave) >> 35) + [(free - leave) & ((32 << 30) - 1)]
    return [torch.empty(n, dtype=torch.uint8, device="cuda") for n in sizes if n > 0]


def _run(c, rows):
    ids, d = c.knn_bucketed(*rows, M)
    return ids.cpu().numpy(), d.cpu().numpy().view(np.uint32)


def test_result_does_not_depend_on_free_memory(fresh, rows):
    import gtann
    ids, bits = _run(fresh, rows)
    fresh.close()
    c = gtann.Context(0)
    taken = _take(4 << 30)
    try:
        ids2, bits2 = _run(c, rows)
    finally:
        del taken
        c.close()
    np.testing.assert_array_equal(ids2, ids)
    np.testing.assert_array_equal(bits2, bits)


def test_copy_is_given_back_and_not_needed(fresh, rows):
    with debug_opts(fresh, knn_collect=False):
        ids32, bits32 = _run(fresh, rows)
    ids, bits = _run(fresh, rows)
    table = np.random.default_rng(1).integers(0, 4_000_000, size=(4_000_000, 40)).astype(np.int32)   # 640 MB
    taken = _take(512 << 20)
    try:
        out = fresh.sanitize(table)          # takes the copy's room
        ids2, bits2 = _run(fresh, rows)      # a copy does not fit any more: the fp32 kernels
    finally:
        del taken
    np.testing.assert_array_equal(out[::1009].view(np.int32), table[::1009])
    np.testing.assert_array_equal(ids2, ids32)
    np.testing.assert_array_equal(bits2, bits32)
    import torch
    torch.cuda.empty_cache()
    ids2, bits2 = _run(fresh, rows)          # made again
    np.testing.assert_array_equal(ids2, ids)
    np.testing.assert_array_equal(bits2, bits)
