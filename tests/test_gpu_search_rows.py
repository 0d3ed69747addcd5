"""The search kernel's row forms and list sizes at their edges, against the
CPU restatement: rows read as they are stored (float32, uint8, int8; widths
around the 16-byte pieces, the quads and the 128-dimension chunks; the byte
path's limit of 256 dimensions), best lists in one register, four, or LDS,
visited tables of 16-bit entries and of ids, rows of the graph around one
wave, entry points drawn in the kernel, and a base that starts at an odd
address.  Distances are compared bit for bit."""
import numpy as np
import pytest

import gt_oracle as O
from test_gpu_search import _compare

pytestmark = pytest.mark.gpu


def _case(rng, N, D, dtype, deg, nq, E=4):
    if dtype == np.float32:
        X, Q = rng.standard_normal((N, D)).astype(np.float32), rng.standard_normal((nq, D)).astype(np.float32)
    else:
        lo, hi = (0, 256) if dtype == np.uint8 else (-128, 128)
        X, Q = rng.integers(lo, hi, size=(N, D)).astype(dtype), rng.integers(lo, hi, size=(nq, D)).astype(dtype)
    Q[Q == 0] = 1       # a zero query ties with every row under the inner product: refused by design
    g = rng.integers(0, N, size=(N, deg))
    g[:, deg // 2] = g[:, 0]            # a repeated id in every row
    g[::5, -1] = -1
    return X, g, Q, rng.integers(-1, N, size=(nq, E)).astype(np.int32)


@pytest.mark.parametrize("metric", ["l2", "ip"])
@pytest.mark.parametrize("D", [1, 2, 3, 4, 5, 15, 16, 17, 31, 33, 100, 127, 128, 131, 132, 255, 256, 257, 300])
@pytest.mark.parametrize("dtype", [np.float32, np.uint8, np.int8])
def test_row_widths(ctx, dtype, D, metric):
    rng = np.random.default_rng(D)
    X, g, Q, ent = _case(rng, 1500, D, dtype, 20, 40)
    print(f"search rows {np.dtype(dtype).name} D={D} {metric}", flush=True)
    _compare(ctx, X, g, Q, ent, 5, 40, metric=metric)


@pytest.mark.parametrize("deg,ef", [(1, 1), (16, 63), (63, 64), (64, 65), (65, 256), (130, 257), (33, 600)])
@pytest.mark.parametrize("dtype", [np.float32, np.uint8])
def test_list_sizes_and_degrees(ctx, dtype, deg, ef):
    rng = np.random.default_rng(deg * 1000 + ef)
    X, g, Q, ent = _case(rng, 4000, 48, dtype, deg, 30)
    for slots in (0, -1, 1024):
        print(f"search {np.dtype(dtype).name} deg={deg} ef={ef} slots={slots}", flush=True)
        _compare(ctx, X, g, Q, ent, min(ef, 7), ef, visited_slots=slots)


@pytest.mark.parametrize("slots", [0, 512])
def test_table_of_ids(ctx, slots):
    # more than 2^18 rows and 64 buckets: a 16-bit entry cannot hold an id
    rng = np.random.default_rng(11)
    X, g, Q, ent = _case(rng, 300_000, 4, np.float32, 12, 50)
    _compare(ctx, X, g, Q, ent, 5, 24, visited_slots=slots)
    st = _compare(ctx, X, g, Q, ent, 5, 200, visited_slots=slots)
    assert slots == 0 or st["requeued"] > 0


def test_drawn_entries(ctx):
    rng = np.random.default_rng(3)
    N, nq, E, seed = 37, 60, 9, 123     # few rows: draws repeat
    X, g, Q, _ = _case(rng, N, 10, np.float32, 6, nq)
    mask, ent = (1 << 64) - 1, np.full((nq, E), -1, np.int32)
    for q in range(nq):
        row = []
        for e in range(E):
            z = (seed + 0x9E3779B97F4A7C15 * (q * E + e + 1)) & mask
            z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & mask
            z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & mask
            row.append((z ^ (z >> 31)) % N)
        row = sorted(set(row))
        ent[q, :len(row)] = row
    ids, d, _ = ctx.search(X, g, Q, topk=4, ef=8, num_entry=E, seed=seed)
    rid, rd, _ = O.search(X, g, Q, ent, 4, 8)
    np.testing.assert_array_equal(ids, rid)
    np.testing.assert_array_equal(d.view(np.uint32), rd.view(np.uint32))


@pytest.mark.parametrize("dtype", [np.float32, np.uint8])
def test_base_at_an_odd_address(ctx, dtype):
    import torch
    rng = np.random.default_rng(5)
    X, g, Q, ent = _case(rng, 2000, 50, dtype, 16, 25)
    t = torch.from_numpy(np.concatenate([X.ravel()[:1], X.ravel()])).cuda()[1:].view(2000, 50)
    gd = torch.from_numpy(np.where(g < 0, 0xFFFFFFFF, g).astype(np.uint32).view(np.int32)).cuda()
    ids, d, _ = ctx.search(t, gd, torch.from_numpy(Q).cuda(), topk=5, ef=32, entries=torch.from_numpy(ent).cuda())
    rid, rd, _ = O.search(X.astype(np.float32), g, Q.astype(np.float32), ent, 5, 32)
    np.testing.assert_array_equal(ids.cpu().numpy(), rid)
    np.testing.assert_array_equal(d.cpu().numpy().view(np.uint32), rd.view(np.uint32))


@pytest.mark.parametrize("metric", ["l2", "ip"])
@pytest.mark.parametrize("D,deg,ef", [(257, 33, 64), (449, 17, 1), (322, 64, 63), (323, 65, 65), (384, 130, 20), (703, 20, 256),
                                      (960, 48, 257), (1024, 32, 40), (321, 33, 128)])
def test_many_queries_over_long_rows(ctx, D, deg, ef, metric):
    """Calls of more than 1,024 queries read float rows beyond 256 dimensions a
    lane each: the restatement's results, and those of the same queries in
    smaller calls."""
    rng = np.random.default_rng(D + deg)
    X, g, Q, ent = _case(rng, 700, D, np.float32, deg, 1029)
    print(f"search long rows D={D} deg={deg} ef={ef} {metric}", flush=True)
    k = min(ef, 5)
    _compare(ctx, X, g, Q, ent, k, ef, metric=metric)
    big = ctx.search(X, g, Q, topk=k, ef=ef, entries=ent, metric=metric)
    for s in (slice(0, 600), slice(600, 1029)):
        part = ctx.search(X, g, Q[s], topk=k, ef=ef, entries=ent[s], metric=metric)
        np.testing.assert_array_equal(part[0], big[0][s])
        np.testing.assert_array_equal(part[1].view(np.uint32), big[1][s].view(np.uint32))
    for slots in (-1, 512):
        out = ctx.search(X, g, Q, topk=k, ef=ef, entries=ent, metric=metric, visited_slots=slots)
        np.testing.assert_array_equal(out[0], big[0])
        np.testing.assert_array_equal(out[1].view(np.uint32), big[1].view(np.uint32))
