"""The library's work as its users call it: graph builds, exact and bucketed
kNN, graph optimisation and graph search, each through the public entry points
of gpu-talored-ann_amd/gtann.py.

A case is a dict of plain values; `kind` names the entry point:

  search        Context.search of `nq` held-out queries over a built graph
  knn_exact     Context.knn_exact of `nq` of the rows against all of them
  knn_bucketed  Context.knn_bucketed, one round over the caller's own buckets
                (`running`: merged into the table of an earlier round)
  optimize      Context.optimize of a host kNN table (sanitized, rank order)
  build         Context.build_graph, rows on the GPU to graph and table there

`dtype` is the stored type of the rows: f32; int (integer-valued float32 in
[0, 255], as SIFT's .fbin files hold); u8; i8.  `data` is their distribution:

  mixture  Gaussian clusters around uniform centres (the benchmark's C1, C2,
           C4 and C5), `clusters` of them; rows of more than 256 dimensions
           vary around their centre in 32 latent directions plus a little
           noise, as real descriptors of such widths do (with independent
           noise in 960 dimensions a row's neighbours all lie at nearly one
           distance, and rounding would decide 1 % of a list's order)
  unit     the same on the unit sphere (C3), for the inner product
  latent   a 16-dimensional latent Gaussian through a random map (S2): a
           connected graph, what a search needs
"""
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gpu-talored-ann_amd"))
import gtann  # noqa: E402

_CTX = None


def _ctx():
    """The one context a program keeps for its GPU."""
    global _CTX
    if _CTX is None:
        _CTX = gtann.Context(0)
    return _CTX


def listed():
    return [
        # one query at a time, the latency an interactive caller sees; a width that is no multiple of 32
        {"name": "search_one_200k_x100", "kind": "search", "n": 200_003, "d": 100, "dtype": "f32", "data": "latent",
         "metric": "l2", "degree": 32, "nq": 1, "ef": 64, "topk": 10},
        # a serving batch over byte descriptors (.u8bin)
        {"name": "search_1000_u8", "kind": "search", "n": 1_000_000, "d": 128, "dtype": "u8", "data": "latent",
         "metric": "l2", "degree": 32, "nq": 1000, "ef": 64, "topk": 10},
        # an offline query set at the command line's own beam width (the benchmark's S2 leg)
        {"name": "search_10k_ef200", "kind": "search", "n": 1_000_000, "d": 128, "dtype": "int", "data": "latent",
         "metric": "l2", "degree": 32, "nq": 10_000, "ef": 200, "topk": 10},
        # ground truth for a query sample (build_knn.py, the recall checks); 100 neighbours, 100 dimensions
        {"name": "knn_exact_10k_x_1m", "kind": "knn_exact", "n": 1_000_003, "d": 100, "dtype": "f32", "data": "mixture",
         "clusters": 1000, "metric": "l2", "nq": 10_000, "k": 100},
        # one round over a caller's own buckets, wide rows (run_round on C4's width)
        {"name": "knn_bucketed_100k_x960", "kind": "knn_bucketed", "n": 100_003, "d": 960, "dtype": "f32",
         "data": "mixture", "clusters": 25, "metric": "l2", "probe": 1, "M": 96, "running": False},
        # `gtann optimize` / prune.py on a kNN table read from a file: host table in, host graph out
        {"name": "optimize_host_200k", "kind": "optimize", "n": 200_003, "M": 64, "K": 32},
        # the smallest build in use (C1): launches and latency
        {"name": "build_10k_x128", "kind": "build", "n": 10_000, "d": 128, "dtype": "f32", "data": "mixture",
         "clusters": 64, "metric": "l2", "buckets": 16, "M": 64, "K": 32, "refine": 0},
        # an ordinary build at sizes that are no multiple of anything, with a refinement pass
        {"name": "build_150k_x100_refine", "kind": "build", "n": 150_011, "d": 100, "dtype": "f32", "data": "mixture",
         "clusters": 300, "metric": "l2", "buckets": 37, "M": 48, "K": 24, "refine": 1},
        # integer-valued float rows (C2, the headline benchmark)
        {"name": "build_1m_x128_int", "kind": "build", "n": 1_000_000, "d": 128, "dtype": "int", "data": "mixture",
         "clusters": 1000, "metric": "l2", "buckets": 256, "M": 64, "K": 32, "refine": 0},
        # unit vectors under the inner product (C3)
        {"name": "build_1m_x96_ip", "kind": "build", "n": 1_000_000, "d": 96, "dtype": "f32", "data": "unit",
         "clusters": 500, "metric": "ip", "buckets": 256, "M": 64, "K": 32, "refine": 0},
        # wide float rows (C4)
        {"name": "build_1m_x960", "kind": "build", "n": 1_000_000, "d": 960, "dtype": "f32", "data": "mixture",
         "clusters": 200, "metric": "l2", "buckets": 512, "M": 96, "K": 48, "refine": 0},
        # the largest dataset: ten million signed bytes (C5)
        {"name": "build_10m_x128_i8", "kind": "build", "n": 10_000_000, "d": 128, "dtype": "i8", "data": "mixture",
         "clusters": 4096, "metric": "l2", "buckets": 2048, "M": 64, "K": 32, "refine": 0},
    ]


def _log(rng, lo, hi):
    """An integer in [lo, hi], uniform over its logarithm."""
    return max(lo, min(hi, int(lo * (hi / lo) ** rng.random())))


def _row_kind(rng, d):
    """(dtype, data, metric) of a drawn dataset; rows beyond 256 dimensions are float."""
    pick = rng.random()
    if d > 256 or pick < 0.35:
        return "f32", "mixture", "l2"
    if pick < 0.5:
        return "f32", "unit", "ip"
    return rng.choice(["int", "u8", "i8"]), "mixture", "l2"


def draw(rng):
    kind = rng.choice(["search", "search", "knn_exact", "knn_bucketed", "optimize", "build", "build", "build"])
    if kind == "search":
        ef = _log(rng, 10, 256)
        dtype = rng.choice(["f32", "int", "u8", "i8"])
        return {"kind": kind, "n": _log(rng, 20_000, 1_000_000), "d": _log(rng, 48, 256), "dtype": dtype,
                "data": "latent", "metric": "ip" if dtype == "f32" and rng.random() < 0.25 else "l2",
                "degree": rng.choice([16, 24, 32, 48, 64]), "nq": _log(rng, 1, 10_000), "ef": ef,
                "topk": _log(rng, 1, min(ef, 100))}
    if kind == "knn_exact":
        d = _log(rng, 32, 960)
        dtype, data, metric = _row_kind(rng, d)
        n = _log(rng, 10_000, 1_000_000)
        return {"kind": kind, "n": n, "d": d, "dtype": dtype, "data": data, "clusters": max(16, n // 1000),
                "metric": metric, "nq": _log(rng, 1, min(n, 10_000)), "k": _log(rng, 1, 128)}
    if kind == "knn_bucketed":
        d = _log(rng, 32, 960)
        dtype, data, metric = _row_kind(rng, d)
        n = _log(rng, 10_000, 200_000)
        return {"kind": kind, "n": n, "d": d, "dtype": dtype, "data": data, "clusters": max(4, n // 4000),
                "metric": metric, "probe": rng.randint(0, 2), "M": _log(rng, 16, 128), "running": rng.random() < 0.5}
    if kind == "optimize":
        M = rng.choice([32, 48, 64, 96, 128])
        return {"kind": kind, "n": _log(rng, 5_000, 400_000), "M": M, "K": min(64, rng.choice([M // 2, M // 3, M // 4]))}
    d = _log(rng, 32, 960)
    dtype, data, metric = _row_kind(rng, d)
    n = _log(rng, 5_000, 1_000_000)
    M = rng.choice([32, 48, 64, 96])
    return {"kind": kind, "n": n, "d": d, "dtype": dtype, "data": data, "clusters": max(16, n // 2000),
            "metric": metric, "buckets": max(4, n // 4000), "M": M, "K": M // 2,
            "refine": 1 if dtype == "f32" and rng.random() < 0.25 else 0}


# ------------------------------------------------------------------ inputs


def _stored(x, dtype):
    """Rows of about [0, 255] (i8: [-128, 127]) in the stored type."""
    if dtype == "f32":
        return x
    if dtype == "i8":
        return x.sub_(128.0).round_().clamp_(-127, 127).to(torch.int8)
    x = x.round_().clamp_(0, 255)
    return x.to(torch.uint8) if dtype == "u8" else x


def _rows(c, n, g):
    """(rows (n, d), cluster of every row or None), drawn from the generator."""
    d, dev = c["d"], "cuda"
    integer = c["dtype"] != "f32"
    if c["data"] == "latent":
        basis = torch.linalg.qr(torch.randn(d, 16, generator=g, device=dev))[0]
    else:
        k = c["clusters"]
        if c["data"] == "unit":
            centres = torch.nn.functional.normalize(torch.randn(k, d, generator=g, device=dev))
            sigma = 0.3 / d ** 0.5
        elif integer:
            # i8 rows spread over [-100, 100] around their centres' offset of 128 with sigma 15, bytes over
            # [0, 255] with sigma 20
            lo, hi, sigma = (28.0, 228.0, 15.0) if c["dtype"] == "i8" else (0.0, 255.0, 20.0)
            centres = torch.rand(k, d, generator=g, device=dev) * (hi - lo) + lo
        else:
            wide = d > 256
            centres = torch.rand(k, d, generator=g, device=dev) * (1.0 if wide else 20.0) - (0.0 if wide else 10.0)
            sigma = 0.02 if wide else 1.0
            if wide:
                directions = torch.linalg.qr(torch.randn(d, 32, generator=g, device=dev))[0].T * (0.1 * (d / 32) ** 0.5)
    out, labels = [], []
    for s in range(0, n, 1 << 18):
        m = min(1 << 18, n - s)
        if c["data"] == "latent":
            x = torch.randn(m, 16, generator=g, device=dev).mul_(24.0) @ basis.T
            x = x.add_(torch.randn(m, d, generator=g, device=dev), alpha=2.0)
            x = x.add_(128.0) if integer else x.div_(32.0)
        else:
            lab = torch.randint(0, k, (m,), generator=g, device=dev)
            x = centres[lab].add_(torch.randn(m, d, generator=g, device=dev), alpha=sigma)
            if c["data"] == "mixture" and d > 256:
                x = x.addmm_(torch.randn(m, 32, generator=g, device=dev), directions)
            if c["data"] == "unit":
                x = torch.nn.functional.normalize(x)
            labels.append(lab)
        out.append(_stored(x, c["dtype"]))
    return torch.cat(out), torch.cat(labels) if labels else None


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _bucketing(labels, nb, probe, X, shift=0):
    """Buckets of a caller who clustered its rows: offsets, members (bucket-major) and, per bucket, the `probe`
    buckets of nearest mean.  shift > 0: another clustering of the same rows (every row's label moved for a
    third of them)."""
    if shift:
        move = (torch.arange(labels.numel(), device=labels.device) % 3) == 0
        labels = torch.where(move, (labels + shift) % nb, labels)
    count = torch.bincount(labels, minlength=nb)
    offsets = torch.cat([count.new_zeros(1), count.cumsum(0)])
    members = torch.sort(labels, stable=True).indices.int()
    if not probe:
        return offsets.cpu().numpy(), members.cpu().numpy(), torch.zeros((nb, 0), dtype=torch.int32).numpy()
    first = X[members[offsets[:-1].clamp(max=labels.numel() - 1)].long()].double()   # one row of each bucket
    dist = torch.cdist(first, first, compute_mode="donot_use_mm_for_euclid_dist")
    dist.fill_diagonal_(float("inf"))
    near = dist.topk(min(probe, nb - 1), largest=False).indices.int()
    return offsets.cpu().numpy(), members.cpu().numpy(), near.cpu().numpy()


def _inputs(c, seed):
    """(rows, the rest of a kNN case's inputs), from the seed alone."""
    g = _generator(seed)
    X, labels = _rows(c, c["n"], g)
    if c["kind"] == "knn_exact":
        return X, torch.randperm(c["n"], generator=g, device="cuda")[:c["nq"]].contiguous()
    return X, labels


def prepare(case, seed):
    c = dict(case)
    ctx = _ctx()
    kind = c["kind"]
    if kind == "search":
        X, _ = _rows(c, c["n"] + c["nq"], _generator(seed))
        X, Q = X[:c["n"]].contiguous(), X[c["n"]:].contiguous()
        M = 2 * c["degree"]
        graph = ctx.build_graph(X, n_buckets=max(4, c["n"] // 4000), M=M, K=c["degree"], metric=c["metric"],
                                return_knn=False).graph
        return {"case": c, "X": X, "Q": Q, "graph": graph}
    if kind == "knn_exact":
        X, q = _inputs(c, seed)
        return {"case": c, "X": X, "q": q}
    if kind == "knn_bucketed":
        X, labels = _inputs(c, seed)
        off, mem, pr = _bucketing(labels, c["clusters"], c["probe"], X)
        running = None
        if c["running"]:
            o2, m2, p2 = _bucketing(labels, c["clusters"], 0, X, shift=1)
            running = ctx.knn_bucketed(X, o2, m2, p2, c["M"], metric=c["metric"])
        return {"case": c, "X": X, "offsets": off, "members": mem, "probe": pr, "running": running}
    if kind == "optimize":
        # the kNN table of integer-valued rows, where no rounding decides an entry
        rows = {"n": c["n"], "d": 64, "dtype": "int", "data": "mixture", "clusters": max(16, c["n"] // 2000)}
        X, _ = _rows(rows, c["n"], _generator(seed))
        ids = ctx.build_graph(X, n_buckets=max(2, c["n"] // 4000), M=c["M"], K=c["K"], rounds=1, prune=False).knn_ids
        return {"case": c, "knn": ctx.sanitize(ids.cpu().numpy())}
    X, _ = _rows(c, c["n"], _generator(seed))
    return {"case": c, "X": X}


def run(state):
    c, ctx = state["case"], _ctx()
    kind = c["kind"]
    if kind == "search":
        ids, d, _ = ctx.search(state["X"], state["graph"], state["Q"], topk=c["topk"], ef=c["ef"], num_entry=4,
                               metric=c["metric"])
        return {"ids": ids, "dists": d}
    if kind == "knn_exact":
        ids, d = ctx.knn_exact(state["X"], c["k"], queries=state["q"], metric=c["metric"])
        return {"ids": ids, "dists": d}
    if kind == "knn_bucketed":
        ids, d = ctx.knn_bucketed(state["X"], state["offsets"], state["members"], state["probe"], c["M"],
                                  metric=c["metric"], running=state["running"])
        return {"ids": ids, "dists": d}
    if kind == "optimize":
        return ctx.optimize(state["knn"], c["K"]).view("int32")
    r = ctx.build_graph(state["X"], n_buckets=c["buckets"], M=c["M"], K=c["K"], metric=c["metric"],
                        refine_passes=c["refine"])
    return {"graph": r.graph, "ids": r.knn_ids, "dists": r.knn_dists}


def work(case):
    """Bytes: inputs once, outputs once (search: the rows and graph rows of a beam of ef points whose neighbours
    are new two times in three; optimize: every neighbour's row of every point, what counting detours reads).
    Operations: 2 d per (query, pool row) pair of the scans that the call asks for."""
    c = case
    esz = 1 if c.get("dtype") in ("u8", "i8") else 4
    if c["kind"] == "search":
        seen = c["nq"] * c["ef"] * c["degree"] * 2 / 3
        return {"bytes": seen * c["d"] * esz + c["nq"] * (c["ef"] * c["degree"] * 4 + c["d"] * esz + c["topk"] * 8),
                "flops": 3 * c["d"] * seen}
    if c["kind"] == "optimize":
        return {"bytes": c["n"] * (4 * c["M"] * c["M"] + 4 * c["K"]) + 28 * c["n"] * c["K"], "flops": 0}
    rows = c["n"] * c["d"] * esz
    if c["kind"] == "knn_exact":
        return {"bytes": rows + c["nq"] * c["k"] * 8, "flops": 2.0 * c["d"] * c["nq"] * c["n"]}
    if c["kind"] == "knn_bucketed":
        pool = c["n"] / c["clusters"] * (1 + c["probe"])
        return {"bytes": rows + c["n"] * c["M"] * 8 * (2 if c["running"] else 1), "flops": 2.0 * c["d"] * c["n"] * pool}
    pool = 2 * c["n"] / c["buckets"]          # own bucket and one probed bucket, two rounds
    return {"bytes": rows + c["n"] * (c["M"] * 8 + c["K"] * 4), "flops": 2.0 * c["d"] * 2 * c["n"] * pool}


def tolerance(case):
    c = case
    if c["kind"] == "optimize" or c["dtype"] != "f32":
        # integer rows: every distance, and every choice that hangs on one, is an exact whole number
        return "exact"
    # About four times what two correct results were seen to differ by.  Lists: the library against 64 bits (L2 by
    # the expanded form, whose error follows |q|^2 + |p|^2: rel 8.9e-6, max 3.3e-5, up to 0.5 % of the positions
    # swapped at near ties; IP 1.6e-7, 8e-7, 0.24 %).  Searches and builds: every input element moved by up to one
    # unit in the last place (searches 7.7e-8, 3e-7, none; builds: rows at a bucket's border change buckets, so a
    # few lists gain or lose far entries: up to 256 dimensions rel 1.1e-4 and 0.27 % of the entries, beyond 6.6e-4
    # and 1.4 %, of which 1 % is allowed).
    if c["kind"] == "search":
        return {"rel": 3e-7, "max": 1.2e-6, "differ": 0.002}
    if c["kind"] == "build":
        return {"rel": 2.6e-3 if c["d"] > 256 else 4.4e-4, "max": 0.9, "differ": 0.01}
    if c["metric"] == "ip":
        return {"rel": 6.4e-7, "max": 3.2e-6, "differ": 0.01}
    return {"rel": 3.6e-5, "max": 1.3e-4, "differ": 0.01}


def _top(key, ids, k):
    """The k smallest of each row of float64 keys, ascending by (key, id)."""
    v, i = key.topk(min(k, key.shape[1]), largest=False, sorted=True)
    return v, ids[i]


def _keys(Q, P, metric):
    """float64 keys (smaller is nearer)."""
    dot = Q @ P.T
    if metric == "ip":
        return -dot
    return (Q.square().sum(1)[:, None] + P.square().sum(1)[None]).sub_(dot, alpha=2.0).clamp_(min=0.0)


def _exact_rows(X, q, pool, k, metric):
    """The k nearest rows of `pool` (ids) to each of the rows q, itself excluded, in 64 bits."""
    Q = X[q].double()
    best_v = torch.full((q.numel(), k), float("inf"), dtype=torch.float64, device=X.device)
    best_i = torch.full((q.numel(), k), -1, dtype=torch.int64, device=X.device)
    step = max(1024, (1 << 28) // max(1, q.numel()))
    for s in range(0, pool.numel(), step):
        ids = pool[s:s + step]
        key = _keys(Q, X[ids].double(), metric)
        key.masked_fill_(q[:, None] == ids[None], float("inf"))
        v, i = _top(key, ids, k)
        best_v, best_i = torch.cat([best_v, v], 1), torch.cat([best_i, i], 1)
        best_v, order = best_v.topk(k, largest=False, sorted=True)
        best_i = best_i.gather(1, order)
    best_i = torch.where(torch.isinf(best_v), torch.full_like(best_i, -1), best_i)
    return best_i.int(), (best_v if metric == "l2" else -best_v)


def exact(case, seed):
    """The exact kNN lists in 64 bits; None where a result is no distance list, or an approximate one."""
    c = case
    if c["kind"] == "knn_exact" and float(c["n"]) * c["nq"] <= 2e10:
        X, q = _inputs(c, seed)
        ids, d = _exact_rows(X, q.long(), torch.arange(c["n"], device=X.device), c["k"], c["metric"])
        return {"ids": ids, "dists": d}
    if c["kind"] == "knn_bucketed" and not c["running"]:
        X, labels = _inputs(c, seed)
        off, mem, pr = _bucketing(labels, c["clusters"], c["probe"], X)
        mem = torch.from_numpy(mem).cuda().long()
        ids = torch.full((c["n"], c["M"]), -1, dtype=torch.int32, device="cuda")
        d = torch.full((c["n"], c["M"]), float("inf") if c["metric"] == "l2" else float("-inf"), dtype=torch.float64,
                       device="cuda")
        for b in range(c["clusters"]):
            q = mem[off[b]:off[b + 1]]
            pool = torch.cat([q] + [mem[off[p]:off[p + 1]] for p in pr[b].tolist()])
            i, v = _exact_rows(X, q, pool, c["M"], c["metric"])
            ids[q], d[q] = i, v
        return {"ids": ids, "dists": d}
    return None
