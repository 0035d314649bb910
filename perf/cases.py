"""What the performance of this framework is measured on: searches of a built index (the framework's main path) from a
single query to batches of 10,000, and whole index builds, each through the package's public entry points.

A search's state is an index and a batch of queries.  The index is what a program builds or loads once and keeps while
queries come and go, so a process makes each index once (from fixed data) and the queries come from the seed.  A build's
state is its dataset and a few queries, both from the seed; its pass is the build and one search of what it built.

Sizes and parameters come from bench.py's workloads (cpu100k, sift1m, deep100m, deep100m-host, gist1m) at row counts whose
index is built in seconds, and from the package's defaults.
"""

import collections

import numpy as np
import torch

import octex_amd

# Search points: the package's defaults, and bench.py's of each workload.
DEFAULT = dict(read=32, starts=128, waves=2, rerank=128, wave_rerank=128)
DEEP = dict(read=12, starts=64, waves=2, rerank=64, wave_rerank=64)
SIFT = dict(read=4, starts=16, waves=1, rerank=16, wave_rerank=16)
GIST = dict(read=32, starts=64, waves=3, rerank=512, wave_rerank=512)
SKETCH = dict(read=16, starts=128, waves=3, rerank=128, wave_rerank=128, sketch_rank=True, final_rerank=32)
LISTS = dict(read=32, starts=32, waves=0, rerank=64, wave_rerank=64)

# The indexes that searches run on: data (a mixture of `clusters` Gaussians, see _rows) and index parameters.  All use
# member lists, which bench.py's deep100m and gist1m use too and which build fastest.
BASE = dict(n=100_000, d=128, clusters=100, kind="gauss", copies=200, list_len=64, table_len=64, min_cell=1,
            sketch=128, log_buckets=16, exact_table=True, passes=3)
SIFT1M = dict(n=1_000_000, d=128, clusters=1000, kind="sift", copies=200, list_len=32, table_len=64, min_cell=1,
              sketch=128, log_buckets=20, exact_table=True, passes=3)
DEEP4M = dict(n=4_000_000, d=96, clusters=400, kind="deep", copies=120, list_len=64, table_len=64, min_cell=10,
              sketch=96, log_buckets=20, exact_table=False, passes=3)
HOST1M = dict(n=1_000_000, d=96, clusters=100, kind="deep", copies=120, list_len=16, table_len=32, min_cell=10,
              sketch=96, log_buckets=20, exact_table=False, passes=2, host=True)
EMBED = dict(n=200_000, d=384, clusters=200, kind="gist", copies=100, list_len=64, table_len=64, min_cell=4,
             sketch=128, log_buckets=18, exact_table=False, passes=2)


def _search(name, index, point, m, k=10, batch=10_000, numpy=False):
    return dict({"host": False}, **index, **point, what="search", name=name, m=m, k=k, batch=batch, numpy=numpy)


def _build(name, n, d, kind, lists, exact_table, copies, list_len=64, log_buckets=20, m=100, clusters=100):
    return dict(DEFAULT, what="build", name=name, n=n, d=d, kind=kind, clusters=clusters, lists=lists,
                exact_table=exact_table, copies=copies, list_len=list_len, table_len=64, min_cell=1, sketch=0,
                log_buckets=log_buckets, passes=3, m=m, k=10, batch=10_000)


def listed():
    return [
        # a service that answers one request at a time: the latency of one query
        _search("one_query", DEEP4M, DEEP, m=1),
        # a service that gathers a few requests
        _search("few_queries", BASE, DEFAULT, m=16),
        # a handful of requests on lists alone (no neighbor table rounds)
        _search("lists_only", SIFT1M, LISTS, m=300, k=20),
        # bench.py's cpu100k: the package's default search over 1,000 queries
        _search("default_1000", BASE, DEFAULT, m=1000),
        # bench.py's sift1m point: the largest batch at the lightest setting
        _search("sift_10000", SIFT1M, SIFT, m=10_000),
        # bench.py's default workload, deep100m's point, at 4M rows
        _search("deep_10000", DEEP4M, DEEP, m=10_000),
        # offline scoring from host arrays: numpy in and out, 100 neighbors, batches of 1,000 and a ragged last one
        _search("numpy_3333", DEEP4M, DEFAULT, m=3333, k=100, batch=1000, numpy=True),
        # long rows and a deep rerank: gist1m's point on rows of 384 (an embedding's width)
        _search("embed_1000", EMBED, GIST, m=1000),
        # deep100m-host: vectors in pinned host memory, ranked by sketch, the best reranked over the host link
        _search("host_10000", HOST1M, SKETCH, m=10_000),
        # the package's default build: IVF lists, exact neighbor table with reverse edges
        _build("build_default", n=20_000, d=64, kind="gauss", lists="ivf", exact_table=True, copies=100),
        # the fast build mode with an exact neighbor table
        _build("build_exact_table", n=150_000, d=128, kind="sift", lists="member", exact_table=True, copies=64,
               list_len=32, log_buckets=16),
        # the fast build mode as it is above exact_table_max rows: the table searched by the index itself
        _build("build_searched_table", n=250_000, d=96, kind="deep", lists="member", exact_table=False, copies=50,
               log_buckets=18),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    if rng.random() < 0.25:  # a build of another size
        d = 2 * _log(rng, 12, 80)
        return {k: v for k, v in _build("", n=_log(rng, 5_000, 60_000), d=d, kind=rng.choice(["gauss", "sift", "deep"]),
                                        lists=rng.choice(["ivf", "member", "exact"]), exact_table=rng.random() < 0.6,
                                        copies=_log(rng, 16, 60), list_len=rng.choice([16, 24, 32, 64]),
                                        log_buckets=rng.choice([12, 16, 18]), m=_log(rng, 20, 400),
                                        clusters=rng.choice([20, 50, 100])).items() if k != "name"}
    if rng.random() < 0.35:  # a search of a small index of odd dimensions
        d = 2 * _log(rng, 10, 150)
        index = dict(n=_log(rng, 8_000, 120_000), d=d, clusters=rng.choice([10, 40, 150]), copies=_log(rng, 16, 120),
                     kind=rng.choice(["gauss", "sift", "deep"]), list_len=rng.choice([16, 20, 32, 64]),
                     table_len=rng.choice([24, 32, 64]), min_cell=rng.choice([1, 2, 10]), sketch=0,
                     log_buckets=rng.choice([12, 14, 16]), exact_table=rng.random() < 0.5, passes=2)
    else:
        index = rng.choice([BASE, SIFT1M, DEEP4M, HOST1M, EMBED])
    ranked = index.get("host", False) or rng.random() < 0.1
    waves = rng.choice([0, 1, 1, 2, 2, 3])
    starts = _log(rng, 12, 128)
    point = dict(read=min(_log(rng, 4, 64), index["list_len"]), starts=starts, waves=waves, rerank=_log(rng, 16, 256),
                 wave_rerank=_log(rng, 16, 256))
    k = _log(rng, 1, min(100, max(starts, 16)))
    if ranked:
        point.update(sketch_rank=True, final_rerank=min(max(k, _log(rng, 16, 64)), max(starts, k)))
    m = _log(rng, 1, 10_000)
    # the entries a batch gathers, held under those of the largest listed case
    while m > 1 and m * (index["copies"] * point["read"] + waves * starts * index["table_len"]) > 90_000_000:
        m = (m + 1) // 2
    case = _search("", index, point, m=m, k=k, batch=rng.choice([10_000, 10_000, max(1, m // 3)]),
                   numpy=rng.random() < 0.2)
    del case["name"]
    return case


# ---------------------------------------------------------------------------------------------------- data and states


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _mixture(case, seed):
    """The cluster centers of a case's data."""
    g, c, d = _gen(7919 + seed), case["clusters"], case["d"]
    if case["kind"] == "sift":
        return 128 * torch.rand((c, d), generator=g, device="cuda")
    if case["kind"] == "gist":
        return 0.1 * torch.rand((c, d), generator=g, device="cuda")
    return torch.randn((c, d), generator=g, device="cuda")


def _rows(case, centers, n, g):
    """n rows of the mixture, as bench.py's workloads draw them: "gauss" around N(0, 1) centers, "deep" the same
    L2-normalized, "sift" rounded to 0..255, "gist" non-negative features."""
    out = torch.empty((n, case["d"]), device="cuda")
    for a in range(0, n, 1 << 18):
        b = min(n, a + (1 << 18))
        x = centers[torch.randint(0, len(centers), (b - a,), generator=g, device="cuda")]
        e = torch.randn(x.shape, generator=g, device="cuda")
        if case["kind"] == "sift":
            x = (x + 12 * e).clamp_(0, 255).round_()
        elif case["kind"] == "gist":
            x = x + (0.05 * e).abs_()
        elif case["kind"] == "deep":
            x = x + 0.4 * e
            x = x / x.norm(dim=1, keepdim=True)
        else:
            x = x + 0.3 * e
        out[a:b] = x
    return out


_DATA = ("kind", "n", "d", "clusters")
_INDEX = _DATA + ("copies", "list_len", "table_len", "min_cell", "sketch", "log_buckets", "exact_table", "passes", "host")
_POINT = ("read", "starts", "waves", "rerank", "wave_rerank", "batch", "sketch_rank", "final_rerank")
_kept = collections.OrderedDict()  # the indexes of this process, the last used ones


def _params(case):
    return dict(copies=case["copies"], list_len=case["list_len"], table_len=case["table_len"],
                min_cell=case["min_cell"], sketch_width=case["sketch"], log_buckets=case["log_buckets"],
                table_passes=case["passes"], exact_table_max=1_000_000 if case["exact_table"] else 0, seed=0,
                member_lists=case.get("lists", "member") == "member", exact_lists=case.get("lists") == "exact")


def _index(case):
    """The index of a search case over its fixed data, made the first time a process asks for it."""
    key = tuple(case[f] for f in _INDEX)
    if key not in _kept:
        while len(_kept) >= 6:
            _kept.popitem(last=False)
        x = _rows(case, _mixture(case, 0), case["n"], _gen(1)).half()
        torch.cuda.synchronize()  # a build does not wait for its dataset's producer
        index, _ = octex_amd.build_in_memory(x, **_params(case))
        if case["host"]:
            index.place_on_host(vectors=True)
        _kept[key] = index
    _kept.move_to_end(key)
    return _kept[key]


def _point(case):
    return {f: case[f] for f in _POINT if f in case}


def prepare(case, seed):
    if case["what"] == "build":
        centers, g = _mixture(case, seed), _gen(2 * seed + 10)
        x = _rows(case, centers, case["n"], g).half()
        return dict(build=_params(case), x=x, q=_rows(case, centers, case["m"], g), k=case["k"], point=_point(case))
    q = _rows(case, _mixture(case, 0), case["m"], _gen(2 * seed + 10))
    return dict(index=_index(case), q=q.cpu().numpy() if case["numpy"] else q, k=case["k"], point=_point(case))


def run(state):
    if "build" in state:
        index, _ = octex_amd.build_in_memory(state["x"], **state["build"])
        distances, ids = index.search(state["q"], k=state["k"], **state["point"])
        return distances, ids, index.array("table", np.int32)
    distances, ids = state["index"].search(state["q"], k=state["k"], **state["point"])
    return distances, ids


# ------------------------------------------------------------------------------------------------ what a pass is held to


def _sketch_width(case):
    return case["sketch"] or max(min(case["d"] // 16 * 16, 128), min(case["d"], 16))


def _search_work(case):
    """Per query: its projections (32 of each copy), the list entries it reads and, per wave, the table rows of its start
    points, a sketch row of each distinct id among them (taken as half of the entries, and an id of an earlier round is
    not scored again), and its reranked vectors.  No array is read more than once in whole."""
    n, d, m, C, S = case["n"], case["d"], case["m"], case["copies"], _sketch_width(case)
    lists = C * min(case["read"], case["list_len"])
    table = case["starts"] * case["table_len"] * min(1, case["waves"])
    rows = min(n, (lists + table) / 2)  # distinct ids of a query
    exact = case.get("final_rerank", 32) if case.get("sketch_rank") else case["rerank"] + case["wave_rerank"] * case["waves"]
    exact = min(exact, rows)
    flops = m * (2.0 * d * (32 * C + S) + 3.0 * S * rows + 3.0 * d * exact)
    reads = 4.0 * m * (d + lists) + 64.0 * C * d + 16.0 * m * C  # queries, list entries, projections, a bucket a copy
    reads += 4.0 * min(m * table, n * case["table_len"]) + min(m * rows, n) * S + 2.0 * min(m * exact, n) * d
    return {"bytes": reads + 12.0 * m * case["k"], "flops": flops}


def work(case):
    w = _search_work(case)
    if case["what"] == "build":
        n, d, C, l = case["n"], case["d"], case["copies"], case["list_len"]
        w["flops"] += 2.0 * n * d * (32 * C + _sketch_width(case))  # every copy's projections, the sketch
        if case["lists"] == "ivf":  # 20 rounds of k-means over half the rows, 4 sqrt(n) centers
            w["flops"] += C * 20 * 2.0 * (n / 2) * 4 * n**0.5 * 32
        if case["exact_table"]:
            w["flops"] += 2.0 * n * n * d
        else:  # every row searched in each pass
            w["flops"] += case["passes"] * n * 3.0 * _sketch_width(case) * C * min(64, l) / 2
        # the rows, the lists of about one cell a row, its key, the sketch and the table
        w["bytes"] += n * (2.0 * d + C * (4.0 * l + 8) + _sketch_width(case) + 4.0 * case["table_len"])
    return w


def tolerance(case):
    """Distances are 32-bit sums.  Ids swap where distances nearly tie: queries changed by half a 32-bit rounding (as sums
    in another order change the projections) left distances within 1.3e-7 and changed 0.33 % of the ids at most on
    integer-valued rows (0.18 % over 10,000 queries), 0.02 % on the others; a handful of queries may hold a swap or two."""
    ids = 0.015 if case["kind"] == "sift" else 0.001
    return {"rel": 1e-5, "differ": min(0.99, max(ids, 2.5 / (case["m"] * case["k"])))}


def exact(case, seed):
    """The true nearest neighbors' distances in 64 bits, by brute force over the stored (fp16) rows: what the search
    approximates, so its misses show here.  Ids and neighbor tables have no such value (ties, approximate tables)."""
    if case["what"] == "build":
        centers, g = _mixture(case, seed), _gen(2 * seed + 10)
        x = _rows(case, centers, case["n"], g).half()
        q = _rows(case, centers, case["m"], g)
    else:
        x = _rows(case, _mixture(case, 0), case["n"], _gen(1)).half()
        q = _rows(case, _mixture(case, 0), case["m"], _gen(2 * seed + 10))
    k, q = case["k"], q.double()
    best = torch.full((len(q), k), float("inf"), dtype=torch.float64, device="cuda")
    qq = (q * q).sum(1, keepdim=True)
    for a in range(0, len(x), 1 << 16):
        b = x[a : a + (1 << 16)].double()
        dist = torch.addmm((b * b).sum(1)[None, :] + qq, q, b.T, alpha=-2)
        best = torch.cat([best, dist.topk(min(k, len(b)), dim=1, largest=False).values], 1)
        best = best.topk(k, dim=1, largest=False).values
    best = best.sort(1).values.clamp_(min=0)
    out = best.cpu().numpy() if case.get("numpy") else best
    return (out, None, None) if case["what"] == "build" else (out, None)
