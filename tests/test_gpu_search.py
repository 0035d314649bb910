"""The whole search on the GPU through the cuvsOctex* C ABI, against the CPU oracle on the same index and queries.

Parity: given the GPU's own projections Y and sketch queries qs (read back from the search plan), the oracle's
search returns the same ids and bit-identical distances; against exact search, recall thresholds of the
reference's tests (test_build.py:48-54, octex_c.cu:196).  Batch splitting / padding, graph replay, device tensors,
sketch-rank mode and the parameter limits are covered too."""

import ctypes as ct

import numpy as np
import pytest
from conftest import exact_knn, recall

from oracle import oracle as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def octex():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import octex_amd

    return octex_amd


PARAMS = dict(read=32, starts=64, waves=2, rerank=64, wave_rerank=64)


def oracle_given_gpu_projections(index, oix, Q, k, **params):
    """The oracle's search fed with the GPU plan's Y and qs of the last (single) batch."""
    info = index.plan_info()
    assert info["m"] == len(Q)
    C, w, S = oix.copies, oix.width, oix.sketch_width
    Y = index.plan_buffer("Y", np.uint16)[: len(Q) * C * w].reshape(len(Q), C * w)
    qs = index.plan_buffer("qs", np.float32)[: len(Q) * S].reshape(len(Q), S)
    D, I, tr = O.search(oix, Q, k=k, Y=Y, qs=qs, trace=True, **params)
    return D, I, tr, Y, qs


def assert_same_results(D, I, D2, I2):
    """Identical ids and distances, except where distances tie (then the ids at the tie may swap)."""
    assert np.array_equal(D, D2), "distances differ"
    diff = I != I2
    if diff.any():
        for q, j in zip(*np.nonzero(diff)):
            assert (D[q] == D[q, j]).sum() > 1, f"query {q} rank {j}: ids differ without a distance tie"


def test_search_matches_oracle(octex, small_index):
    index = octex.load(small_index["path"])
    oix = O.Index(small_index["path"])
    Q = small_index["Q"]
    D, I = index.search(Q, k=10, **PARAMS)
    Do, Io, tr, Y, qs = oracle_given_gpu_projections(index, oix, Q, 10, **PARAMS)
    assert_same_results(D, I, Do, Io)
    # stage by stage: probe segments, first-round candidate counts, the final kept list
    seg = index.plan_buffer("seg", np.int32)[: len(Q) * oix.copies * 2].reshape(len(Q), oix.copies, 2)
    assert np.array_equal(seg, tr["seg"])
    nin = index.plan_buffer("nin", np.int32)[: len(Q)]
    assert np.array_equal(nin, tr["n1"])
    KO = max(PARAMS["starts"], 10)
    sd = index.plan_buffer("sd", np.float32)[: len(Q) * KO].reshape(len(Q), KO)
    assert np.array_equal(sd, tr["sd"])
    # the projections themselves against the fp64 oracle: within one fp16 ulp
    qc, qh = O.center(Q, oix.mean)
    from test_gpu_stages import check_projection

    check_projection(Y, qh, oix.ucat, oix.shift)
    assert np.allclose(qs, O.sketch_query(qc, oix.basis), rtol=1e-5, atol=1e-4)


@pytest.mark.parametrize("sketch_rank", [False, True])
def test_large_wave_gather_matches_oracle(octex, small_index, sketch_rank):
    """starts 512 over table rows of 32 (configs[4]'s setting): the wave gather's hash set of 2^15 slots leaves
    no LDS for the candidates' slot list, which then lives in the query's row of cand; results as the oracle's."""
    index = octex.load(small_index["path"])
    oix = O.Index(small_index["path"])
    Q = small_index["Q"]
    assert oix.table_len == 32
    p = dict(read=16, starts=512, waves=2, rerank=128, wave_rerank=128, sketch_rank=sketch_rank, final_rerank=32)
    D, I = index.search(Q, k=10, **p)
    assert index.plan_info()["W2"] == 1 << 15
    Do, Io, tr, _, _ = oracle_given_gpu_projections(index, oix, Q, 10, **p)
    assert_same_results(D, I, Do, Io)


def test_search_recall_and_distances(octex, small_index):
    index = octex.load(small_index["path"])
    Q = small_index["Q"]
    D, I = index.search(Q, k=10, **PARAMS)
    assert recall(I, small_index["gt"]) >= 0.95
    Xh = small_index["X"].astype(np.float16).astype(np.float64)
    exact = ((Xh[I] - Q[:, None, :].astype(np.float64)) ** 2).sum(-1)
    assert np.allclose(D, exact, rtol=1e-3)
    assert (np.diff(D, axis=1) >= 0).all()


def test_batch_split_and_padding(octex, small_index):
    """Results do not depend on the batch size: batches of 37 (last one padded) equal one batch."""
    index = octex.load(small_index["path"])
    Q = small_index["Q"]
    D1, I1 = index.search(Q, k=10, batch=1000, **PARAMS)
    D2, I2 = index.search(Q, k=10, batch=37, **PARAMS)
    assert np.array_equal(I1, I2) and np.array_equal(D1, D2)


@pytest.mark.parametrize("batch,use_graph", [(37, True), (1000, True), (37, False)])
@pytest.mark.parametrize("sketch_rank", [False, True])
def test_results_written_in_place(octex, small_index, batch, use_graph, sketch_rank):
    """Device queries are read and their results written in place by a batch's first and last kernel, the last batch's
    only as far as it has queries: rows of larger tensors, through the C ABI, with nothing around them touched."""
    import ctypes as ct

    from octex_amd import _lib
    from octex_amd.index import search_params

    index = octex.load(small_index["path"])
    Q = small_index["Q"][:100]
    p = dict(PARAMS, batch=batch, use_graph=use_graph, sketch_rank=sketch_rank, final_rerank=32)
    D1, I1 = index.search(Q, k=10, **p)
    m = len(Q)
    q = torch.full((m + 2, Q.shape[1]), float("nan"), device="cuda")
    q[1:-1] = torch.from_numpy(Q).cuda()
    I = torch.full((m + 2, 10), -9, dtype=torch.int64, device="cuda")
    D = torch.full((m + 2, 10), -9.0, device="cuda")
    res, sp = _lib.Resources(stream=0), search_params(**p)
    t = [_lib.Dl(x[1:-1]) for x in (q, I, D)]
    _lib.call("cuvsOctexSearch", res.h, ct.byref(sp), index._handle, *(x.ptr for x in t))
    assert np.array_equal(I[1:-1].cpu().numpy(), I1) and np.array_equal(D[1:-1].cpu().numpy(), D1)
    assert (I[[0, -1]] == -9).all() and (D[[0, -1]] == -9).all()


def test_graph_equals_direct_launches(octex, small_index):
    index = octex.load(small_index["path"])
    Q = small_index["Q"]
    D1, I1 = index.search(Q, k=10, **PARAMS)
    assert index.plan_info()["graph"] == 1
    D2, I2 = index.search(Q, k=10, use_graph=False, **PARAMS)
    assert index.plan_info()["graph"] == 0
    assert np.array_equal(I1, I2) and np.array_equal(D1, D2)
    for _ in range(3):  # replays of one graph, with eager work in between
        D3, I3 = index.search(Q, k=10, **PARAMS)
        assert np.array_equal(I1, I3) and np.array_equal(D1, D3)


def test_concurrent_searches(octex, small_index):
    """Threads searching one index with different parameter sets (each call evicts the other's cached plan,
    search.cu:804-813, while that plan's batch may still run) get the results of serial searches."""
    import threading

    index = octex.load(small_index["path"])
    Q = small_index["Q"]
    sets = [dict(k=10, **PARAMS), dict(k=5, read=8, starts=32, waves=1), dict(k=10, batch=37, **PARAMS)]
    want = [index.search(Q, **p) for p in sets]
    errors = []

    def worker(t):
        try:
            for r in range(6):
                j = (t + r) % len(sets)
                D, I = index.search(Q, **sets[j])
                if not (np.array_equal(I, want[j][1]) and np.array_equal(D, want[j][0])):
                    errors.append((t, r, j))
        except Exception as e:  # noqa: BLE001 - reported below
            errors.append((t, repr(e)))

    threads = [threading.Thread(target=worker, args=(t,)) for t in range(3)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    assert not errors, errors


class _Foreign:
    """An array of a framework octex_amd does not know, exporting DLPack only (as CuPy's arrays do)."""

    __module__ = "fakearrays"

    def __init__(self, t):
        self.t = t

    def __dlpack__(self, **kw):
        return self.t.__dlpack__(**kw)

    def __dlpack_device__(self):
        return self.t.__dlpack_device__()


def test_foreign_arrays(octex, small_index, monkeypatch):
    """Queries of another framework are searched without a copy and answered in that framework (through its
    module's from_dlpack, octex/_arrays.py); given output arrays of it are written (int32 ids too)."""
    import sys
    import types

    mod = types.ModuleType("fakearrays")
    mod.from_dlpack = lambda x: _Foreign(torch.from_dlpack(x))
    monkeypatch.setitem(sys.modules, "fakearrays", mod)
    index = octex.load(small_index["path"])
    Q = small_index["Q"]
    D1, I1 = index.search(Q, k=10, **PARAMS)
    q = _Foreign(torch.from_numpy(Q).cuda())
    D2, I2 = index.search(q, k=10, **PARAMS)
    assert isinstance(D2, _Foreign) and isinstance(I2, _Foreign) and I2.t.is_cuda
    assert np.array_equal(I1, I2.t.cpu().numpy()) and np.array_equal(D1, D2.t.cpu().numpy())
    nb = _Foreign(torch.empty((len(Q), 10), dtype=torch.int32, device="cuda"))
    ds = _Foreign(torch.empty((len(Q), 10), dtype=torch.float32, device="cuda"))
    D3, I3 = index.search(q, k=10, neighbors=nb, distances=ds, **PARAMS)
    assert I3 is nb and D3 is ds
    assert np.array_equal(nb.t.cpu().numpy(), I1) and np.array_equal(ds.t.cpu().numpy(), D1)
    host_ids = np.empty((len(Q), 10), np.uint32)  # numpy outputs of device queries
    index.search(torch.from_numpy(Q).cuda(), k=10, neighbors=host_ids, **PARAMS)
    assert np.array_equal(host_ids, I1)


def test_device_tensors(octex, small_index):
    index = octex.load(small_index["path"])
    Q = small_index["Q"]
    D1, I1 = index.search(Q, k=10, **PARAMS)
    D2, I2 = index.search(torch.from_numpy(Q).cuda(), k=10, **PARAMS)
    assert D2.is_cuda and I2.dtype == torch.int64
    assert np.array_equal(I1, I2.cpu().numpy()) and np.array_equal(D1, D2.cpu().numpy())


def test_search_on_a_side_stream(octex, small_index):
    """Device queries written on a torch side stream (after long work on it) are searched on that stream: the
    search waits for them, and its results are ready on that stream, as a serial host search's."""
    index = octex.load(small_index["path"])
    Q = small_index["Q"]
    D1, I1 = index.search(Q, k=10, **PARAMS)
    side = torch.cuda.Stream()  # default priority
    with torch.cuda.stream(side):
        q = torch.zeros(Q.shape, dtype=torch.float32, device="cuda")
        src = torch.from_numpy(Q).cuda()
        a = torch.randn((4096, 4096), device="cuda")
        for _ in range(12):  # keeps the side stream busy before the queries are written
            a = torch.mm(a, a) * 1e-3
        q.copy_(src + a[:1, :1] * 0)
        D2, I2 = index.search(q, k=10, **PARAMS)
        D2, I2 = D2.cpu().numpy(), I2.cpu().numpy()
    assert np.array_equal(I1, I2) and np.array_equal(D1, D2)
    torch.cuda.synchronize()


@pytest.mark.parametrize("starts,waves,k", [(128, 4, 10), (100, 3, 100), (16, 6, 1), (256, 2, 20), (20, 1, 50)])
@pytest.mark.parametrize("sketch_rank", [False, True])
def test_start_points_of_the_kept_list_kernels(octex, small_index, starts, waves, k, sketch_rank):
    """Start points taken by the kept-list kernels (up to 256 ids expanded before) and by their own kernel (more: four
    waves of 128), and the results taken from the last kept list: as the oracle's, and as the sorts in global memory."""
    index = octex.load(small_index["path"])
    oix = O.Index(small_index["path"])
    Q = small_index["Q"][:90]
    p = dict(read=16, starts=starts, waves=waves, rerank=96, wave_rerank=64, sketch_rank=sketch_rank,
             final_rerank=max(k, 32))
    if sketch_rank and p["final_rerank"] > max(starts, k):
        p["final_rerank"] = k
    D, I = index.search(Q, k=k, **p)
    Do, Io, _, _, _ = oracle_given_gpu_projections(index, oix, Q, k, **p)
    assert_same_results(D, I, Do, Io)
    Du, Iu = index.search(Q, k=k, fused_merge=False, **p)
    assert_same_results(D, I, Du, Iu)


def test_searches_alternating_between_streams(octex, small_index):
    """Searches enqueued on several streams in turn, without waiting, share one plan's buffers (and replace the plan,
    with another parameter set in between): each waits for the one before, whatever its stream."""
    index = octex.load(small_index["path"])
    Q = torch.from_numpy(small_index["Q"]).cuda()
    parts = [Q[:200].contiguous(), Q[200:400].contiguous(), Q[100:300].contiguous()]
    sets = [dict(k=10, **PARAMS), dict(k=5, read=8, starts=32, waves=1)]
    want = [[index.search(x, **p) for x in parts] for p in sets]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream(), torch.cuda.default_stream()]
    got = []
    for r in range(24):
        j = 1 if r % 8 == 7 else 0
        with torch.cuda.stream(streams[r % 3]):
            got.append((j, (r // 3) % 3, index.search(parts[(r // 3) % 3], **sets[j])))
    torch.cuda.synchronize()
    for j, i, (D, I) in got:
        assert torch.equal(I, want[j][i][1]) and torch.equal(D, want[j][i][0])


def test_sketch_rank_matches_oracle(octex, small_index):
    index = octex.load(small_index["path"])
    oix = O.Index(small_index["path"])
    Q = small_index["Q"]
    p = dict(read=16, starts=96, waves=2, sketch_rank=True, final_rerank=48)
    D, I = index.search(Q, k=10, **p)
    Do, Io, _, _, _ = oracle_given_gpu_projections(index, oix, Q, 10, **p)
    assert_same_results(D, I, Do, Io)
    p0 = dict(p, final_rerank=0)  # sketch order, sketch distances out
    D, I = index.search(Q, k=10, **p0)
    Do, Io, _, _, _ = oracle_given_gpu_projections(index, oix, Q, 10, **p0)
    assert_same_results(D, I, Do, Io)


def test_waves_zero_and_k_above_starts(octex, small_index):
    index = octex.load(small_index["path"])
    oix = O.Index(small_index["path"])
    Q = small_index["Q"][:50]
    for p, k in ((dict(read=8, starts=32, waves=0), 10), (dict(read=32, starts=8, waves=1), 20)):
        D, I = index.search(Q, k=k, **p)
        Do, Io, _, _, _ = oracle_given_gpu_projections(index, oix, Q, k, **p)
        assert_same_results(D, I, Do, Io)


def test_wide_index_matches_oracle(octex, wide_index):
    """Sketch width 96 (8 lanes per candidate, two of them idle), 3 blocks, dimension 96."""
    index = octex.load(wide_index["path"])
    oix = O.Index(wide_index["path"])
    Q = wide_index["Q"]
    D, I = index.search(Q, k=10, **PARAMS)
    Do, Io, _, _, _ = oracle_given_gpu_projections(index, oix, Q, 10, **PARAMS)
    assert_same_results(D, I, Do, Io)
    gt, _ = exact_knn(wide_index["X"].astype(np.float16).astype(np.float32), Q)
    assert recall(I, gt) >= 0.9


def test_load_limits_match_oracle(octex, small_index):
    index = octex.load(small_index["path"], copies_limit=5, list_limit=8)
    assert index.copies == 5
    oix = O.Index(small_index["path"], copies_limit=5, list_limit=8)
    Q = small_index["Q"][:40]
    D, I = index.search(Q, k=10, **PARAMS)
    Do, Io, _, _, _ = oracle_given_gpu_projections(index, oix, Q, 10, **PARAMS)
    assert_same_results(D, I, Do, Io)


def test_probe_without_bucket_lines(octex, small_index, monkeypatch):
    """The search's probe reads each bucket's line (first key and key range) when the index has its bucket lines,
    the offsets and keys otherwise (OCTEX_PROBE_LINES=0 at load): the same segments and results, and the lines are
    C L 2^log_buckets 16-byte entries of device memory."""
    oix = O.Index(small_index["path"])
    Q = small_index["Q"][:60]
    a = octex.load(small_index["path"])
    Da, Ia = a.search(Q, k=10, **PARAMS)
    seg_a = a.plan_buffer("seg", np.int32)[: len(Q) * oix.copies * 2].copy()
    monkeypatch.setenv("OCTEX_PROBE_LINES", "0")
    b = octex.load(small_index["path"])
    Db, Ib = b.search(Q, k=10, **PARAMS)
    seg_b = b.plan_buffer("seg", np.int32)[: len(Q) * oix.copies * 2]
    assert np.array_equal(seg_a, seg_b) and np.array_equal(Ia, Ib) and np.array_equal(Da, Db)
    lines = oix.copies * len(oix.spacings) * 2**oix.log_buckets * 16
    assert a.device_bytes[0] - b.device_bytes[0] == lines


@pytest.mark.parametrize("mode", ["1", "prev", "all"])
def test_wave_gathers_with_and_without_earlier_scores(octex, small_index, monkeypatch, mode):
    """The first wave's gather takes the scores of candidates found in the first round's row; with prev every wave from
    the previous round's row, with all the later waves also from the first round's.  With OCTEX_GATHER_REUSE=0 (read
    when a plan is made) they score every candidate: the same results, and the profile counts the candidates found
    (three waves)."""
    Q = small_index["Q"][:60]
    params = dict(PARAMS, waves=3)
    monkeypatch.setenv("OCTEX_GATHER_REUSE", mode)
    a = octex.load(small_index["path"])
    Da, Ia = a.search(Q, k=10, **params)
    _, cnt = a.profile_batch(Q, k=10, reps=1, **params)
    monkeypatch.setenv("OCTEX_GATHER_REUSE", "0")
    b = octex.load(small_index["path"])
    Db, Ib = b.search(Q, k=10, **params)
    _, cnt0 = b.profile_batch(Q, k=10, reps=1, **params)
    assert np.array_equal(Ia, Ib) and np.array_equal(Da, Db)
    used = 3 if mode != "1" else 1  # the waves that read earlier rows
    assert all(k > 0 for k in cnt["known2"][:used]) and all(o > 0 for o in cnt["oldread2"][:used])
    assert sum(cnt["known2"][used:]) == 0 and sum(cnt["oldread2"][used:]) == 0
    assert sum(cnt0["known2"]) == 0 and sum(cnt0["oldread2"]) == 0
    assert cnt["distinct2"][:3] == cnt0["distinct2"][:3]


def test_placements_on_host(octex, small_index):
    """Vectors, table and sketch in pinned host memory give the same results."""
    Q = small_index["Q"][:40]
    D1, I1 = octex.load(small_index["path"]).search(Q, k=10, **PARAMS)
    index = octex.load(small_index["path"], vectors_on_host=True, table_on_host=True, sketch="host")
    D2, I2 = index.search(Q, k=10, **PARAMS)
    assert np.array_equal(I1, I2) and np.array_equal(D1, D2)


def test_errors(octex, small_index):
    from octex_amd._lib import OctexError

    index = octex.load(small_index["path"])
    Q = small_index["Q"][:4]
    with pytest.raises(ValueError, match="dimension"):
        index.search(Q[:, :10], k=10)
    with pytest.raises(OctexError, match="max\\(starts, k\\) must be <= 512"):
        index.search(Q, k=10, starts=600)
    with pytest.raises(OctexError, match="read, starts >= 1"):
        index.search(Q, k=10, read=0)
    with pytest.raises(FileNotFoundError):
        octex.load(small_index["path"] + "_missing")
    assert index.size == 4000 and index.dim == 64 and index.copies == 16 and len(index.devices) == 1
    assert index.device_bytes[0] > 0


def hip_runtime():
    """The HIP runtime that this process has loaded."""
    return ct.CDLL(next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line))


@pytest.mark.parametrize("mode", [0, 1, 2])  # global, thread-local, relaxed
def test_null_stream_search_while_a_blocking_stream_is_captured(octex, small_index, mode):
    """The null stream takes no launch while a blocking stream is being captured: searches on it run on the index's
    stream then, with the same results (host and device queries), and their work does not enter the capture."""
    index = octex.load(small_index["path"])
    Q = small_index["Q"][:40]
    q = torch.from_numpy(Q).cuda()
    D0, I0 = index.search(Q, k=10, **PARAMS)
    torch.cuda.synchronize()
    hip = hip_runtime()
    stream, graph, nodes = ct.c_void_p(), ct.c_void_p(), ct.c_size_t(99)
    assert hip.hipStreamCreate(ct.byref(stream)) == 0
    assert hip.hipStreamBeginCapture(stream, ct.c_int(mode)) == 0
    try:
        found = [index.search(Q, k=10, **PARAMS), index.search(q, k=10, **PARAMS)]
    finally:
        assert hip.hipStreamEndCapture(stream, ct.byref(graph)) == 0
    assert hip.hipGraphGetNodes(graph, None, ct.byref(nodes)) == 0 and nodes.value == 0
    assert hip.hipGraphDestroy(graph) == 0 and hip.hipStreamDestroy(stream) == 0
    torch.cuda.synchronize()
    for D, I in found + [index.search(Q, k=10, **PARAMS)]:
        assert np.array_equal(I0, np.asarray(torch.as_tensor(I).cpu()))
        assert np.array_equal(D0, np.asarray(torch.as_tensor(D).cpu()))


def search_into(index, q, I, D, stream, **params):
    """cuvsOctexSearch of device queries on `stream` into I and D."""
    from octex_amd import _lib
    from octex_amd import index as octex_index

    res = _lib.Resources(stream=stream.cuda_stream)
    tensors = [_lib.Dl(t) for t in (q, I, D)]
    _lib.call("cuvsOctexSearch", res.h, ct.byref(octex_index.search_params(**params)), index.handle,
              *(t.ptr for t in tensors))


@pytest.mark.parametrize("extra", [dict(use_graph=False), dict(use_graph=True), dict(batch=17),
                                   dict(sketch_rank=True, final_rerank=32), dict(waves=0)])
def test_captured_search_replays(octex, small_index, extra):
    """Two searches captured into one graph, on the captured stream and on one forked from it: every replay gives the
    eager results of the queries then in place, beside eager searches of the same shape on another stream and after a
    plan of another shape replaced the cached one."""
    index = octex.load(small_index["path"])
    params = dict(PARAMS, **extra)
    Q = small_index["Q"][:40]
    q, side, fork = [torch.from_numpy(Q).cuda() for _ in range(2)], torch.cuda.Stream(), torch.cuda.Stream()
    I = [torch.full((40, 10), -7, dtype=torch.int64, device="cuda") for _ in range(2)]
    D = [torch.full((40, 10), float("nan"), device="cuda") for _ in range(2)]
    index.search(q[0], k=10, **params)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        fork.wait_stream(side)
        search_into(index, q[0], I[0], D[0], side, **params)
        search_into(index, q[1], I[1], D[1], fork, **params)
        side.wait_stream(fork)
    assert index.plan_info()["m"] == min(40, params.get("batch", 40))  # the captured plan's
    torch.cuda.synchronize()
    g = np.random.default_rng(1)
    for rep in range(4):
        Qr = [np.ascontiguousarray(Q[g.permutation(40)]) for _ in range(2)]
        want = [index.search(x, k=10, **params) for x in Qr]
        for t, x in zip(q, Qr):
            t.copy_(torch.from_numpy(x))
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            graph.replay()
        Ds, Is = index.search(q[0], k=10, **params)  # on the null stream, beside the replay
        index.search(Q[:7], k=5, **PARAMS)           # another plan takes its place in the cache
        torch.cuda.synchronize()
        print(f"replay {rep}", flush=True)
        for (Dw, Iw), Dg, Ig in zip(want + want[:1], D + [Ds], I + [Is]):
            assert np.array_equal(Iw, Ig.cpu().numpy()) and np.array_equal(Dw, Dg.cpu().numpy())


@pytest.mark.parametrize("mode", ["global", "thread_local", "relaxed"])
@pytest.mark.parametrize("searched", [False, True])
def test_captured_search_without_an_earlier_one(octex, small_index, mode, searched):
    """A search captured without an earlier one of its shape, as the index's first search or after others: its buffers
    are allocated beside the capture, which goes on, and every replay gives the eager results."""
    index = octex.load(small_index["path"])
    Q = small_index["Q"][:40]
    if searched:
        index.search(Q[:5], k=10, **PARAMS)
    q, side = torch.from_numpy(Q).cuda(), torch.cuda.Stream()
    I, D = torch.zeros((40, 10), dtype=torch.int64, device="cuda"), torch.ones((40, 10), device="cuda")
    other = torch.ones(100, device="cuda")
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    print(f"capture mode {mode}, searched {searched}", flush=True)
    with torch.cuda.graph(graph, stream=side, capture_error_mode=mode):
        other.mul_(2)
        search_into(index, q, I, D, side, **PARAMS)
        other.add_(1)
    for rep in range(3):
        Qr = np.ascontiguousarray(np.roll(Q, rep, axis=0))
        q.copy_(torch.from_numpy(Qr))
        Dw, Iw = index.search(Qr, k=10, **PARAMS)
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(Iw, I.cpu().numpy()) and np.array_equal(Dw, D.cpu().numpy())
    assert (other == 2 ** 3 + 2**2 + 2 + 1).all()


def test_plan_buffers_read_behind_a_running_search(octex, small_index):
    """A plan buffer copied to the host while a search on another stream still runs holds that search's results."""
    index = octex.load(small_index["path"])
    Q = np.concatenate([small_index["Q"]] * 40)
    q, side = torch.from_numpy(Q).cuda(), torch.cuda.Stream()
    g = torch.Generator().manual_seed(0)
    for _ in range(5):
        q.copy_(q[torch.randperm(len(q), generator=g).cuda()])
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            D, I = index.search(q, k=10, **PARAMS)
        bi, bd = index.plan_buffer("bi", np.int64), index.plan_buffer("bd", np.float32)
        torch.cuda.synchronize()
        assert np.array_equal(bi, I.cpu().numpy().ravel()) and np.array_equal(bd, D.cpu().numpy().ravel())


def test_search_after_a_failed_allocation(octex, small_index):
    """A search whose batch buffers do not fit the GPU is an error, and the next search runs: the failed call's error does
    not stay behind for the next launch's check."""
    from octex_amd._lib import OctexError

    index = octex.load(small_index["path"])
    Q = small_index["Q"][:40]
    D1, I1 = index.search(Q, k=10, **PARAMS)
    m = 1 + torch.cuda.get_device_properties(0).total_memory // (8 * 2048)  # 2048 (id, score) slots a query at least
    q = torch.zeros((m, index.dim), device="cuda")
    print(f"a batch of {m} queries", flush=True)
    with pytest.raises(OctexError, match="hipErrorOutOfMemory"):
        index.search(q, k=1, batch=m, read=1, starts=1, waves=0, rerank=1)
    del q
    D2, I2 = index.search(Q, k=10, **PARAMS)
    assert np.array_equal(I1, I2) and np.array_equal(D1, D2)


def test_oracle_index_with_probed_rows_only(octex, small_index):
    """The host copy that keeps only the list rows a sample's probes reach (the CPU baseline of an index
    too large for host memory) searches that sample exactly like the full copy; array ranges read the
    same bytes as whole arrays and reject ranges outside them."""
    from octex_amd._lib import OctexError

    index = octex.load(small_index["path"])
    Q = small_index["Q"][:50]
    full = O.Index(index)
    part = O.Index(index, queries=Q, read=PARAMS["read"])
    assert (part.lists != 0).sum() < (full.lists != 0).sum()
    D1, I1 = O.search(full, Q, k=10, **PARAMS)
    D2, I2 = O.search(part, Q, k=10, **PARAMS)
    assert np.array_equal(I1, I2) and np.array_equal(D1, D2)
    lists3 = index.array("lists", np.int32, copy=3)
    assert np.array_equal(index.array_range("lists", np.int32, 100, 37, copy=3), lists3[100:137])
    assert index.array_size("lists", copy=3) == lists3.nbytes
    starts = np.array([0, 64, 7, len(lists3) - 16])
    got = index.array_ranges("lists", np.int32, starts, 16, copy=3)
    assert np.array_equal(got, np.stack([lists3[s : s + 16] for s in starts]))
    with pytest.raises(OctexError, match="outside the array"):
        index.array_ranges("lists", np.int32, [len(lists3) - 8], 16, copy=3)
    with pytest.raises(OctexError, match="outside the array"):
        index.array_range("lists", np.int32, len(lists3) - 2, 3, copy=3)
