"""GPU parity of the kNN-graph stage (hdb_nndescent, hdb_knn_merge,
hdb_build_knng_blocked, hdb_bruteforce_knn) against the CPU oracle.

Bars: init lists bit-exact (ids and FP32 distances) against the oracle's
restatement of InitKNNGraphIndexKernel; NN-Descent lists sorted, self-free,
duplicate-free, every stored distance bit-equal to the oracle's FP32 formula
on the returned neighbour; recall@32 >= 0.95 against FP64 brute force.
"""
import ctypes as C

import numpy as np
import pytest

from gpu_hdbscan_amd import api, datasets
from oracle import nnd_oracle as N
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _check_lists(X, L, n_valid=None):
    n = len(X)
    ids = L["label"]
    assert np.all(ids >= 0)
    assert not np.any(ids == np.arange(n)[:, None])
    for i in range(0, n, max(1, n // 300)):
        row = ids[i]
        valid = row[row != 0x7FFFFFFF]
        assert len(set(valid.tolist())) == len(valid)
        d = L["distance"][i][: len(valid)]
        assert np.all(np.diff(d) >= 0)
        ref = np.array([O.d2(X[i], X[j]) for j in valid], np.float32)
        np.testing.assert_array_equal(d, ref)


def _recall(X, L, m=1000, seed=0):
    rng = np.random.default_rng(seed)
    q = rng.choice(len(X), size=min(m, len(X)), replace=False).astype(np.int32)
    gt, _ = O.bruteforce_fp64(X, q, 32)
    return O.recall(L["label"][q], gt, 32)


@pytest.mark.parametrize("d", [12, 3, 15, 16, 31, 40])
def test_init_bit_exact(ctx, d):
    """Random init against the oracle, ids and FP32 distances bit for bit,
    at every layout the init reads: the padded point rows (16 floats for
    d <= 15, 32 for 16 <= d <= 31, the list bound in the last column) and
    the points themselves (d >= 32)."""
    print(f"case: init 5000x{d}", flush=True)
    X = datasets.tiny_blobs(5000, d, 8, seed=11 + d)
    L = api.NNDescent(ctx, X, iteration=0)
    ref = O.init_random(X)
    np.testing.assert_array_equal(L["label"], ref["label"])
    np.testing.assert_array_equal(L["distance"].view(np.uint32), ref["distance"].view(np.uint32))


@pytest.mark.parametrize("d", [12, 32, 20, 3, 8])
def test_nndescent_recall(ctx, d):
    print(f"case: nndescent 20000x{d}", flush=True)
    X = datasets.tiny_blobs(20000, d, 12, seed=d)
    L = api.NNDescent(ctx, X, iteration=8)
    _check_lists(X, L)
    r = _recall(X, L)
    print("recall", r, ctx.nnd_stats(), flush=True)
    assert r >= 0.95


def test_nndescent_mix10_100k(ctx):
    print("case: nndescent mix10_100k_d12", flush=True)
    X = datasets.make("mix10_100k_d12")
    L = api.NNDescent(ctx, X, iteration=6)
    _check_lists(X, L)
    r = _recall(X, L, m=2000)
    print("recall", r, ctx.nnd_stats(), flush=True)
    assert r >= 0.95


def test_small_n_exact(ctx):
    # n <= K+1: every list holds all other points (closed form)
    print("case: nndescent n=20", flush=True)
    X = datasets.tiny_blobs(20, 12, 2, seed=3)
    L = api.NNDescent(ctx, X, iteration=3)
    for i in range(20):
        row = L["label"][i]
        valid = row[row != 0x7FFFFFFF]
        assert sorted(valid.tolist()) == [j for j in range(20) if j != i]


def test_bruteforce_matches_oracle(ctx):
    print("case: bruteforce 3000x12", flush=True)
    X = datasets.tiny_blobs(3000, 12, 4, seed=5)
    q = np.arange(0, 3000, 7, dtype=np.int32)
    ids, d2 = api.bruteforce_knn(ctx, X, q, 32)
    gt, _ = O.bruteforce_fp64(X, q, 32)
    assert O.recall(ids, gt, 32) >= 0.999  # FP32 vs FP64 ties only
    for r, qq in enumerate(q[:50]):
        np.testing.assert_array_equal(d2[r], np.array([O.d2(X[qq], X[j]) for j in ids[r]], np.float32))


@pytest.mark.parametrize("d", [12, 32, 20])
def test_bruteforce_tiled_and_bad_ids(ctx, d):
    """The tiled brute force (d = 12, 32) and the one-wave form (other d)
    against the oracle's FP64 ranking, with an out-of-range query id."""
    print(f"case: bruteforce 7000x{d} with a bad id", flush=True)
    X = datasets.tiny_blobs(7000, d, 5, seed=50 + d)
    q = np.array([0, 6999, 123, 7000, 4567], np.int32)
    ids, d2 = api.bruteforce_knn(ctx, X, q, 32)
    assert np.all(ids[3] == -1)
    ok = np.array([0, 1, 2, 4])
    gt, _ = O.bruteforce_fp64(X, q[ok], 32)
    assert O.recall(ids[ok], gt, 32) >= 0.999
    for r in ok:
        assert np.all(np.diff(d2[r]) >= 0) and q[r] not in ids[r]
        np.testing.assert_array_equal(d2[r], np.array([O.d2(X[q[r]], X[j]) for j in ids[r]], np.float32))
    # fewer than kq other points
    ids_s, _ = api.bruteforce_knn(ctx, X[:20], np.array([3], np.int32), 32)
    assert sorted(ids_s[0][ids_s[0] >= 0].tolist()) == [j for j in range(20) if j != 3]


@pytest.mark.parametrize("d", [7, 33, 128])
@pytest.mark.parametrize("m", [1, 16, 3000])
def test_bruteforce_point_chunks(ctx, m, d):
    """Other dimensions split the points into chunks for few queries: one
    chunk of all points or many ragged ones, the same exact lists."""
    print(f"case: bruteforce {m} queries of 5003x{d}", flush=True)
    X = datasets.tiny_blobs(5003, d, 5, seed=m + d)
    q = np.random.default_rng(m).choice(5003, m, replace=False).astype(np.int32)
    ids, d2 = api.bruteforce_knn(ctx, X, q, 32)
    want, wd = O.bruteforce_fp32(X, q, 32)
    np.testing.assert_array_equal(ids, want)
    np.testing.assert_array_equal(d2, wd)
    few, _ = api.bruteforce_knn(ctx, X, q, 5)
    np.testing.assert_array_equal(few, want[:, :5])


@pytest.mark.parametrize("n,d", [(600, 7), (64, 128), (5000, 33)])
def test_bruteforce_many_queries_keep_no_scratch(n, d):
    """More queries than waves fill the chip: the lists are written by the
    scan itself, and the context keeps no memory that grows with the queries
    (it once kept 256 bytes for each: 51 MB here)."""
    def free(c):  # through the library's own HIP runtime
        a, b = C.c_size_t(), C.c_size_t()
        assert c.lib.hipMemGetInfo(C.byref(a), C.byref(b)) == 0
        return a.value

    print(f"case: bruteforce 200000 queries of {n}x{d}", flush=True)
    X = datasets.tiny_blobs(n, d, 5, seed=d)
    q = (np.arange(200_000) % (n + 2) - 1).astype(np.int32)
    with api.Context(0) as c:
        api.bruteforce_knn(c, X, q[:1], 32)
        before = free(c)
        ids, d2 = api.bruteforce_knn(c, X, q, 32)
        assert before - free(c) < 16 << 20
    rows = np.r_[1:40, 1 + n // 2, n]
    want, wd = O.bruteforce_fp32(X, q[rows], 32)
    np.testing.assert_array_equal(ids[rows], want)
    np.testing.assert_array_equal(d2[rows], wd)
    assert np.all(ids[[0, n + 1]] == -1) and np.all(np.isinf(d2[[0, n + 1]]))


def test_recall_on_device_matches_oracle(ctx):
    """hdb_recall (Evaluate, tools/evaluate.hpp:13-52) equals the oracle's
    recall on the same rows, for lists of varying quality."""
    print("case: device recall 5000x12", flush=True)
    X = datasets.tiny_blobs(5000, 12, 6, seed=77)
    q = np.arange(0, 5000, 9, dtype=np.int32)
    gt, _ = O.bruteforce_fp64(X, q, 32)
    for its in (0, 1, 3):
        L = api.NNDescent(ctx, X, iteration=its)
        want = O.recall(L["label"][q], gt, 32)
        got = api.recall(ctx, L, q, gt.astype(np.int32))
        assert got == pytest.approx(want, abs=0)
    for kq in (1, 10):
        L = api.NNDescent(ctx, X, iteration=2)
        want = O.recall(L["label"][q][:, :kq], gt[:, :kq], kq)
        assert api.recall(ctx, L, q, np.ascontiguousarray(gt[:, :kq], np.int32), kq) == pytest.approx(want, abs=0)


def test_size_guard_rejects_large_n(ctx):
    """n >= 2^26 is rejected before any kernel runs (the n x 32 reverse
    pairs use int32 positions); tiny buffers are passed on purpose, and no
    kernel may touch them."""
    import ctypes as C
    from gpu_hdbscan_amd import _lib
    X = ctx.empty((64,), np.float32)
    out = ctx.empty((64,), api.NND_ELEMENT)
    p = api.default_params()
    st = ctx.lib.hdb_nndescent(ctx.handle, X.ptr, 1 << 26, 12, C.byref(p), out.ptr)
    assert st == _lib.HDB_EINVAL and b"2^26" in ctx.lib.hdb_last_error(ctx.handle)
    nidx = ctx.empty((64,), np.int64)
    E = C.c_int64()
    st = ctx.lib.hdb_mrd_graph(ctx.handle, X.ptr, out.ptr, X.ptr, None, 0, 1 << 26, 12, 32, nidx.ptr, None, None,
                               C.byref(E))
    assert st == _lib.HDB_EINVAL


def test_knn_merge(ctx):
    """KNNMergeFromHost alone: a valid graph of the whole set that finds the
    cross-half neighbours the inputs lack (its lists start from each input's
    16 best plus 16 random cross-half ids, knnmerge.cu:80-185).  As the
    reference uses it -- unique-merged into each half's running lists, the
    2-shard GenLargeKNNGraph -- the result's recall on the whole set is at
    least the inputs' recall on their own halves."""
    print("case: knn_merge 2x8000x12", flush=True)
    X = datasets.tiny_blobs(16000, 12, 10, seed=21)
    a, b = X[:8000], X[8000:]
    ga = api.NNDescent(ctx, a, iteration=6)
    gb = api.NNDescent(ctx, b, iteration=6)
    gm = api.KNNMergeFromHost(ctx, a, ga, b, gb)
    _check_lists(X, gm)
    r = _recall(X, gm)
    ra, rb = _recall(a, ga, seed=1), _recall(b, gb, seed=2)
    lifted = np.concatenate([ga, gb])
    lifted["label"][8000:] += 8000
    r_inputs = _recall(X, lifted)
    blocked = api.GenLargeKNNGraph(ctx, X, 2)
    r_blocked = _recall(X, blocked)
    print("merge recall", r, "inputs on their halves", ra, rb, "inputs on the whole set", r_inputs,
          "2-shard build", r_blocked, flush=True)
    assert r >= 0.95 and r > r_inputs + 0.2
    assert r_blocked >= min(ra, rb)


def test_blocked_equals_oracle_composition(ctx):
    """hdb_build_knng_blocked with 3 blocks equals the composition of the
    reference schedule's steps (MultiMerge, gen_large_knngraph.cu:249-407):
    per-block hdb_nndescent, hdb_knn_merge of every pair i < j in order, and
    the oracle's UniqueMergeSequential of each pair result into the running
    lists of both blocks -- bit for bit, since no step drops a proposal here
    (every step is then deterministic)."""
    print("case: blocked x3 vs composition with the oracle unique merge, 30000x12", flush=True)
    X = datasets.tiny_blobs(30000, 12, 12, seed=61)
    n, nb = len(X), 3
    off = [n * i // nb for i in range(nb + 1)]
    got = api.GenLargeKNNGraph(ctx, X, nb)
    assert ctx.nnd_stats()["bucket_drops"] == 0
    local = []
    for i in range(nb):
        local.append(api.NNDescent(ctx, X[off[i]:off[i + 1]], iteration=6))
        assert ctx.nnd_stats()["bucket_drops"] == 0
    running = np.concatenate(local).copy()
    for i in range(nb):
        lab = running[off[i]:off[i + 1]]["label"]
        running[off[i]:off[i + 1]]["label"] = np.where(lab == 0x7FFFFFFF, lab, lab + off[i])
    for i in range(nb):
        for j in range(i + 1, nb):
            ni = off[i + 1] - off[i]
            pair = api.KNNMergeFromHost(ctx, X[off[i]:off[i + 1]], local[i], X[off[j]:off[j + 1]], local[j])
            assert ctx.nnd_stats()["bucket_drops"] == 0
            running[off[i]:off[i + 1]] = O.unique_merge(running[off[i]:off[i + 1]], pair, 0, ni, off[i], off[j])
            running[off[j]:off[j + 1]] = O.unique_merge(running[off[j]:off[j + 1]], pair, ni, ni, off[i], off[j])
    np.testing.assert_array_equal(got["label"], running["label"])
    np.testing.assert_array_equal(got["distance"].view(np.uint32), running["distance"].view(np.uint32))


def test_reference_pairing_recall(ctx):
    """join_keep = 0 is the reference's pairing (NEIGHB_CACHE_NUM = 1,
    nndescent.cuh:24: each candidate proposes its nearest new and, if new,
    its nearest old partner); it still converges to a high recall."""
    print("case: join_keep 0 recall 20000x12", flush=True)
    X = datasets.tiny_blobs(20000, 12, 12, seed=12)
    for its in (6, 10):
        L = api.NNDescent(ctx, X, iteration=its, params=api.default_params(join_keep=0))
        _check_lists(X, L)
        r = _recall(X, L)
        print("join_keep 0 iterations", its, "recall", r, flush=True)
    assert r >= 0.9


def test_blocked_build(ctx):
    print("case: blocked 4 blocks 40000x12", flush=True)
    X = datasets.tiny_blobs(40000, 12, 16, seed=31)
    L = api.GenLargeKNNGraph(ctx, X, 4)
    _check_lists(X, L)
    r = _recall(X, L)
    print("blocked recall", r, flush=True)
    assert r >= 0.95


def test_replay_same_seed_inputs(ctx):
    print("case: replay 10000x12", flush=True)
    X = datasets.tiny_blobs(10000, 12, 6, seed=41)
    a = api.NNDescent(ctx, X, iteration=6)
    st = ctx.nnd_stats()
    b = api.NNDescent(ctx, X, iteration=6)
    if st["bucket_drops"] == 0 and st["reverse_drops"] == 0:
        np.testing.assert_array_equal(a, b)
    else:
        # drops depend on atomic arrival order; sets still agree closely
        assert O.recall(a["label"], b["label"], 32) > 0.99


@pytest.mark.parametrize("keep", [0, 3])
def test_list_distances_never_grow(ctx, keep):
    """An update only replaces entries by closer ones, so after every
    iteration (from the second on) each list's k-th distance, and the sum
    over its entries, is at most what it was.  Runs of 0..4 iterations are
    prefixes of one another: the path is deterministic."""
    print(f"case: per-iteration list monotonicity 20000x12 keep={keep}", flush=True)
    X = datasets.tiny_blobs(20000, 12, 10, seed=53)
    prev = None
    for its in range(0, 5):
        p = api.default_params(nnd_iteration=its, join_keep=keep)
        L = api.NNDescent(ctx, X, iteration=its, params=p)
        d = L["distance"].astype(np.float64)
        if prev is not None and its >= 2:  # the first update also removes repeated random ids
            assert np.all(d[:, -1] <= prev[:, -1])
            assert np.all(d.sum(1) <= prev.sum(1) * (1 + 1e-12))
        prev = d


def _points_with_ties(n, d, seed, ties):
    """A mixture; `ties`: coordinates on a coarse grid, with repeated points,
    so that many candidate distances are equal."""
    X = datasets.tiny_blobs(n, d, 6, seed=seed, spread=4.0)
    if ties:
        X = np.round(X).astype(np.float32)
        X[: n // 8] = X[n // 2: n // 2 + n // 8]
    return X


@pytest.mark.parametrize("d", [1, 2, 4, 5, 8, 9, 11, 13, 15, 16, 17, 20, 21, 24, 25, 31])
@pytest.mark.parametrize("ties", [False, True])
def test_join_rows_equals_wider_join(ctx, d, ties):
    """Zero columns change no distance, so the same points padded past the
    dimensions of the register-row join take another join kernel to the same
    lists, bit for bit, for every join_keep and for the merge schedule."""
    print(f"case: join at d={d} against the same points padded to d=40, ties={ties}", flush=True)
    n = 3001
    X = _points_with_ties(n, d, 90 + d, ties)
    P = np.zeros((n, 40), np.float32)
    P[:, :d] = X
    for keep in (0, 1, 2, 3, 4, 8):
        p = api.default_params(join_keep=keep, bucket_cap=1024)  # room for every proposal of join_keep 8
        a = api.NNDescent(ctx, X, iteration=4, params=p)
        b = api.NNDescent(ctx, P, iteration=4, params=p)
        assert ctx.nnd_stats()["bucket_drops"] == 0
        np.testing.assert_array_equal(a["label"], b["label"])
        np.testing.assert_array_equal(a["distance"].view(np.uint32), b["distance"].view(np.uint32))
    for keep in (0, 4):
        p = api.default_params(join_keep=keep, bucket_cap=1024)
        a = api.GenLargeKNNGraph(ctx, X, 2, params=p)
        b = api.GenLargeKNNGraph(ctx, P, 2, params=p)
        assert ctx.nnd_stats()["bucket_drops"] == 0
        np.testing.assert_array_equal(a["label"], b["label"])
        np.testing.assert_array_equal(a["distance"].view(np.uint32), b["distance"].view(np.uint32))


@pytest.mark.parametrize("d", [33, 37, 63, 64, 65, 100, 128, 255])
@pytest.mark.parametrize("ties", [False, True])
def test_join_wide_dimensions(ctx, d, ties):
    """The chunked join at ragged dimensions: its lists hold the oracle's
    distances and do not change when zero columns move the chunk ends."""
    print(f"case: join at d={d} against zero columns before it, ties={ties}", flush=True)
    n = 1501
    X = _points_with_ties(n, d, 190 + d, ties)
    lead = min(255 - d, 7)
    P = np.zeros((n, d + lead), np.float32)
    P[:, lead:] = X
    for keep in (0, 2, 4, 8):
        p = api.default_params(join_keep=keep, bucket_cap=1024)
        a = api.NNDescent(ctx, X, iteration=3, params=p)
        b = api.NNDescent(ctx, P, iteration=3, params=p)
        assert ctx.nnd_stats()["bucket_drops"] == 0
        np.testing.assert_array_equal(a["label"], b["label"])
        np.testing.assert_array_equal(a["distance"].view(np.uint32), b["distance"].view(np.uint32))
    for i in range(0, n, 150):
        np.testing.assert_array_equal(a["distance"][i], np.array([O.d2(X[i], X[j]) for j in a["label"][i]], np.float32))


@pytest.mark.parametrize("d", [12, 32])
@pytest.mark.parametrize("S", [1, 3, 4, 5, 11, 16])
def test_join_matrix_values_equal_general(ctx, d, S):
    """The joins of d = 12 and 32 rank by matrix products.  With small whole
    coordinates every ranking value is exact, and in merge mode a candidate's
    partners are of one kind, so ties go to the smaller id in every kernel: a
    zero column, which takes the same points to the kernels of other
    dimensions, changes no list.  S moves the candidate counts over the
    products' blocks of four."""
    print(f"case: merge join d={d} S={S} against d={d + 1}", flush=True)
    n = 700
    X = np.clip(np.round(datasets.tiny_blobs(2 * n, d, 6, seed=7 * d + S, spread=4.0)), -40, 40).astype(np.float32)
    P = np.zeros((2 * n, d + 1), np.float32)
    P[:, :d] = X
    for keep in (0, 1, 2, 3, 4, 8):
        p = api.default_params(join_keep=keep, merge_sample_num=S, bucket_cap=1024)
        ga = api.NNDescent(ctx, P[:n], iteration=2, params=p)
        gb = api.NNDescent(ctx, P[n:], iteration=2, params=p)
        a = api.KNNMergeFromHost(ctx, X[:n], ga, X[n:], gb, params=p)
        b = api.KNNMergeFromHost(ctx, P[:n], ga, P[n:], gb, params=p)
        assert ctx.nnd_stats()["bucket_drops"] == 0
        np.testing.assert_array_equal(a["label"], b["label"])
        np.testing.assert_array_equal(a["distance"].view(np.uint32), b["distance"].view(np.uint32))


@pytest.mark.parametrize("n", [256, 257, 12500, 12501, 40000])
@pytest.mark.parametrize("S", [3, 16])
def test_reverse_sort_without_unused_slots(ctx, n, S):
    """The reverse sort leaves out the slots no sample uses: at the one-block
    sort's largest point count and past it, at both sides of the change of
    tile size (n x 32 slots), and with few of the slots in use (S = 3).  The
    lists are distinct, sorted and hold the oracle's distances; with S = 16
    they reach the recall of the other sizes."""
    print(f"case: reverse sort n={n} S={S}", flush=True)
    X = datasets.tiny_blobs(n, 12, 8, seed=n + S)
    p = api.default_params(sample_num=S, bucket_cap=1024)
    L = api.NNDescent(ctx, X, iteration=6, params=p)
    _check_lists(X, L)
    assert ctx.nnd_stats()["bucket_drops"] == 0
    if S == 16:
        assert _recall(X, L) >= 0.95


@pytest.mark.parametrize("d", [12, 32])
@pytest.mark.parametrize("shift", [300, 1000, 3000, 30000])
def test_join_far_from_the_origin(ctx, d, shift):
    """A shift of every point changes neighbours by the points' own rounding
    only: the joins that rank by |a|^2 - 2 a.b + |b|^2 reach the recall of the
    kernels that rank by distances (the same points with a zero column), for
    every pairing and a merge."""
    print(f"case: join at d={d}, points {shift} from the origin", flush=True)
    n = 20000
    X = (datasets.tiny_blobs(n, d, 12, seed=d) + np.float32(shift)).astype(np.float32)
    P = np.zeros((n, d + 1), np.float32)
    P[:, :d] = X
    for keep in (0, 1, 2, 3, 4, 8):
        p = api.default_params(join_keep=keep)
        a, b = (_recall(X, api.NNDescent(ctx, Y, iteration=8, params=p)) for Y in (X, P))
        assert a > b - 0.01, (keep, a, b)
    for keep in (0, 4):
        p = api.default_params(join_keep=keep)
        a, b = (_recall(X, api.GenLargeKNNGraph(ctx, Y, 2, params=p)) for Y in (X, P))
        assert a > b - 0.01, (keep, a, b)


def _whole_points(n, d, seed, kind):
    """Points with whole coordinates, so that every distance, and every value
    the joins rank by, is exact in FP32 (distances below 2^18 for d = 12 and 32,
    whose keys drop six bits; below 2^24 otherwise), and their float32 squared
    distances.  kind: fine, coarse (many equal distances and repeated points),
    or nonfinite (some NaN and infinite coordinates)."""
    r = int(np.sqrt((1 << (18 if d in (12, 32) else 24)) / d) / 2) - 1
    X = np.clip(datasets.tiny_blobs(n, d, 6, seed=seed, spread=4.0) / 9, -1, 1)
    X = np.round(X * (4 if kind == "coarse" else r)).astype(np.float32)
    if kind == "coarse":
        X[: n // 8] = X[n // 2: n // 2 + n // 8]
    if kind == "nonfinite":
        X[7::101, 0], X[31::101, d - 1], X[57::101, d // 2] = np.nan, np.inf, -np.inf
    with np.errstate(invalid="ignore"):
        D = np.stack([((X - x).astype(np.float64) ** 2).sum(1) for x in X]).astype(np.float32)
    D.view(np.uint32)[np.isnan(D)] = 0x7FC00000
    return X, D


def _equal_lists(L, lists):
    ids, bits = N.arrays(lists)
    np.testing.assert_array_equal(np.where(L["label"] == 0x7FFFFFFF, -1, L["label"]), ids)
    np.testing.assert_array_equal(L["distance"], bits.view(np.float32))  # a NaN's sign is the hardware's


# d = 12 and 32 rank by |a|^2 - 2 a.b + |b|^2: no exact order among infinite values
@pytest.mark.parametrize("d,kind", [(d, kind) for d in (2, 8, 11, 12, 13, 20, 24, 31, 32, 40)
                                    for kind in ("fine", "coarse", "nonfinite")
                                    if kind != "nonfinite" or d not in (12, 32)])
def test_nndescent_equals_oracle(ctx, d, kind):
    """Every list of three iterations, ids and distances, against the numpy
    NN-Descent, for every pairing and a merge: each join kernel chooses the
    nearest partners (equal distances: the smaller id; at d = 12 and 32 the
    earlier candidate).  Pairs at no finite distance are never proposed."""
    print(f"case: NN-Descent of 330x{d}, {kind} points, against the oracle", flush=True)
    n = 330
    X, D = _whole_points(n, d, 11 * d, kind)
    B = D.view(np.uint32)
    slot = d in (12, 32)
    for keep, S in ((0, 16), (1, 16), (3, 7), (8, 16)):
        p = api.default_params(join_keep=keep, sample_num=S, bucket_cap=1024)
        L = api.NNDescent(ctx, X, iteration=3, params=p)
        assert ctx.nnd_stats()["bucket_drops"] == 0
        _equal_lists(L, N.descend(D, N.init_random(B), S, keep, 3, by_slot=slot))
    n1 = 180
    for keep in (0, 4):
        p = api.default_params(join_keep=keep, merge_sample_num=9, merge_iteration=2, bucket_cap=1024)
        g1, g2 = api.NNDescent(ctx, X[:n1], iteration=2, params=p), api.NNDescent(ctx, X[n1:], iteration=2, params=p)
        L = api.KNNMergeFromHost(ctx, X[:n1], g1, X[n1:], g2, params=p)
        _equal_lists(L, N.descend(D, N.init_merge(B, g1["label"], g2["label"]), 9, keep, 2, split=n1, by_slot=slot))
