"""Exact BF16 refinement (hdb_refine_knng, distance_mode 2) against the
oracle's exact FP32 brute force (or_bruteforce_fp32: the kNN under the same
FP32 distance, ties by id): ids and distances bit-exact on sampled points,
from tight and from loose (random) bounds, at d = 20 (FP32 matrix-core
tiles), d = 50 and d = 128 (split BF16); and the
distance_mode 2 pipeline at 200,000 x 128 (the anisotropic d = 128 mixture):
recall@32 against FP64 brute force, core distances within 1e-6 relative of
FP64, and the MST bit-exact against Kruskal on the same graph."""
import numpy as np
import pytest

from gpu_hdbscan_amd import api, datasets
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _mixture(n, d, seed):
    rng = np.random.default_rng(seed)
    c = rng.normal(0.0, 6.0, (20, d))
    lab = rng.integers(0, 20, n)
    return (c[lab] + rng.normal(0.0, 1.0, (n, d)) * rng.uniform(0.3, 1.5, d)).astype(np.float32)


def _check_exact(X, L, q):
    ids, dd = O.bruteforce_fp32(X, q, 32)
    np.testing.assert_array_equal(L["label"][q], ids)
    np.testing.assert_array_equal(L["distance"][q], dd)


@pytest.mark.parametrize("d", [20, 50, 128])
def test_refine_exact_from_nndescent_lists(ctx, d):
    print(f"case: refine 20000x{d} from 2-iteration NN-Descent lists", flush=True)
    X = datasets.make("aniso50_2m_d128", n=20000, seed=5) if d == 128 else _mixture(20000, d, 7)
    Xd = ctx.to_device(X)
    L = api.NNDescent(ctx, Xd, iteration=2, store_result_in_device=True)
    before = L.numpy()
    cand, ovf = api.refine_knng(ctx, Xd, L)
    print("survivors per point", cand / len(X), "overflow", ovf, flush=True)
    after = L.numpy()
    q = np.arange(0, len(X), 67, dtype=np.int32)
    _check_exact(X, after, q)
    # every list stays sorted, distinct and self-free; no distance grows
    assert np.all(np.diff(after["distance"], axis=1) >= 0)
    assert not np.any(after["label"] == np.arange(len(X))[:, None])
    assert np.all(after["distance"] <= before["distance"])
    assert cand >= 32 * (len(X) - ovf)


@pytest.mark.parametrize("d", [20, 50, 128])
def test_refine_with_nonfinite_points(ctx, d):
    """Points with NaN or infinite coordinates are at no finite distance from
    any other: they survive no test, and the lists of the other points are the
    exact ones, from bounds that hold no finite distance too."""
    print(f"case: refine 3000x{d} with NaN and infinite coordinates", flush=True)
    X = _mixture(3000, d, 13)
    X[7::97, 0], X[31::97, d - 1], X[57::97, d // 2] = np.nan, np.inf, -np.inf
    L = api.NNDescent(ctx, X, iteration=2)
    Ld = ctx.to_device(L)
    api.refine_knng(ctx, ctx.to_device(X), Ld)
    finite = np.flatnonzero(np.isfinite(X).all(1)).astype(np.int32)
    assert not np.isfinite(L["distance"][finite, 31]).all()
    at = np.arange(0, len(finite), 7, dtype=np.int32)  # the oracle ranks the finite points alone
    ids, dd = O.bruteforce_fp32(X[finite], at, 32)
    got = Ld.numpy()[finite[at]]
    np.testing.assert_array_equal(got["label"], finite[ids])
    np.testing.assert_array_equal(got["distance"], dd)


def test_refine_overflow_falls_back_to_bruteforce(ctx):
    """Random initial lists bound nothing useful: (almost) every point has
    more than 128 survivors and is answered by the exact brute force; the
    lists are exact either way."""
    print("case: refine 3000x40 from random lists (overflow path)", flush=True)
    X = _mixture(3000, 40, 11)
    Xd = ctx.to_device(X)
    L = api.NNDescent(ctx, Xd, iteration=0, store_result_in_device=True)
    cand, ovf = api.refine_knng(ctx, Xd, L)
    print("overflow", ovf, flush=True)
    assert ovf > 0
    _check_exact(X, L.numpy(), np.arange(0, 3000, 7, dtype=np.int32))


def test_refine_rejects_bad_input(ctx):
    X = _mixture(100, 130, 1)
    Xd = ctx.to_device(X)
    L = ctx.empty((100, 32), api.NND_ELEMENT)
    with pytest.raises(api.HdbError):
        api.refine_knng(ctx, Xd, L)  # d > 128
    with pytest.raises(api.HdbError):
        api.pipeline(ctx, Xd, params=api.default_params(distance_mode=3))


def test_distance_mode2_pipeline_200k_d128(ctx):
    print("case: distance_mode 2 pipeline aniso50 200000x128", flush=True)
    n = 200000
    X = datasets.make("aniso50_2m_d128", n=n, seed=3)
    Xd = ctx.to_device(X)
    p = api.default_params(distance_mode=2, join_keep=4, nnd_iteration=6)
    res = api.pipeline(ctx, Xd, params=p)
    L = res.lists
    q = np.arange(0, n, 661, dtype=np.int32)
    gt, _ = O.bruteforce_fp64(X, q, 32)
    r = O.recall(L["label"][q], gt, 32)
    print("recall@32", r, flush=True)
    assert r >= 0.99
    _check_exact(X, L, q[:60])
    # core distances: FP64 recomputation on the returned neighbours
    j = L["label"][:, 31]
    f64 = np.sqrt(((X.astype(np.float64) - X[j].astype(np.float64)) ** 2).sum(1))
    rel = np.max(np.abs(res.core.astype(np.float64) - f64) / f64)
    print("max relative core error", rel, flush=True)
    assert rel < 1e-6
    # MST on the same graph: Kruskal over the oracle's CSR
    counts = O.hub_counts(L)
    np.testing.assert_array_equal(res.counts, counts)
    ah = O.antihubs(L, counts)
    ni, nl, w = O.mrd_csr(X, L, O.core(X, L, 32), ah)
    edges, _ = O.kruskal(ni, nl, w)
    edges = O.sort_edges(edges)
    assert res.n_edges == len(edges)
    np.testing.assert_array_equal(res.edges[: res.n_edges], edges)


def test_distance_mode2_mst_equals_fp32_only_path(ctx):
    """The FP32-only path to the same graph: the exact FP32 brute force of
    every point (hdb_bruteforce_knn, no BF16 anywhere) fed to the pipeline as
    given lists.  The BF16 path's lists, core distances, MST and sorted edges
    equal it bit for bit."""
    print("case: distance_mode 2 vs FP32-only exact graph 40000x128", flush=True)
    n = 40000
    X = datasets.make("aniso50_2m_d128", n=n, seed=8)
    Xd = ctx.to_device(X)
    res = api.pipeline(ctx, Xd, params=api.default_params(distance_mode=2, join_keep=4, nnd_iteration=4))
    ids, d2 = api.bruteforce_knn(ctx, Xd, np.arange(n, dtype=np.int32), 32)
    L = np.empty((n, 32), api.NND_ELEMENT)
    L["label"], L["distance"] = ids, d2
    ref = api.pipeline(ctx, Xd, params=api.default_params(), knng_mode=4, outputs={"lists": ctx.to_device(L)})
    np.testing.assert_array_equal(res.lists, ref.lists)
    np.testing.assert_array_equal(res.core.view(np.uint32), ref.core.view(np.uint32))
    assert res.n_edges == ref.n_edges and res.components == ref.components
    np.testing.assert_array_equal(res.edges[: res.n_edges], ref.edges[: ref.n_edges])


@pytest.mark.parametrize("n,d", [(30000, 12), (20000, 128), (5000, 40)])
def test_exact_knn_bounded_equals_bruteforce(ctx, n, d):
    """Bounded exact kNN of sampled queries (the learned check's ground
    truth) equals the FP32 brute force bit for bit, from good and from
    random lists, bad ids included; the lists are left as they are."""
    print(f"case: exact_knn_bounded {n}x{d}", flush=True)
    X = datasets.make("mix30_1m_d12", n=n, seed=4) if d == 12 else (
        datasets.make("aniso50_2m_d128", n=n, seed=6) if d == 128 else _mixture(n, d, 3))
    Xd = ctx.to_device(X)
    q = np.r_[np.arange(0, n, 37), [-1, n, n + 5]].astype(np.int32)
    want_ids, want_d2 = api.bruteforce_knn(ctx, Xd, q, 32)
    for its in (3, 0):
        L = api.NNDescent(ctx, Xd, iteration=its, store_result_in_device=True)
        before = L.numpy()
        ids, d2 = api.exact_knn_bounded(ctx, Xd, L, q, 32)
        np.testing.assert_array_equal(ids, want_ids)
        np.testing.assert_array_equal(d2[ids >= 0], want_d2[want_ids >= 0])
        np.testing.assert_array_equal(L.numpy(), before)
    good = q[(q >= 0) & (q < n)]
    ref, _ = O.bruteforce_fp32(X, good, 32)
    np.testing.assert_array_equal(ids[: len(good)], ref)
