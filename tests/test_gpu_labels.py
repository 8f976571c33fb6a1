"""GPU hierarchy and labels (hdb_labels_gpu) against the host version
(hdb_labels, itself checked against the tree.cu restatement in
oracle/tree_oracle.py and scikit-learn's tree code): labels and cluster
counts must be equal, on random trees with distinct, tied and zero weights,
on the hand-solved quirk cases, on disconnected input, and on the MST of a
100k-point pipeline run."""
import numpy as np
import pytest

from gpu_hdbscan_amd import api, datasets

pytestmark = pytest.mark.gpu


def _random_tree(rng, n, mode):
    par = np.array([rng.integers(0, i) if i else 0 for i in range(n)])
    e = np.empty(n - 1, api.MST_EDGE)
    e["from_node"], e["to_node"] = par[1:], np.arange(1, n)
    w = rng.gamma(2.0, 1.0, n - 1)
    if mode == 1:
        w = np.round(w, 1)  # ties
    if mode == 2:
        w[: n // 5] = 0.0  # zero weights: lambda = (float)INT_MAX
    if mode == 3:
        w = rng.integers(0, 4, n - 1).astype(float)
    e["weight"] = w.astype(np.float32)
    return e[np.argsort(e["weight"], kind="stable")]


def test_labels_gpu_random_trees(ctx):
    print("case: hdb_labels_gpu vs hdb_labels on random trees", flush=True)
    rng = np.random.default_rng(17)
    for trial in range(80):
        n = int(rng.integers(2, 3000))
        e = _random_tree(rng, n, trial % 4)
        mpts = int(rng.integers(2, 40))
        want, wnc = api.get_clusters(e, n, mpts)
        got, gnc = api.get_clusters_gpu(ctx, e, n, mpts)
        assert gnc == wnc, (trial, n, mpts)
        np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("m", [1, 2, 3, 1023, 1024, 1025, 2047, 2048, 2049, 4097, 40001])
@pytest.mark.parametrize("shape", ["path", "star", "random"])
def test_labels_gpu_segment_edges(ctx, m, shape):
    """Edge counts around the linkage's LDS segments (1024 edges) and the
    halving levels above them, on the deepest, the widest and random trees."""
    print(f"case: hdb_labels_gpu {shape} tree of {m} edges", flush=True)
    rng = np.random.default_rng(m)
    n = m + 1
    e = _random_tree(rng, n, m % 4)
    if shape != "random":
        ids = rng.permutation(n)
        e["from_node"] = ids[:-1] if shape == "path" else ids[0]
        e["to_node"] = ids[1:]
        e = e[rng.permutation(m)]
        e["weight"] = np.sort(e["weight"])
    for mpts in (2, 5, 32):
        want, wnc = api.get_clusters(e, n, mpts)
        got, gnc = api.get_clusters_gpu(ctx, e, n, mpts)
        assert gnc == wnc
        np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("per", [1000, 1025, 5000, 17500, 70001])
@pytest.mark.parametrize("weights", ["tied", "distinct", "zeros"])
def test_labels_gpu_long_clusters(ctx, per, weights):
    """Clusters of more than 1024 stability addends (summed in parallel, bit
    for bit as one by one): a few dense blobs joined by long edges, with
    weights whose exact and rounded sums tie, differ, or start at infinity's
    stand-in (zero weights)."""
    print(f"case: hdb_labels_gpu blobs of {per} points, {weights} weights", flush=True)
    rng = np.random.default_rng(per)
    blobs = 3
    n = blobs * per
    m = n - 1
    e = np.empty(m, api.MST_EDGE)
    child = np.arange(1, n)
    start = (child // per) * per
    joint = child == start
    prev = start + (rng.random(m) * np.maximum(child - start, 1)).astype(np.int64)
    e["from_node"] = np.where(joint, child - per, prev)
    e["to_node"] = child
    if weights == "distinct":
        w = rng.gamma(2.0, 0.1, m)
    else:
        w = rng.choice([0.0, 0.25, 0.5] if weights == "zeros" else [0.25, 0.3, 0.5, 0.75, 1.0], m)
    e["weight"] = np.where(joint, 4.0 + child / n, w).astype(np.float32)
    e = e[np.argsort(e["weight"], kind="stable")]
    for mpts in (2, 32):
        want, wnc = api.get_clusters(e, n, mpts)
        got, gnc = api.get_clusters_gpu(ctx, e, n, mpts)
        assert gnc == wnc
        np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("m", [524_287, 524_288, 524_365, 4_194_381])
@pytest.mark.parametrize("shape", ["path", "star", "random"])
def test_labels_gpu_several_edges_per_thread(ctx, m, shape):
    """From 524,288 edges on a block of the linkage's upper levels takes several
    edges a thread (16 from 4,194,304), the last block a ragged share, and its
    tables and the union-find meet whole trees' worth of contention."""
    print(f"case: hdb_labels_gpu {shape} tree of {m} edges", flush=True)
    rng = np.random.default_rng(m)
    n = m + 1
    ids = rng.permutation(n).astype(np.int32)
    e = np.empty(m, api.MST_EDGE)
    e["from_node"] = {"path": ids[:-1], "star": ids[0], "random": ids[(rng.random(m) * np.arange(1, n)).astype(np.int64)]}[shape]
    e["to_node"] = ids[1:]
    e = e[rng.permutation(m)]
    e["weight"] = np.sort(rng.gamma(2.0, 1.0, m).astype(np.float32).round(3))
    for mpts in (3, 32):
        want, wnc = api.get_clusters(e, n, mpts)
        got, gnc = api.get_clusters_gpu(ctx, e, n, mpts)
        assert gnc == wnc
        np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("weights", ["inf", "nan", "subnormal", "negative"])
@pytest.mark.parametrize("n", [50, 3000, 30_011])
def test_labels_gpu_unusual_weights(ctx, n, weights):
    """Infinite, NaN, subnormal and negative weights give the host's labels
    (lambda 0 or infinity's stand-in, stabilities that are not finite)."""
    print(f"case: hdb_labels_gpu {n} points, {weights} weights", flush=True)
    rng = np.random.default_rng(n)
    e = _random_tree(rng, n, 0)
    w = e["weight"]
    some = rng.random(n - 1) < 0.1
    if weights == "subnormal":
        w *= np.float32(1e-42)
    elif weights == "negative":
        w[some] *= -1
    else:
        w[some] = np.inf if weights == "inf" else np.nan
    e = e[np.argsort(w, kind="stable")]
    for mpts in (2, 7, 32, 1000):
        want, wnc = api.get_clusters(e, n, mpts)
        got, gnc = api.get_clusters_gpu(ctx, e, n, mpts)
        assert gnc == wnc
        np.testing.assert_array_equal(got, want)


def test_labels_gpu_quirk_cases(ctx):
    from test_labels import HAND_CASES, _edges
    for name, rows, n, want, want_nc in HAND_CASES:
        print(f"case: hdb_labels_gpu {name}", flush=True)
        got, nc = api.get_clusters_gpu(ctx, _edges(rows), n, 2)
        assert got.tolist() == want and nc == want_nc, name


def test_labels_gpu_edge_cases(ctx):
    print("case: hdb_labels_gpu edge cases", flush=True)
    one, nc = api.get_clusters_gpu(ctx, np.empty(0, api.MST_EDGE), 1, 5)
    assert one.tolist() == [-1] and nc == 0
    e = np.array([(0, 1, 1.0), (2, 3, 1.0)], api.MST_EDGE)
    with pytest.raises(api.HdbError) as ex:
        api.get_clusters_gpu(ctx, e, 5, 2)  # a forest
    from gpu_hdbscan_amd import _lib
    assert ex.value.status == _lib.HDB_EDISCONNECTED
    # fewer points than mpts: no cluster, every point noise
    e = np.array([(0, 1, 1.0), (1, 2, 2.0)], api.MST_EDGE)
    got, nc = api.get_clusters_gpu(ctx, e, 3, 5)
    assert got.tolist() == [-1, -1, -1] and nc == 0


def test_labels_gpu_pipeline_mst(ctx):
    print("case: hdb_labels_gpu on the mix10 100k pipeline MST", flush=True)
    X = datasets.make("mix10_100k_d12")
    res = api.pipeline(ctx, X, keep_on_device=True)
    assert res.components == 1
    edges = res.edges.numpy()[: res.n_edges]
    want, wnc = api.get_clusters(edges, len(X), 32)
    got, gnc = api.get_clusters_gpu(ctx, res.edges, len(X), 32)
    print("clusters", gnc, "noise", int((got < 0).sum()), flush=True)
    assert gnc == wnc
    np.testing.assert_array_equal(got, want)
