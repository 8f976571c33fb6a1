"""Workloads of the HDBSCAN hot path whose speed is tracked.

Each case is one call (or the few calls) that a program using this package
makes on points already on the GPU, over the sizes it is used at: from a few
thousand points, where launches and round trips decide, to ten million; at
the dimension the mixtures have (12), at other and odd ones, and at 32 and 128.

  whole    kNN graph -> hub counts -> core distances -> MRD graph -> MST ->
           sorted edges (api.pipeline), then the GPU labels when the tree spans
  learned  the same path from learned initial lists with its sampled recall
           check (learned.pipeline_learned_checked), networks in hand
  fit      training of those networks, subsample graph included
  knng     the kNN graph alone (api.NNDescent)
  refined  the path with the BF16 join and the exact refinement (distance_mode 2)
  blocked  the reference's schedule: block graphs, all-pairs merge
  graph    the graph stage on a kNN graph in hand (knng_mode 4)
  core_sg  Core-SG and the MSTs of several mpts from it
"""
from __future__ import annotations

import math

import numpy as np
import torch

from gpu_hdbscan_amd import api, learned
from gpu_hdbscan_amd._lib import MST_EDGE, NND_ELEMENT

K = 32
CORE_SG_MPTS = (4, 16, 32)


def listed():
    return [
        # the smoke test's size: a first look at a small data set, bound by launches and host round trips
        dict(name="whole_5k_d12", kind="whole", n=5000, d=12, data="iso", keep=4, iters=6),
        # a desktop-sized clustering job (the mix10_100k_d12 workload's size), library defaults
        dict(name="whole_100k_d12", kind="whole", n=100_000, d=12, data="iso", keep=4, iters=6),
        # the mix30_1m_d12 workload at the setting the benchmark's plain leg runs
        dict(name="whole_1m_d12", kind="whole", n=1_000_000, d=12, data="iso", keep=3, iters=6),
        # the headline workload's size and plain setting (mix100_10m_d12)
        dict(name="whole_10m_d12", kind="whole", n=10_000_000, d=12, data="iso", keep=2, iters=9),
        # a program that reuses trained networks on new points
        dict(name="learned_1m_d12", kind="learned", n=1_000_000, d=12, data="iso", keep=4, iters=4),
        # training for one run, as the benchmark's learned leg counts it
        dict(name="fit_1m_d12", kind="fit", n=1_000_000, d=12, data="iso"),
        # feature vectors of another dimension, a ragged point count
        dict(name="knng_300k_d20", kind="knng", n=300_007, d=20, data="iso", keep=4, iters=6),
        # the aniso200_5m_d32 workload's shape, a tenth of its points
        dict(name="knng_500k_d32", kind="knng", n=500_000, d=32, data="aniso", keep=3, iters=7),
        # the aniso50_2m_d128 workload's shape: embeddings, exact lists wanted
        dict(name="refined_100k_d128", kind="refined", n=100_000, d=128, data="aniso", keep=4, iters=6),
        # the reference's block schedule (GenLargeKNNGraph), ragged last block
        dict(name="blocked_400k_d12", kind="blocked", n=400_001, d=12, data="iso", blocks=4),
        # a kNN graph computed elsewhere (read from a .kgraph file), odd sizes
        dict(name="graph_50k_d16", kind="graph", n=50_021, d=16, data="iso"),
        # one graph for the hierarchies of several mpts
        dict(name="core_sg_50k_d12", kind="core_sg", n=50_000, d=12, data="iso"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(["whole", "knng", "learned", "refined", "blocked", "graph", "core_sg", "fit"],
                       [4, 4, 1, 1, 1, 2, 1, 1])[0]
    c = dict(kind=kind, data=rng.choice(["iso", "aniso"]))
    if kind == "whole":
        c.update(n=_log_int(rng, 2000, 2_000_000), d=rng.choice([12, rng.randint(2, 40)]), keep=rng.choice([2, 3, 4]),
                 iters=rng.randint(4, 9))
    elif kind == "knng":
        c.update(n=_log_int(rng, 1000, 1_000_000), d=rng.choice([12, 32, rng.randint(2, 64), rng.randint(2, 64)]),
                 keep=rng.choice([0, 1, 2, 3, 4, 4, 8]), iters=rng.randint(4, 9))
    elif kind == "learned":
        c.update(n=_log_int(rng, 100_000, 2_000_000), d=12, data="iso", keep=4, iters=rng.randint(4, 6))
    elif kind == "fit":
        c.update(n=_log_int(rng, 50_000, 2_000_000), d=rng.choice([12, rng.randint(4, 32)]))
    elif kind == "refined":
        c.update(n=_log_int(rng, 5000, 150_000), d=rng.choice([128, rng.randint(33, 127)]), data="aniso", keep=4,
                 iters=rng.randint(4, 6))
    elif kind == "blocked":
        c.update(n=_log_int(rng, 20_000, 600_000), d=rng.choice([12, rng.randint(3, 32)]), blocks=rng.randint(2, 5))
    else:
        c.update(n=_log_int(rng, 3000, 60_000), d=rng.randint(2, 32))
    return c


# ------------------------------------------------------------------ inputs --
def _points(case, seed):
    """A seeded Gaussian mixture with 2% background noise, shuffled: isotropic
    clusters of Zipf sizes, or anisotropic ones of equal size (the two kinds
    of the named workloads)."""
    n, d = case["n"], case["d"]
    g = torch.Generator("cuda").manual_seed(int(seed))
    k = 10 if n <= 200_000 else 30 if n <= 2_000_000 else 100
    if case["data"] == "iso":
        w = 1.0 / torch.arange(1, k + 1, device="cuda", dtype=torch.float64) ** 1.1
        edges = torch.cumsum(w / w.sum(), 0)
        lab = torch.searchsorted(edges, torch.rand(n, generator=g, device="cuda", dtype=torch.float64)).clamp_(max=k - 1)
        centre = (torch.rand(k, d, generator=g, device="cuda") * 2 - 1) * (20.0 if k < 100 else 50.0)
        std = torch.rand(k, 1, generator=g, device="cuda") * 1.5 + 0.5
        X = torch.randn(n, d, generator=g, device="cuda")
        X.mul_(std[lab]).add_(centre[lab])
    else:
        centre = torch.randn(k, d, generator=g, device="cuda") * 15.0
        axis = torch.exp(torch.rand(k, 1, d, generator=g, device="cuda") * math.log(20.0) + math.log(0.1))
        rot = torch.linalg.qr(torch.randn(k, d, d, generator=g, device="cuda").cpu())[0].cuda()
        X = torch.randn(n, d, generator=g, device="cuda")
        for c in range(k):
            s, e = n * c // k, n * (c + 1) // k
            X[s:e] = (X[s:e] * axis[c]) @ rot[c] + centre[c]
        X = X[torch.randperm(n, generator=g, device="cuda")]
    noisy = torch.rand(n, generator=g, device="cuda") < 0.02
    lo, hi = X.amin(0), X.amax(0)
    X[noisy] = lo + torch.rand(int(noisy.sum()), d, generator=g, device="cuda") * (hi - lo)
    return X


def _exact_ids(X):
    """32 nearest neighbours of every point, by rows of the distance matrix."""
    n = X.shape[0]
    nrm = (X * X).sum(1)
    out = torch.empty(n, K, dtype=torch.int64, device="cuda")
    step = max(1, (1 << 28) // n)
    for s in range(0, n, step):
        e = min(n, s + step)
        d2 = nrm[None, :] - 2.0 * (X[s:e] @ X.t())
        d2[torch.arange(e - s, device="cuda"), torch.arange(s, e, device="cuda")] = math.inf
        out[s:e] = d2.topk(K, dim=1, largest=False).indices
    return out


def _given_lists(X):
    """(n, 32, 2) int32 image of the exact lists: rows sorted by (d2, id)."""
    ids = _exact_ids(X)
    d2 = torch.zeros(ids.shape, device="cuda")
    for c in range(X.shape[1]):
        diff = X[:, c, None] - X[:, c][ids]
        d2 += diff * diff
    order = ids.argsort(1)
    ids, d2 = ids.gather(1, order), d2.gather(1, order)
    order = d2.argsort(dim=1, stable=True)
    ids, d2 = ids.gather(1, order), d2.gather(1, order)
    return torch.stack([d2.view(torch.int32), ids.to(torch.int32)], 2).contiguous()


_context = None


def _ctx():
    """The one context a program keeps (device, streams, scratch)."""
    global _context
    if _context is None:
        _context = api.Context(0)
    return _context


class _Span:
    def __init__(self, arr, shape, typestr):
        self.owner = arr
        self.__cuda_array_interface__ = dict(shape=shape, typestr=typestr, data=(arr.ptr, False), version=2)


def _tensor(arr):
    """A torch view of a DeviceArray (records as rows of int32 words)."""
    shape, typestr = arr.shape, arr.dtype.str
    if arr.dtype in (NND_ELEMENT, MST_EDGE):
        shape, typestr = (*shape, arr.dtype.itemsize // 4), "<i4"
    return torch.as_tensor(_Span(arr, shape, typestr), device="cuda")


def _resident(ctx, t, shape, dtype):
    a = ctx.empty(shape, dtype)
    _tensor(a).copy_(t)
    return a


def prepare(case, seed):
    ctx = _ctx()
    n, d, kind = case["n"], case["d"], case["kind"]
    Xt = _points(case, seed)
    s = dict(case=case, ctx=ctx, X=_resident(ctx, Xt, (n, d), np.float32))
    if kind != "fit":
        s["params"] = api.default_params(join_keep=case.get("keep", 4), nnd_iteration=case.get("iters", 6),
                                         distance_mode=2 if kind == "refined" else 0)
    if kind in ("whole", "learned", "refined", "graph", "core_sg"):
        s["out"] = dict(lists=ctx.empty((n, K), NND_ELEMENT), counts=ctx.empty((n,), np.int32),
                        core=ctx.empty((n,), np.float32), edges=ctx.empty((n - 1,), MST_EDGE))
    if kind in ("graph", "core_sg"):
        _tensor(s["out"]["lists"]).copy_(_given_lists(Xt))
    torch.cuda.synchronize()
    if kind == "learned":
        s["model"] = learned.LearnedInit(ctx, d).fit(s["X"])
    if kind == "core_sg":  # the MST of mpts = 32, as the pipeline gave it
        res = api.pipeline(ctx, s["X"], s["params"], knng_mode=4, keep_on_device=True, outputs=s["out"])
        s["mst"] = _resident(ctx, _tensor(s["out"]["edges"])[: res.n_edges], (res.n_edges,), MST_EDGE)
        torch.cuda.synchronize()
    return s


# --------------------------------------------------------------------- run --
def _lists_out(lists):
    t = _tensor(lists)
    return dict(distance=t.view(torch.float32)[..., 0], label=t[..., 1])


def _path_out(res):
    e = _tensor(res.edges)[: res.n_edges]
    return dict(lists=_lists_out(res.lists), counts=_tensor(res.counts), core=_tensor(res.core),
                ends=e[:, :2], weight=e.view(torch.float32)[:, 2], components=res.components, csr_edges=res.csr_edges)


def run(state):
    case, ctx, X = state["case"], state["ctx"], state["X"]
    kind, n = case["kind"], case["n"]
    if kind == "knng":
        return _lists_out(api.NNDescent(ctx, X, iteration=case["iters"], params=state["params"],
                                        store_result_in_device=True))
    if kind == "blocked":
        return _lists_out(api.GenLargeKNNGraph(ctx, X, case["blocks"], store_result_in_device=True))
    if kind == "fit":
        m = learned.LearnedInit(ctx, case["d"]).fit(X)
        out = [m.get_params(t) for t in range(len(m.handles))]
        m.close()
        return out
    if kind == "core_sg":
        g = api.build_CoreSG(ctx, X, state["out"]["lists"], state["mst"])
        out = {}
        for mpts in CORE_SG_MPTS:
            e, _ = api.core_sg_mst(ctx, X, state["out"]["lists"], g, mpts)
            out["mst%d" % mpts] = dict(a=e["from_node"], b=e["to_node"], weight=e["weight"])
        # the rows in buffers of their largest size (the library's stream has
        # ended with the last edges above)
        nlist = torch.zeros(2 * n * (K + 1), dtype=torch.int32, device="cuda")
        dist = torch.zeros(2 * n * (K + 1), device="cuda")
        nlist[: g.edges] = _tensor(g.nlist)[: g.edges]
        dist[: g.edges] = _tensor(g.dist)[: g.edges]
        out.update(nindex=_tensor(g.nindex), nlist=nlist, dist=dist)
        return out
    if kind == "learned":
        r = learned.pipeline_learned_checked(ctx, X, state["model"], params=state["params"], outputs=state["out"])
        return dict(_path_out(r.result), recall=r.sampled_recall, fell_back=r.fell_back)
    res = api.pipeline(ctx, X, state["params"], knng_mode=4 if kind == "graph" else 0, keep_on_device=True,
                       outputs=state["out"])
    out = _path_out(res)
    if kind == "whole" and res.components == 1:
        labels, clusters = api.get_clusters_gpu(ctx, res.edges, n, 32, keep_on_device=True)
        out.update(labels=_tensor(labels), clusters=clusters)
    return out


# -------------------------------------------------------------------- work --
def work(case):
    n, d, kind = case["n"], case["d"], case["kind"]
    points, lists, edges = 4.0 * n * d, 8.0 * K * n, 12.0 * n
    pair = 3.0 * d  # flops of one squared distance
    if kind in ("knng", "blocked"):
        return dict(bytes=points + lists, flops=n * K * pair)
    if kind == "fit":  # the subsample's rows and graph, one epoch of 8 (or 6) tables
        m = min(200_000, n)
        tables = 8 if d <= 16 else 6
        params = 32 * 128 + 128 * 128 + 128 * 16
        return dict(bytes=m * (4.0 * d + 8 * K) + tables * 4.0 * params, flops=6.0 * 3 * m * params * tables)
    if kind == "core_sg":
        csr = 2.0 * n * K * 8
        return dict(bytes=points + lists + csr + len(CORE_SG_MPTS) * (csr + edges), flops=2.0 * n * K * pair)
    total = points + lists + 8.0 * n + edges + (4.0 * n if kind == "whole" else 0.0)
    if kind == "refined":  # every pair's product once
        return dict(bytes=total, flops=float(n) * n * d)
    return dict(bytes=total, flops=n * K * pair)


# ------------------------------------------------------------------- exact --
def _dist(X, a, b):
    out = torch.empty(a.shape[0], dtype=torch.float64, device="cuda")
    step = (1 << 26) // X.shape[1]
    for s in range(0, a.shape[0], step):
        out[s:s + step] = (X[a[s:s + step]] - X[b[s:s + step]]).square().sum(1).sqrt()
    return out


def _mst(n, a, b, w):
    """Indices of the minimum spanning forest's edges (Boruvka on the order
    (w, min id, max id))."""
    lo, hi = torch.minimum(a, b), torch.maximum(a, b)
    pair = (lo * n + hi).argsort(stable=True)
    order = pair[w[pair].argsort(stable=True)]
    a, b = a[order], b[order]
    comp = torch.arange(n, device="cuda")
    edge = torch.arange(a.shape[0], device="cuda")
    chosen = []
    while True:
        ca, cb = comp[a[edge]], comp[b[edge]]
        alive = ca != cb
        if not bool(alive.any()):
            break
        edge, ca, cb = edge[alive], ca[alive], cb[alive]
        best = torch.full((n,), a.shape[0], device="cuda")
        best.scatter_reduce_(0, ca, edge, "amin")
        best.scatter_reduce_(0, cb, edge, "amin")
        roots = (best < a.shape[0]).nonzero().flatten()
        e = best[roots]
        chosen.append(e)
        other = comp[a[e]] + comp[b[e]] - roots
        to = torch.arange(n, device="cuda")
        to[roots] = other
        mutual = (to[to[roots]] == roots) & (roots < other)
        to[roots[mutual]] = roots[mutual]
        while True:
            nxt = to[to]
            if torch.equal(nxt, to):
                break
            to = nxt
        comp = to[comp]
    return order[torch.cat(chosen).unique()]


def _enhanced_graph(X, ids):
    """kNN edges and the anti-hub clique with their mutual-reachability weights."""
    n = X.shape[0]
    a = torch.arange(n, device="cuda")[:, None].expand(-1, K).reshape(-1)
    b = ids.reshape(-1)
    core = _dist(X, torch.arange(n, device="cuda"), ids[:, K - 1])
    counts = torch.bincount(b, minlength=n)
    score = counts[ids].sum(1)
    order = score.argsort(stable=True)
    order = order[counts[order].argsort(stable=True)]
    hubs = order[: math.isqrt(n)]
    p = torch.combinations(hubs, 2)
    wk = torch.maximum(core[a], core[b])
    wc = torch.maximum(torch.maximum(core[p[:, 0]], core[p[:, 1]]), _dist(X, p[:, 0], p[:, 1]))
    return torch.cat([a, p[:, 0]]), torch.cat([b, p[:, 1]]), torch.cat([wk, wc]), core


def exact(case, seed):
    kind, n = case["kind"], case["n"]
    if kind not in ("graph", "core_sg", "refined") or n > 200_000:
        return None  # approximate lists (and weights trained on them) have no value of their own
    Xt = _points(case, seed)
    X = Xt.double()
    ids = _given_lists(Xt)[..., 1].long() if kind != "refined" else None
    if ids is None:  # the true lists
        idx = torch.empty(n, K, dtype=torch.int64, device="cuda")
        dist = torch.empty(n, K, dtype=torch.float64, device="cuda")
        nrm = X.square().sum(1)
        step = max(1, (1 << 27) // n)
        for s in range(0, n, step):
            e = min(n, s + step)
            d2 = nrm[None, :] + nrm[s:e, None] - 2.0 * (X[s:e] @ X.t())
            d2[torch.arange(e - s, device="cuda"), torch.arange(s, e, device="cuda")] = math.inf
            dist[s:e], idx[s:e] = d2.topk(K, dim=1, largest=False)
        ids = idx
    a, b, w, core = _enhanced_graph(X, ids)
    tree = _mst(n, a, b, w)
    if kind == "core_sg":
        out = dict(nindex=None, nlist=None, dist=None)
        ua, ub = torch.cat([a[: n * K], a[tree]]), torch.cat([b[: n * K], b[tree]])
        du = _dist(X, ua, ub)
        for mpts in CORE_SG_MPTS:
            c = _dist(X, torch.arange(n, device="cuda"), ids[:, mpts - 1])
            wm = torch.maximum(torch.maximum(c[ua], c[ub]), du)
            out["mst%d" % mpts] = dict(a=None, b=None, weight=wm[_mst(n, ua, ub, wm)].sort().values)
        return out
    d2 = torch.zeros(n, K, dtype=torch.float64, device="cuda")
    for c in range(X.shape[1]):
        d2 += (X[:, c, None] - X[:, c][ids]).square()
    return dict(lists=dict(distance=d2, label=None), counts=None, core=core, ends=None, weight=w[tree].sort().values,
                components=None, csr_edges=None)
