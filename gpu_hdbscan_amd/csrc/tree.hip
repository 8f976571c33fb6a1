// Hierarchy and labels on the GPU: single linkage over the sorted MST edges
// -> condensed tree -> stability -> EOM selection -> labels, with the
// semantics of HDBSCAN/trees/tree.cu:171-746 as the host version
// (labels.cpp) implements them, quirks included (lambda = (float)INT_MAX for
// a zero weight, tree.cu:308-313; a point labelled only when its lambda is
// strictly above its cluster's birth lambda, tree.cu:609-618).
//
// 1. Linkage (build_Linkage_tree, tree.cu:171-202).  Node n + i merges the
//    components of edge i's two ends as they stand before edge i; its
//    children are the nodes that root those components.  Instead of a
//    sequential union-find, every edge end is a query (end vertex, time i)
//    answered by halving the edge range: at bit b (highest first) the
//    queries of edges whose index has bit b set move from the start of
//    their segment to its middle -- the edges of the segment's first half
//    join the components they touch (connected components over component
//    names, one union-find on the GPU per level), and a query whose
//    component is among them takes the merged component, its last edge (the
//    node that roots it) and its point count.  Three launches per level down
//    to segments of 1024 edges, which finish their levels in LDS.  Bound by
//    the random reads of the top levels.  Replaced one radix sort of all
//    queries by (segment, component) per level, which cost 45 launches and
//    4-6 passes over them each; path and labels together 6.94 -> 3.71 ms at
//    5k x 12, 12.9 -> 8.4 ms at 100k and 531 -> 491 ms at 10M.
// 2. The condensed tree (build_Condensed_tree, tree.cu:255-442) follows from
//    the linkage tree without a traversal: a node is processed when it is
//    the root or holds at least mpts points; a processed node whose two
//    children both hold mpts points is a split, and its children start new
//    clusters, numbered in the level order of the splits (depth, then
//    preorder); every other processed node continues its cluster, and the
//    points of its small children leave that cluster at its lambda.  Depths,
//    preorder numbers and cluster starts come from one pointer jumping over
//    16-byte node records, whose log2(m) rounds are queued without a host
//    round trip.
// 3. Stability (compute_stability, tree.cu:444-528): per cluster, the terms
//    (lambda - birth) * size are added in the order of the condensed list
//    (the cluster's nodes top-down, then its two split children), and the
//    FP32 sums are those of the host's sequential loop, bit for bit.
// 4. EOM selection (get_clusters, tree.cu:627-746) runs on the host over the
//    cluster tree (one entry per cluster); labelling (do_labelling,
//    tree.cu:569-625) is one GPU pass over the points.
#include <algorithm>
#include <climits>
#include <cstring>
#include <vector>

#include "hdb_internal.hpp"

namespace hdb {

namespace {

constexpr int kRepBits = 26;  // n < 2^26

// ---------------------------------------------------------------- linkage --
// A component of a segment is named by its lowest end: the smallest query q
// (end q & 1 of edge q >> 1) of the segment that lies in it.  Names of a
// segment therefore fall in its own index range, so every per-component
// array is read near the segment's own positions once segments are small,
// and no sort, scan or count of components is needed.  top and sz hold, at
// a component's name, the node that roots it and its point count.
constexpr int kLkBits = 10;             // segments of 1024 edges are finished in LDS
constexpr int kLkEdges = 1 << kLkBits;  // one per thread of k_lk_local
constexpr int32_t kNoName = INT_MAX;

// The find is ECL-CC's (Jaiganesh and Burtscher 2018) with intermediate
// pointer jumping.  What it relies on: every value an entry ever holds is one
// of the element's ancestors, and smaller than the element unless it is a
// root; a root changes only by the hook's compare-and-swap at device scope;
// and an element, once hooked, is never a root again.  An entry may rise: a
// path-halving store of an earlier read, or the write-back of another XCD's
// L2, can replace a lower ancestor by a higher one, and a cached load can
// return an old value.  Both still give an ancestor, so finds end, at a root
// or at an element that was one; the swap tells which.  So finds use plain
// cached loads and stores (kernels that follow see every hook).
__device__ __forceinline__ int32_t uf_load(const int32_t* uf, int32_t x) {
  return __hip_atomic_load(uf + x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
}

// Root of x, as far as this XCD knows.
__device__ __forceinline__ int32_t uf_find(int32_t* uf, int32_t x) {
  int32_t cur = uf_load(uf, x);
  if (cur != x) {
    int32_t next, prev = x;
    while (cur > (next = uf_load(uf, cur))) {
      __hip_atomic_store(uf + prev, next, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
      prev = cur;
      cur = next;
    }
  }
  return cur;
}

// The larger root c is hooked under the smaller.  A failed swap returns what
// c points to by now, a smaller element, and the search goes on from there:
// every failure moves down, so the loop ends whatever the caches hold.
__device__ __forceinline__ void uf_join(int32_t* uf, int32_t a, int32_t c) {
  while (true) {
    a = uf_find(uf, a);
    c = uf_find(uf, c);
    if (a == c) return;
    if (a > c) {
      const int32_t t = a;
      a = c;
      c = t;
    }
    const int32_t was = atomicCAS(&uf[c], c, a);
    if (was == c) return;
    c = was;
  }
}

// *p = min(*p, v), skipping the atomic when *p (which only falls, so a stale
// read only costs an atomic) is already there: the members of a component
// arrive roughly in ascending order, so a large one takes few atomics.
__device__ __forceinline__ void lower_to(int32_t* p, int32_t v) {
  if (v < __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMin(p, v);
}

// The union-find and the per-component accumulators of one level: names of
// the two halves' components, last first-half edge, point count.
struct LkLevel {
  int32_t *uf, *rep_l, *rep_r, *cmax, *csize;
};

__device__ __forceinline__ void lk_reset(const LkLevel& a, int64_t q) {
  a.uf[q] = static_cast<int32_t>(q);
  a.rep_l[q] = kNoName;
  a.rep_r[q] = kNoName;
  a.cmax[q] = -1;
  a.csize[q] = 0;
}

// first[v] = the lowest end at point v, through the level's rep_l (2m >= n
// entries for m >= 1); an end outside [0, n) marks the input bad.
__global__ void k_lk_first(const hdb_mst_edge* __restrict__ e, int64_t m, int64_t n, int32_t* __restrict__ first,
                           int32_t* __restrict__ bad) {
  const int64_t q = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (q >= 2 * m) return;
  const int32_t v = (q & 1) ? e[q >> 1].to_node : e[q >> 1].from_node;
  if (v < 0 || v >= n) *bad = 1;
  else lower_to(first + v, static_cast<int32_t>(q));
}

// Also clears the parents that k_tr_nodes fills in (par: m, leaf_par: n <= 2m).
__global__ void k_lk_init(const hdb_mst_edge* __restrict__ e, int64_t m, int64_t n, const int32_t* __restrict__ first,
                          int32_t* __restrict__ vid, int32_t* __restrict__ top, int32_t* __restrict__ sz, LkLevel a,
                          int32_t* __restrict__ par, int32_t* __restrict__ leaf_par) {
  const int64_t q = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (q >= 2 * m) return;
  if (q < m) par[q] = -2;
  if (q < n) leaf_par[q] = -2;
  const int32_t v = (q & 1) ? e[q >> 1].to_node : e[q >> 1].from_node;
  vid[q] = v >= 0 && v < n ? first[v] : static_cast<int32_t>(q);
  top[q] = v;
  sz[q] = 1;
  lk_reset(a, q);
}

// Combines updates per component in an LDS table before the global atomics:
// at every level a few huge components take most of them, and same-address
// atomics serialise (a quarter of a million on one name made the union take
// 340 us a level at 1M edges).  Linear probing over four slots, one
// global atomic per root and block; a root that finds no slot goes to the
// global atomic directly.  Max, min and integer sums do not depend on the
// order.
constexpr int kAggSlots = 1024;
enum class Agg { kMin, kMax, kSum };

template <Agg OP>
__device__ __forceinline__ void agg_apply(int32_t* p, int32_t v) {
  if (OP == Agg::kMin) atomicMin(p, v);
  else if (OP == Agg::kMax) atomicMax(p, v);
  else atomicAdd(p, v);
}

template <Agg OP>
struct AggTable {
  int32_t keys[kAggSlots], acc[kAggSlots];
  __device__ __forceinline__ void init() {
    for (int s = threadIdx.x; s < kAggSlots; s += 256) {
      keys[s] = -1;
      acc[s] = OP == Agg::kMin ? INT_MAX : OP == Agg::kMax ? -1 : 0;
    }
  }
  __device__ __forceinline__ void put(int32_t* glob, int32_t root, int32_t v) {
    uint32_t h = static_cast<uint32_t>(root) * 0x9E3779B1u;
    h >>= 22;  // 10 bits: kAggSlots
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const int slot = static_cast<int>((h + p) & (kAggSlots - 1));
      const int32_t k = atomicCAS(&keys[slot], -1, root);
      if (k == -1 || k == root) {
        agg_apply<OP>(&acc[slot], v);
        return;
      }
    }
    agg_apply<OP>(&glob[root], v);
  }
  __device__ __forceinline__ void flush(int32_t* glob) {
    for (int s = threadIdx.x; s < kAggSlots; s += 256)
      if (keys[s] >= 0) agg_apply<OP>(&glob[keys[s]], acc[s]);
  }
};

// Level b, first kernel: the first-half edges (bit b clear) of every segment
// join their ends' components, and the components they touch get their name
// in the first half.  `items` edges per thread.
__global__ __launch_bounds__(256) void k_lk_union(int64_t m, int b, int items, const int32_t* __restrict__ vid,
                                                  LkLevel a) {
  __shared__ AggTable<Agg::kMin> name;
  name.init();
  __syncthreads();
  const int64_t base = static_cast<int64_t>(blockIdx.x) * (256 * items);
  for (int k = 0; k < items; ++k) {
    const int64_t i = base + k * 256 + threadIdx.x;
    if (i >= m) break;
    if ((i >> b) & 1) continue;
    const int32_t v0 = vid[2 * i], v1 = vid[2 * i + 1];
    name.put(a.rep_l, v0, static_cast<int32_t>(2 * i));
    name.put(a.rep_l, v1, static_cast<int32_t>(2 * i + 1));
    uf_join(a.uf, v0, v1);
  }
  __syncthreads();
  name.flush(a.rep_l);
}

// Per merged component: its last (highest) first-half edge, its point count
// (each component a first-half edge touches counts once, at its name) and
// its name in the second half.
__global__ __launch_bounds__(256) void k_lk_merge(int64_t m, int b, int items, int32_t* __restrict__ vid,
                                                  const int32_t* __restrict__ sz, LkLevel a) {
  __shared__ AggTable<Agg::kMax> last;
  __shared__ AggTable<Agg::kSum> count;
  __shared__ AggTable<Agg::kMin> name;
  last.init();
  count.init();
  name.init();
  __syncthreads();
  const int64_t base = static_cast<int64_t>(blockIdx.x) * (256 * items);
  for (int k = 0; k < items; ++k) {
    const int64_t i = base + k * 256 + threadIdx.x;
    if (i >= m) break;
    const int32_t v0 = vid[2 * i], v1 = vid[2 * i + 1];
    const int32_t r0 = uf_find(a.uf, v0);
    const int32_t q0 = static_cast<int32_t>(2 * i);
    if (!((i >> b) & 1)) {
      last.put(a.cmax, r0, static_cast<int32_t>(i));
      const int32_t s = (a.rep_l[v0] == q0 ? sz[v0] : 0) + (a.rep_l[v1] == q0 + 1 ? sz[v1] : 0);
      if (s) count.put(a.csize, r0, s);
    } else {
      const int32_t r1 = uf_find(a.uf, v1);
      vid[2 * i] = r0;
      vid[2 * i + 1] = r1;
      name.put(a.rep_r, r0, q0);
      name.put(a.rep_r, r1, q0 + 1);
    }
  }
  __syncthreads();
  last.flush(a.cmax);
  count.flush(a.csize);
  name.flush(a.rep_r);
}

// Every end takes its component's name in its half, and the component's
// named end its root node and point count: unchanged in the first half and
// for a component no first-half edge touched, else the last first-half
// edge's node and the merged count.  The next level's arrays are reset.
__global__ void k_lk_rename(int64_t m, int b, int64_t n, int32_t* __restrict__ vid, const int32_t* __restrict__ top,
                            const int32_t* __restrict__ sz, int32_t* __restrict__ top2, int32_t* __restrict__ sz2,
                            LkLevel a, LkLevel next) {
  const int64_t q = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (q >= 2 * m) return;
  const int32_t v = vid[q];
  const bool second = ((q >> (b + 1)) & 1) != 0;
  const int32_t nv = second ? a.rep_r[v] : a.rep_l[v];
  vid[q] = nv;
  if (nv == static_cast<int32_t>(q)) {
    const int32_t last = second ? a.cmax[v] : -1;
    top2[q] = last >= 0 ? static_cast<int32_t>(n + last) : top[v];
    sz2[q] = last >= 0 ? a.csize[v] : sz[v];
  }
  lk_reset(next, q);
}

// The remaining levels of one segment of up to 1024 edges in LDS (56 KB, two
// blocks per CU), the same three steps per level between block barriers; one
// edge per thread.  Doing the last ten levels here is what keeps the
// linkage at 3 launches and one pass over the edges per remaining level: at
// 5k points three levels are left.  Writes top and sz of each end itself.
__global__ __launch_bounds__(kLkEdges) void k_lk_local(int64_t m, int levels, int64_t n,
                                                       const int32_t* __restrict__ vid,
                                                       const int32_t* __restrict__ top,
                                                       const int32_t* __restrict__ sz, int32_t* __restrict__ top_end,
                                                       int32_t* __restrict__ sz_end) {
  constexpr int Q = 2 * kLkEdges;
  __shared__ int32_t uf[Q], rep_l[Q], rep_r[Q], cmax[Q], csize[Q], s_top[Q], s_sz[Q];
  const int t = static_cast<int>(threadIdx.x);
  const int64_t i0 = static_cast<int64_t>(blockIdx.x) << kLkBits, q0 = 2 * i0;
  const bool live = i0 + t < m;
  int32_t v[2] = {0, 0};
  for (int k = 0; k < 2; ++k) {
    const int64_t q = q0 + 2 * t + k;
    if (live) {
      v[k] = static_cast<int32_t>(vid[q] - q0);
      s_top[2 * t + k] = top[q];
      s_sz[2 * t + k] = sz[q];
    }
  }
  for (int b = levels - 1; b >= 0; --b) {
    for (int x = t; x < Q; x += kLkEdges) {
      uf[x] = x;
      rep_l[x] = rep_r[x] = kNoName;
      cmax[x] = -1;
      csize[x] = 0;
    }
    __syncthreads();
    const bool second = ((t >> b) & 1) != 0;
    if (live && !second) {
      atomicMin(&rep_l[v[0]], 2 * t);
      atomicMin(&rep_l[v[1]], 2 * t + 1);
      uf_join(uf, v[0], v[1]);
    }
    __syncthreads();
    if (live) {
      const int32_t r = uf_find(uf, v[0]);
      if (!second) {
        atomicMax(&cmax[r], t);
        const int32_t s = (rep_l[v[0]] == 2 * t ? s_sz[v[0]] : 0) + (rep_l[v[1]] == 2 * t + 1 ? s_sz[v[1]] : 0);
        if (s) atomicAdd(&csize[r], s);
      } else {
        v[0] = r;
        v[1] = uf_find(uf, v[1]);
        atomicMin(&rep_r[v[0]], 2 * t);
        atomicMin(&rep_r[v[1]], 2 * t + 1);
      }
    }
    __syncthreads();
    int32_t nt[2] = {0, 0}, ns[2] = {0, 0};
    bool mine[2] = {false, false};
    if (live) {
      for (int k = 0; k < 2; ++k) {
        const int32_t x = v[k];
        const int32_t nv = second ? rep_r[x] : rep_l[x];
        mine[k] = nv == 2 * t + k;
        if (mine[k]) {
          const int32_t last = second ? cmax[x] : -1;
          nt[k] = last >= 0 ? static_cast<int32_t>(n + i0 + last) : s_top[x];
          ns[k] = last >= 0 ? csize[x] : s_sz[x];
        }
        v[k] = nv;
      }
    }
    __syncthreads();
    for (int k = 0; k < 2; ++k)
      if (mine[k]) {
        s_top[2 * t + k] = nt[k];
        s_sz[2 * t + k] = ns[k];
      }
    __syncthreads();
  }
  __syncthreads();
  if (live)
    for (int k = 0; k < 2; ++k) {
      top_end[q0 + 2 * t + k] = s_top[v[k]];
      sz_end[q0 + 2 * t + k] = s_sz[v[k]];
    }
}

// ------------------------------------------------------- condensed tree --
// Internal node i = node n + i.  par[i]: parent's internal index (-1 at
// the root); lam[i]: 1 / weight rounded from FP64, (float)INT_MAX for 0.
// A child is a point or an earlier node: anything else marks the linkage
// inconsistent (*bad), and nothing is written through it.
__global__ void k_tr_nodes(const hdb_mst_edge* __restrict__ e, int64_t m, int64_t n, const int32_t* __restrict__ top,
                           const int32_t* __restrict__ sz, int32_t* __restrict__ left, int32_t* __restrict__ right,
                           int32_t* __restrict__ nsize, int32_t* __restrict__ par, int32_t* __restrict__ leaf_par,
                           float* __restrict__ lam, int32_t* __restrict__ bad) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= m) return;
  const int32_t l = top[2 * i], r = top[2 * i + 1];
  if (l < 0 || r < 0 || l >= n + i || r >= n + i || l == r) {
    *bad = 1;
    left[i] = right[i] = 0;
    nsize[i] = 0;
    lam[i] = 0.0f;
    return;
  }
  left[i] = l;
  right[i] = r;
  nsize[i] = sz[2 * i] + sz[2 * i + 1];
  if (l >= n) par[l - n] = static_cast<int32_t>(i);
  else leaf_par[l] = static_cast<int32_t>(i);
  if (r >= n) par[r - n] = static_cast<int32_t>(i);
  else leaf_par[r] = static_cast<int32_t>(i);
  const float w = e[i].weight;
  lam[i] = w > 0.0f ? static_cast<float>(1.0 / static_cast<double>(w)) : static_cast<float>(INT_MAX);
  if (i == m - 1) par[i] = -1;
}

__device__ __forceinline__ int32_t node_size(int32_t x, int64_t n, const int32_t* nsize) {
  return x >= n ? nsize[x - n] : 1;
}

// State of a node in the pointer jumping: anc, the ancestor reached (-1 past
// the root); the sums of depth and preorder steps up to it; and link, the
// node searched for on the way up (its cluster's start for a processed node,
// the highest small ancestor-or-self for a small one) or anc while that
// lies further up.  One 16-byte record, so a round is one gather per node.
struct __attribute__((aligned(16))) TrRec {
  int32_t anc, depth, pre, link;
};

constexpr uint8_t kProc = 1, kSplit = 2;

// Per internal node: processed (the root, or at least mpts points), split
// (both children hold mpts points), the points of its small children
// (they leave its cluster at its lambda), and its record before any jump:
// its parent, one step down, its preorder increment.  Split nodes are
// appended to `splits` (in any order).  Every node but the root must have a
// later node as parent, every point a node; otherwise *bad is set and the
// node treated as a root, so that the passes below stay in bounds.
__global__ void k_tr_classify(int64_t m, int64_t n, int mpts, const int32_t* __restrict__ left,
                              const int32_t* __restrict__ right, const int32_t* __restrict__ nsize,
                              const int32_t* __restrict__ par, const int32_t* __restrict__ leaf_par,
                              uint8_t* __restrict__ flags, int32_t* __restrict__ cnt, TrRec* __restrict__ rec,
                              int32_t* __restrict__ splits, int32_t* __restrict__ nsplit, int32_t* __restrict__ bad) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) {
    const int32_t lp = leaf_par[i];
    if (lp < 0 || lp >= m) *bad = 1;
  }
  bool sp = false;
  if (i < m) {
    int32_t p = par[i];
    if (i != m - 1 && (p <= i || p >= m)) {
      *bad = 1;
      p = -1;
    }
    const bool root = p < 0;
    const bool pr = root || nsize[i] >= mpts;
    const int32_t ls = node_size(left[i], n, nsize), rs = node_size(right[i], n, nsize);
    sp = pr && ls >= mpts && rs >= mpts;
    flags[i] = (pr ? kProc : 0) | (sp ? kSplit : 0);
    cnt[i] = pr ? (ls < mpts ? ls : 0) + (rs < mpts ? rs : 0) : 0;
    TrRec r{p, 0, 0, static_cast<int32_t>(i)};
    if (!root) {
      const int32_t pl = node_size(left[p], n, nsize);
      const bool is_right = right[p] == static_cast<int32_t>(n + i);
      r.depth = 1;
      r.pre = 1 + (is_right ? 2 * pl - 1 : 0);
      // a search ends here at a cluster start (a child of a split) and at a
      // small node under a processed one
      const bool ppr = p == m - 1 || nsize[p] >= mpts;
      const bool psp = ppr && pl >= mpts && node_size(right[p], n, nsize) >= mpts;
      if (pr ? !psp : !ppr) r.link = p;
    }
    rec[i] = r;
  }
  const uint64_t bal = __ballot(sp);
  if (bal) {
    const unsigned lane = __lane_id();
    int32_t base = 0;
    if (lane == static_cast<unsigned>(__builtin_ctzll(bal))) base = atomicAdd(nsplit, __popcll(bal));
    base = __shfl(base, __builtin_ctzll(bal));
    if (sp) splits[base + __popcll(bal & lanemask_lt())] = static_cast<int32_t>(i);
  }
}

// One round: anc doubles its reach.  link, while it equals anc, takes what
// anc's record found (or its anc); once it differs it is final.
__global__ void k_tr_jump(int64_t m, const TrRec* __restrict__ in, TrRec* __restrict__ out) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= m) return;
  TrRec r = in[i];
  if (r.anc >= 0) {
    const TrRec a = in[r.anc];
    if (r.link == r.anc) r.link = a.link;
    r.anc = a.anc;
    r.depth += a.depth;
    r.pre += a.pre;
  }
  out[i] = r;
}

// Up to kSplitSmall splits: ranked by (depth, preorder), their level order,
// by one block in LDS.  The left child of the split of rank k starts
// cluster 1 + 2k, the right one 2 + 2k (the root's cluster is 0); ids
// relative to n.  One launch where a radix sort takes over fifty.
constexpr int kSplitSmall = 2048;
__global__ __launch_bounds__(1024) void k_tr_split_rank_small(int S2, const int32_t* __restrict__ splits,
                                                              const TrRec* __restrict__ rec,
                                                              int32_t* __restrict__ srank) {
  __shared__ uint64_t key[kSplitSmall];
  __shared__ int32_t node[kSplitSmall];
  int p = 1;
  while (p < S2) p <<= 1;
  for (int t = threadIdx.x; t < p; t += 1024) {
    key[t] = kKeyMax;
    node[t] = -1;
    if (t < S2) {
      const int32_t i = splits[t];
      const TrRec r = rec[i];
      key[t] = (static_cast<uint64_t>(static_cast<uint32_t>(r.depth)) << 32) | static_cast<uint32_t>(r.pre);
      node[t] = i;
    }
  }
  __syncthreads();
  for (int k = 2; k <= p; k <<= 1)
    for (int j = k >> 1; j > 0; j >>= 1) {
      for (int t = threadIdx.x; t < p; t += 1024) {
        const int o = t ^ j;
        if (o > t && (key[t] > key[o]) == ((t & k) == 0)) {
          const uint64_t x = key[t];
          key[t] = key[o];
          key[o] = x;
          const int32_t y = node[t];
          node[t] = node[o];
          node[o] = y;
        }
      }
      __syncthreads();
    }
  for (int t = threadIdx.x; t < S2; t += 1024) srank[node[t]] = t;
}

__global__ void k_tr_split_keys(int64_t S2, const int32_t* __restrict__ splits, const TrRec* __restrict__ rec,
                                uint64_t* __restrict__ keys, uint32_t* __restrict__ vals) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= S2) return;
  const int32_t i = splits[t];
  const TrRec r = rec[i];
  keys[t] = (static_cast<uint64_t>(static_cast<uint32_t>(r.depth)) << 32) | static_cast<uint32_t>(r.pre);
  vals[t] = static_cast<uint32_t>(i);
}

__global__ void k_tr_split_rank(int64_t S2, const uint32_t* __restrict__ vals, int32_t* __restrict__ srank) {
  const int64_t k = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (k < S2) srank[vals[k]] = static_cast<int32_t>(k);
}

// Relative cluster id of the cluster that starts at node s.
__device__ __forceinline__ int32_t cluster_of(int32_t s, int64_t n, const int32_t* __restrict__ par,
                                              const int32_t* __restrict__ left, const int32_t* __restrict__ srank) {
  const int32_t p = par[s];
  if (p < 0) return 0;
  return (left[p] == static_cast<int32_t>(n + s) ? 1 : 2) + 2 * srank[p];
}

// Cluster of every processed node (relative id) and, per cluster, its birth
// lambda, parent cluster and length.  A cluster's nodes are one path down
// from its start (a processed node that does not split has at most one child
// of mpts points), so a node's position on it is a difference of depths and
// its last node gives the length.  na is cleared for k_tr_addend_count.
__global__ void k_tr_clusters(int64_t m, int64_t n, int mpts, const uint8_t* __restrict__ flags,
                              const TrRec* __restrict__ rec, const int32_t* __restrict__ par,
                              const int32_t* __restrict__ left, const int32_t* __restrict__ right,
                              const int32_t* __restrict__ nsize, const int32_t* __restrict__ srank,
                              const float* __restrict__ lam, int32_t* __restrict__ cid, int32_t* __restrict__ pos,
                              float* __restrict__ birth, int32_t* __restrict__ cparent, int32_t* __restrict__ clen,
                              int32_t* __restrict__ na) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= m) return;
  na[i] = 0;
  const uint8_t f = flags[i];
  if (!(f & kProc)) {
    cid[i] = -1;
    return;
  }
  const TrRec r = rec[i];
  const int32_t c = cluster_of(r.link, n, par, left, srank);
  const int32_t at = r.depth - rec[r.link].depth;
  cid[i] = c;
  pos[i] = at;
  if (r.link == static_cast<int32_t>(i)) {
    const int32_t p = par[i];
    birth[c] = p < 0 ? 0.0f : lam[p];
    cparent[c] = p < 0 ? -1 : cluster_of(rec[p].link, n, par, left, srank);
  }
  if ((f & kSplit) || (node_size(left[i], n, nsize) < mpts && node_size(right[i], n, nsize) < mpts)) clen[c] = at + 1;
}

// Stability: per cluster, the addends of the host version in its order --
// for each of the cluster's nodes top-down, (lambda - birth) once per point
// that leaves there, then (lambda - birth) * size for each child of a split
// -- are laid out flat (one count per path position, cluster after cluster, a
// scan, then each node writes its addends), and the sums below add them in
// that order.
__global__ void k_tr_addend_count(int64_t m, const uint8_t* __restrict__ flags, const int32_t* __restrict__ cid,
                                  const int32_t* __restrict__ pos, const int64_t* __restrict__ cbeg,
                                  const int32_t* __restrict__ cnt, int32_t* __restrict__ na) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= m) return;
  const uint8_t f = flags[i];
  if (f & kProc) na[cbeg[cid[i]] + pos[i]] = cnt[i] + ((f & kSplit) ? 2 : 0);
}

__global__ void k_tr_addends(int64_t m, int64_t n, const uint8_t* __restrict__ flags, const int32_t* __restrict__ cid,
                             const int32_t* __restrict__ pos, const int64_t* __restrict__ cbeg,
                             const int32_t* __restrict__ cnt, const float* __restrict__ lam,
                             const int32_t* __restrict__ left, const int32_t* __restrict__ right,
                             const int32_t* __restrict__ nsize, const float* __restrict__ birth,
                             const int64_t* __restrict__ off, float* __restrict__ add) {
#pragma clang fp contract(off)  // products rounded on their own, as on the host
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= m) return;
  const uint8_t f = flags[i];
  if (!(f & kProc)) return;
  const int32_t c = cid[i];
  const float term = lam[i] - birth[c];
  float* dst = add + off[cbeg[c] + pos[i]];
  const int k = cnt[i];
  for (int r = 0; r < k; ++r) dst[r] = term;
  if (f & kSplit) {
    dst[k] = term * static_cast<float>(node_size(left[i], n, nsize));
    dst[k + 1] = term * static_cast<float>(node_size(right[i], n, nsize));
  }
}

// s += t[0] + ... in order, one rounding per add (the host's sequential
// loop): lanes load 64 addends at a time, the wave takes them lane by lane.
__device__ __forceinline__ float add_in_order(float s, const float* __restrict__ add, int64_t t0, int64_t t1) {
  const unsigned lane = __lane_id();
  for (; t0 < t1; t0 += 64) {
    // past the end, +0: adding it leaves s as it is (s >= 0 throughout)
    const float v = t0 + lane < t1 ? add[t0 + lane] : 0.0f;
    const int32_t vb = __float_as_int(v);
#pragma unroll
    for (int j = 0; j < 64; ++j) s += __int_as_float(__builtin_amdgcn_readlane(vb, j));
  }
  return s;
}

constexpr int64_t kStabShort = 1024;  // addends a wave adds one by one

// Clusters of at most kStabShort addends: one wave each.
__global__ __launch_bounds__(256) void k_tr_stability(int64_t S, const int64_t* __restrict__ cbeg,
                                                      const int64_t* __restrict__ off, const float* __restrict__ add,
                                                      float* __restrict__ stab) {
  const int64_t c = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (c >= S) return;
  const int64_t a0 = off[cbeg[c]], a1 = off[cbeg[c + 1]];
  if (a1 - a0 > kStabShort) return;
  const float s = add_in_order(0.0f, add, a0, a1);
  if (__lane_id() == 0) stab[c] = s;
}

// Longer clusters, bit for bit the same sequential FP32 sum, in parallel.
// While s stays in one binade [2^e, 2^(e+1)) it is an integer multiple S of
// u = 2^(e-23), and adding t >= 0 moves it by RNE(S + t/u) - S units.  That
// step depends on S only through its parity (which decides ties), so a run
// of addends is a map (parity of S) -> (units added), and such maps compose
// associatively.  The step for an even and an odd S is read off the bits of
// 2^e + t and 2^e + u + t, which the hardware rounds the same way.  Each of
// the block's 16 waves composes the map of 1024 addends; the maps are then
// applied in order until one would leave the binade (or its addends are not
// all finite and >= 0), whose 1024 addends are added one by one.  s leaves at
// most ~log2(addends) binades, so nearly all the work is parallel: the
// serial chain took 8 cycles per addend, 28.7 ms for the largest cluster of
// 10M x 12; this kernel takes 0.84 ms there.
constexpr int kStabWaves = 16;
constexpr uint32_t kStabBig = 1u << 25;  // more units than any binade holds

__global__ __launch_bounds__(kStabWaves * 64) void k_tr_stability_long(
    int64_t S, const int64_t* __restrict__ cbeg, const int64_t* __restrict__ off, const float* __restrict__ add,
    float* __restrict__ stab) {
  __shared__ uint32_t s_even[kStabWaves], s_odd[kStabWaves];
  __shared__ float s_sum;
  const unsigned lane = __lane_id();
  const int w = static_cast<int>(threadIdx.x >> 6);
  for (int64_t c = blockIdx.x; c < S; c += gridDim.x) {
    const int64_t a0 = off[cbeg[c]], a1 = off[cbeg[c + 1]];
    if (a1 - a0 <= kStabShort) continue;  // uniform across the block
    // the first addends one by one, up to a 16-byte aligned position
    int64_t pos = a0 + 1024 - (a0 & 3);
    if (w == 0) {
      const float s = add_in_order(0.0f, add, a0, pos);
      if (lane == 0) s_sum = s;
    }
    __syncthreads();
    float s = s_sum;
    while (pos < a1) {  // uniform
      uint32_t sb = __float_as_uint(s);
      const uint32_t base = sb & 0xFF800000u;
      const float b0 = __uint_as_float(base), b1 = __uint_as_float(base | 1u);
      // units added by this lane's 16 addends from an even (e) and odd (o) S
      uint32_t e = 0, o = 0;
      const int64_t p0 = pos + w * 1024 + lane * 16;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int64_t p = p0 + 4 * q;
        float t[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        if (p + 3 < a1) {
          const float4 v = *reinterpret_cast<const float4*>(add + p);
          t[0] = v.x, t[1] = v.y, t[2] = v.z, t[3] = v.w;
        } else {
#pragma unroll
          for (int k = 0; k < 4; ++k)
            if (p + k < a1) t[k] = add[p + k];
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const bool ok = t[k] >= 0.0f && t[k] < __uint_as_float(0x7F800000u);
          const uint32_t i0 = ok ? __float_as_uint(b0 + t[k]) - base : kStabBig;
          const uint32_t i1 = ok ? __float_as_uint(b1 + t[k]) - (base | 1u) : kStabBig;
          e = min(e + min((e & 1u) ? i1 : i0, kStabBig), kStabBig);
          o = min(o + min((o & 1u) ? i0 : i1, kStabBig), kStabBig);
        }
      }
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {  // lane i takes lanes [i, i + 2d)
        const uint32_t re = __shfl_down(e, d), ro = __shfl_down(o, d);
        e = min(e + ((e & 1u) ? ro : re), kStabBig);
        o = min(o + ((o & 1u) ? re : ro), kStabBig);
      }
      if (lane == 0) {
        s_even[w] = e;
        s_odd[w] = o;
      }
      __syncthreads();
      // s must be a normal number: 0, denormals and infinities go one by one
      const uint32_t ex = (sb >> 23) & 0x1FFu;
      const bool normal = ex >= 1u && ex <= 254u;
      int k = 0;
      for (; k < kStabWaves && normal; ++k) {
        const uint32_t inc = (sb & 1u) ? s_odd[k] : s_even[k];
        if (inc >= 0x800000u - (sb & 0x7FFFFFu)) break;
        sb += inc;
      }
      s = __uint_as_float(sb);
      pos += static_cast<int64_t>(k) * 1024;
      if (k < kStabWaves && pos < a1) {  // uniform
        if (w == 0) {
          const float r = add_in_order(s, add, pos, pos + 1024 < a1 ? pos + 1024 : a1);
          if (lane == 0) s_sum = r;
        }
        pos += 1024;
        __syncthreads();
        s = s_sum;
      }
      __syncthreads();
    }
    if (threadIdx.x == 0) stab[c] = s;
    __syncthreads();
  }
}

// Point p leaves at its lowest processed ancestor: its parent, or the parent
// of the highest small node above it.  Its label is its cluster's selected
// ancestor's, when its lambda is strictly above that cluster's birth.
__global__ void k_tr_label(int64_t n, const int32_t* __restrict__ leaf_par, const uint8_t* __restrict__ flags,
                           const TrRec* __restrict__ rec, const int32_t* __restrict__ par,
                           const int32_t* __restrict__ cid, const float* __restrict__ lam,
                           const int32_t* __restrict__ clab, const float* __restrict__ cbirth,
                           int32_t* __restrict__ labels) {
  const int64_t p = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (p >= n) return;
  int32_t f = leaf_par[p];
  if (!(flags[f] & kProc)) f = par[rec[f].link];
  const int32_t c = cid[f];
  const int32_t l = clab[c];
  labels[p] = (l >= 0 && lam[f] > cbirth[c]) ? l : -1;
}

__global__ void k_tr_fill_neg(int32_t* __restrict__ p, int64_t n) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) p[i] = -1;
}

}  // namespace

int labels_gpu(hdb_ctx* ctx, const hdb_mst_edge* edges, int64_t m, int64_t n, int mpts, int32_t* labels,
               int32_t* clusters_out) {
  if (!labels || n < 1 || mpts < 2 || m < 0 || m > n - 1 || (m > 0 && !edges))
    return ctx->fail(HDB_EINVAL, "bad labels arguments");
  if (n >= (static_cast<int64_t>(1) << kRepBits)) return ctx->fail(HDB_EINVAL, "n must be below 2^26 (67,108,864)");
  if (clusters_out) *clusters_out = 0;
  if (m != n - 1) return ctx->fail(HDB_EDISCONNECTED, "the hierarchy needs the n - 1 edges of a spanning tree");
  Stage st(ctx, "labels_gpu");
  if (n == 1) {
    hipLaunchKernelGGL(k_tr_fill_neg, dim3(1), dim3(64), 0, ctx->stream, labels, n);
    HDB_LAUNCHED();
    return HDB_OK;
  }
  const int64_t Q = 2 * m;
  // node arrays and controls {bad, number of splits}
  int32_t *left, *right, *nsize, *par, *leaf_par, *cnt, *cid, *pos, *srank, *splits, *ctrl;
  float* lam;
  HDB_CALL(scratch_t(ctx, kSlotMstParent, 10 * m + n + 8, &ctrl));
  left = ctrl + 8;
  right = left + m;
  nsize = right + m;
  par = nsize + m;
  cnt = par + m;
  cid = cnt + m;
  pos = cid + m;
  srank = pos + m;
  splits = srank + m;
  lam = reinterpret_cast<float*>(splits + m);
  leaf_par = reinterpret_cast<int32_t*>(lam + m);
  int32_t *bad = ctrl, *nsplit = ctrl + 1;
  HDB_CALL(fill_u64(ctx, reinterpret_cast<uint64_t*>(ctrl), 1, 0));
  // ---- linkage
  int32_t *vid, *top, *sz, *top2, *sz2, *lv;
  HDB_CALL(scratch_t(ctx, kSlotMisc0, 5 * Q, &vid));
  top = vid + Q;
  sz = top + Q;
  top2 = sz + Q;
  sz2 = top2 + Q;
  HDB_CALL(scratch_t(ctx, kSlotMisc1, 10 * Q, &lv));
  LkLevel cur{lv, lv + Q, lv + 2 * Q, lv + 3 * Q, lv + 4 * Q};
  LkLevel alt{lv + 5 * Q, lv + 6 * Q, lv + 7 * Q, lv + 8 * Q, lv + 9 * Q};
  const unsigned gq = grid_for(Q, 256), gm = grid_for(m, 256);
  // the lowest end of every point, in an array the first level resets later
  HDB_CALL(fill_i32(ctx, alt.rep_l, Q, kNoName));  // Q >= n for m = n - 1 >= 1
  hipLaunchKernelGGL(k_lk_first, dim3(gq), dim3(256), 0, ctx->stream, edges, m, n, alt.rep_l, bad);
  HDB_LAUNCHED();
  hipLaunchKernelGGL(k_lk_init, dim3(gq), dim3(256), 0, ctx->stream, edges, m, n, alt.rep_l, vid, top, sz, cur, par,
                     leaf_par);
  HDB_LAUNCHED();
  const int L = bits_for(m - 1);
  // edges per thread of k_lk_union and k_lk_merge: blocks of 4096 edges where they fill the
  // chip, fewer where that would leave it idle
  const int items = static_cast<int>(std::min<int64_t>(16, std::max<int64_t>(1, m / (256 * 1024))));
  for (int b = L - 1; b >= kLkBits; --b) {
    hipLaunchKernelGGL(k_lk_union, dim3(grid_for(m, 256 * items)), dim3(256), 0, ctx->stream, m, b, items, vid, cur);
    HDB_LAUNCHED();
    hipLaunchKernelGGL(k_lk_merge, dim3(grid_for(m, 256 * items)), dim3(256), 0, ctx->stream, m, b, items, vid, sz,
                       cur);
    HDB_LAUNCHED();
    hipLaunchKernelGGL(k_lk_rename, dim3(gq), dim3(256), 0, ctx->stream, m, b, n, vid, top, sz, top2, sz2, cur, alt);
    HDB_LAUNCHED();
    std::swap(cur, alt);
    std::swap(top, top2);
    std::swap(sz, sz2);
  }
  hipLaunchKernelGGL(k_lk_local, dim3(grid_for(m, kLkEdges)), dim3(kLkEdges), 0, ctx->stream, m, std::min(L, kLkBits),
                     n, vid, top, sz, top2, sz2);
  HDB_LAUNCHED();
  std::swap(top, top2);
  std::swap(sz, sz2);
  // ---- linkage tree, node classes, depth / preorder / cluster starts
  uint8_t* flags;
  TrRec *rec, *rec2;
  HDB_CALL(scratch_t(ctx, kSlotMstFlag, m, &flags));
  HDB_CALL(scratch_t(ctx, kSlotMstWl1, 2 * m, &rec));
  rec2 = rec + m;
  hipLaunchKernelGGL(k_tr_nodes, dim3(gm), dim3(256), 0, ctx->stream, edges, m, n, top, sz, left, right, nsize, par,
                     leaf_par, lam, bad);
  HDB_LAUNCHED();
  hipLaunchKernelGGL(k_tr_classify, dim3(grid_for(n, 256)), dim3(256), 0, ctx->stream, m, n, mpts, left, right, nsize,
                     par, leaf_par, flags, cnt, rec, splits, nsplit, bad);
  HDB_LAUNCHED();
  // the controls come back while the jumps run: a node is at most m - 1
  // deep, so bits_for(m - 1) rounds reach the root from everywhere
  static_assert(2 * sizeof(int32_t) == sizeof(int64_t), "both controls in one word");
  HDB_CALL(read_i64_async(ctx, reinterpret_cast<const int64_t*>(ctrl), 0));
  for (int round = 0; round < L; ++round) {
    hipLaunchKernelGGL(k_tr_jump, dim3(gm), dim3(256), 0, ctx->stream, m, rec, rec2);
    HDB_LAUNCHED();
    std::swap(rec, rec2);
  }
  int64_t both = 0;
  HDB_CALL(wait_i64(ctx, 0, &both));
  if (static_cast<int32_t>(both) != 0) return ctx->fail(HDB_EDEVICE, "inconsistent linkage tree");
  const int64_t S2 = both >> 32;
  // ---- splits in level order -> cluster ids
  if (S2 > kSplitSmall) {
    uint64_t* keys;
    uint32_t* vals;
    HDB_CALL(scratch_t(ctx, kSlotRowCursor, S2, &keys));
    HDB_CALL(scratch_t(ctx, kSlotMisc2, S2, &vals));
    const unsigned gs = grid_for(S2, 256);
    hipLaunchKernelGGL(k_tr_split_keys, dim3(gs), dim3(256), 0, ctx->stream, S2, splits, rec, keys, vals);
    HDB_LAUNCHED();
    HDB_CALL(radix_sort_u64_u32(ctx, keys, vals, S2, 0, bits_for(2 * n)));
    HDB_CALL(radix_sort_u64_u32(ctx, keys, vals, S2, 32, 32 + bits_for(m - 1)));
    hipLaunchKernelGGL(k_tr_split_rank, dim3(gs), dim3(256), 0, ctx->stream, S2, vals, srank);
    HDB_LAUNCHED();
  } else if (S2 > 0) {
    hipLaunchKernelGGL(k_tr_split_rank_small, dim3(1), dim3(1024), 0, ctx->stream, static_cast<int>(S2), splits, rec,
                       srank);
    HDB_LAUNCHED();
  }
  const int64_t S = 1 + 2 * S2;  // clusters
  float *birth, *stab, *cbirth;
  int32_t *cparent, *clab, *clen, *na;
  int64_t *cbeg, *aoff;
  float* add;
  HDB_CALL(scratch_t(ctx, kSlotMstCw, 6 * S, &birth));
  stab = birth + S;
  cparent = reinterpret_cast<int32_t*>(stab + S);
  clab = cparent + S;
  cbirth = reinterpret_cast<float*>(clab + S);
  clen = reinterpret_cast<int32_t*>(cbirth + S);
  HDB_CALL(scratch_t(ctx, kSlotMstCnt, S + 1, &cbeg));
  HDB_CALL(scratch_t(ctx, kSlotTreeAddCnt, m, &na));
  HDB_CALL(scratch_t(ctx, kSlotTreeAddOff, m + 1, &aoff));
  // a point leaves one cluster, and a split adds two terms
  HDB_CALL(scratch_t(ctx, kSlotTreeAdd, n + 2 * S2, &add));
  hipLaunchKernelGGL(k_tr_clusters, dim3(gm), dim3(256), 0, ctx->stream, m, n, mpts, flags, rec, par, left, right, nsize,
                     srank, lam, cid, pos, birth, cparent, clen, na);
  HDB_LAUNCHED();
  HDB_CALL(scan_i32_to_i64(ctx, clen, S, cbeg));
  // ---- stability: each cluster's nodes top-down
  hipLaunchKernelGGL(k_tr_addend_count, dim3(gm), dim3(256), 0, ctx->stream, m, flags, cid, pos, cbeg, cnt, na);
  HDB_LAUNCHED();
  HDB_CALL(scan_i32_to_i64(ctx, na, m, aoff));
  hipLaunchKernelGGL(k_tr_addends, dim3(gm), dim3(256), 0, ctx->stream, m, n, flags, cid, pos, cbeg, cnt, lam, left,
                     right, nsize, birth, aoff, add);
  HDB_LAUNCHED();
  hipLaunchKernelGGL(k_tr_stability, dim3(grid_for(S, 4)), dim3(256), 0, ctx->stream, S, cbeg, aoff, add, stab);
  HDB_LAUNCHED();
  if (n + 2 * S2 > kStabShort) {
    hipLaunchKernelGGL(k_tr_stability_long, dim3(static_cast<unsigned>(std::min<int64_t>(S, 512))),
                       dim3(kStabWaves * 64), 0, ctx->stream, S, cbeg, aoff, add, stab);
    HDB_LAUNCHED();
  }
  // ---- EOM selection over the cluster tree (host; one entry per cluster)
  std::vector<float> h_in(3 * S);  // birth, stability and parent, adjacent on the device
  HDB_HIP(hipMemcpyAsync(h_in.data(), birth, 3 * S * sizeof(float), hipMemcpyDeviceToHost, ctx->stream));
  HDB_HIP(hipStreamSynchronize(ctx->stream));
  const float* h_birth = h_in.data();
  float* h_stab = h_in.data() + S;
  std::vector<int32_t> h_par(S);
  std::memcpy(h_par.data(), h_in.data() + 2 * S, S * sizeof(int32_t));
  // cluster c's children are the two clusters its bottom split starts: for
  // c > 0 their ids are c's split rank's 1 + 2k, 2 + 2k; descending ids put
  // children before parents (a split starts clusters after its own)
  std::vector<int32_t> kid0(S, -1), kid1(S, -1);
  for (int64_t c = 1; c < S; ++c) {
    const int32_t p = h_par[c];
    if (p < 0 || p >= S) return ctx->fail(HDB_EDEVICE, "inconsistent cluster tree");
    if (c & 1) kid0[p] = static_cast<int32_t>(c);
    else kid1[p] = static_cast<int32_t>(c);
  }
  std::vector<uint8_t> kept(S, 0);
  for (int64_t c = S - 1; c >= 1; --c) {
    float sub = 0.0f;
    if (kid0[c] >= 0) sub += h_stab[kid0[c]];
    if (kid1[c] >= 0) sub += h_stab[kid1[c]];
    if (sub > h_stab[c]) h_stab[c] = sub;
    else kept[c] = 1;
  }
  // selected: kept with no kept ancestor (the root cluster never counts);
  // parents precede children in ascending ids
  std::vector<uint8_t> blocked(S, 0), sel(S, 0);
  std::vector<int32_t> sel_anc(S, -1);
  for (int64_t c = 1; c < S; ++c) {
    const int32_t p = h_par[c];
    blocked[c] = p > 0 && (blocked[p] || kept[p]);
    sel[c] = kept[c] && !blocked[c];
    sel_anc[c] = sel[c] ? static_cast<int32_t>(c) : (p > 0 ? sel_anc[p] : -1);
  }
  std::vector<int32_t> cmap(S, -1);
  int32_t nsel = 0;
  for (int64_t c = 1; c < S; ++c)
    if (sel[c]) cmap[c] = nsel++;
  std::vector<int32_t> h_out(2 * S);  // label and birth of the selected ancestor
  for (int64_t c = 0; c < S; ++c) {
    const int32_t a = sel_anc[c];
    const float bl = a >= 0 ? h_birth[a] : 0.0f;
    h_out[c] = a >= 0 ? cmap[a] : -1;
    std::memcpy(&h_out[S + c], &bl, sizeof(bl));
  }
  HDB_HIP(hipMemcpyAsync(clab, h_out.data(), 2 * S * sizeof(int32_t), hipMemcpyHostToDevice, ctx->stream));
  hipLaunchKernelGGL(k_tr_label, dim3(grid_for(n, 256)), dim3(256), 0, ctx->stream, n, leaf_par, flags, rec, par, cid,
                     lam, clab, cbirth, labels);
  HDB_LAUNCHED();
  HDB_HIP(hipStreamSynchronize(ctx->stream));  // the host vectors above are sources of the copies
  if (clusters_out) *clusters_out = nsel;
  return HDB_OK;
}

}  // namespace hdb
