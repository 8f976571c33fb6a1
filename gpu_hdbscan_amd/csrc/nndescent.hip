// NN-Descent kNN-graph construction for gfx950.
//
// Layout in HBM (n points, K = 32):
//   lists     n x 32 hdb_nnd_element {float d2, int label}, each list sorted
//             by the key (d2 bits, id, old-before-new); label < 0 marks "old"
//             (tools/nndescent_element.cuh:13-18).
//   fwd_*     n x 16 int32 forward samples (+ counts n).
//   rev pairs n x 32 (key = 2q + old, value = p) for every forward sample
//             q of p, new pairs before old ones, radix-sorted by key >> 1;
//             rev_se = [start, end) per key.
//   proposals (target u32, key u64) appended per workgroup into 64 segments,
//             radix-sorted by target >> 4; prop_se = [start, end) per group
//             of 16 lists.
//   worst     n f32: d2 of entry 31 of each list (proposal prefilter); for
//             the FP32 join with d <= 31 the last column of a padded copy
//             of the points (rows of 16 or 32 floats), so that the join
//             reads a candidate's coordinates and bound in one aligned row.
//
// One iteration (gpuknn/nndescent.cu:2133-2166):
//   k_nnd_sample   PrepareGraph (:44-98): forward samples, reverse pairs
//   radix sort     PrepareReverseGraph (:293-346) without global atomics;
//                  each reverse list keeps S of its pairs, evenly spaced
//                  in source order (the reference keeps the first S arrivals)
//   k_nnd_join*    ShrinkGraph + NewNeighborsCompareKernel +
//                  TiledNewOldNeighborsCompareKernel (:405-510, :1030-1326):
//                  one wave64 per point; candidates propose their nearest
//                  partners to their own lists
//   radix sort     proposals grouped by list group (target >> 4)
//   k_nnd_update   MarkAllToOld + InsertToGlobalGraph (:1398-1403, :969-1028):
//                  one 4-wave block per group of 16 lists buckets the group's
//                  proposals by list in LDS; a wave merges each of its four
//                  buckets into its list 64 proposals at a time (sort,
//                  unique, bitonic merge); no locks, and the result is the
//                  first 32 distinct keys of the union whatever the proposal
//                  order.
#include <algorithm>
#include <type_traits>

#include "hdb_internal.hpp"

namespace hdb {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kSMax = 16;  // sample list stride (SAMPLE_NUM <= 16)
// Largest point count: the n x 32 reverse pairs and list entries are
// addressed with int32 positions.
constexpr int64_t kMaxPoints = static_cast<int64_t>(1) << 26;
constexpr int kJoinWaves = 4;
// Join blocks append proposals to one of kPropSegs segments (block % kPropSegs),
// each with its own counter kCtrStride words apart: atomics on one address
// serialise, so one counter for every block would limit the join.
constexpr int kPropSegs = 64;
constexpr int kCtrStride = 32;

struct NndBufs {
  int32_t* fwd_new;
  int32_t* fwd_old;
  int32_t* fwd_new_n;
  int32_t* fwd_old_n;
  uint32_t* rev_key;
  uint32_t* rev_val;
  int32_t* rev_s;  // 2n
  int32_t* rev_e;  // 2n
  uint32_t* prop_tgt;
  uint64_t* prop_key;
  int64_t* prop_s;  // per list group (16 lists); the proposal stream can pass 2^31
  int64_t* prop_e;
  unsigned long long* prop_cnt;  // kPropSegs counters, kCtrStride apart
  int64_t prop_cap;
  int64_t seg_cap;  // proposals per segment: prop_cap / kPropSegs
  // List bound of point t at worst[t * wstride].  FP32 joins with d <= 31
  // read their candidates from a padded copy of the points (rows of rstride
  // = 16 or 32 floats, zeros past d) whose last column holds that bound, so
  // one aligned 64- or 128-byte row brings both; otherwise rows = X
  // (rstride = d) and the bounds are an array of their own (wstride = 1).
  float* worst;
  const float* norms;  // BF16 join: |x|^2 of every point
  const float* rows;
  int rstride;
  int wstride;
  unsigned long long* part;  // per join wave (point): [0] proposals, [1] capacity drops, [2] reverse drops, [3] candidates
  int join_keep;
  int distance_mode;  // 0: FP32 join, 1: BF16 MFMA shortlist + exact FP32 re-rank
  int iter;           // iteration index: seeds the rotation of the sample choice
  uint32_t s_recip;   // floor(2^32 / S) + 1 (S >= 2) and ceil(65536 / S): divisions by the sample count
  uint32_t s_recip16;
  int rerank_deep;    // BF16 join: re-rank the 16 nearest BF16 partners (else join_keep + 2)
};

// Rotation of the sample choice of list (or reverse segment) `key` in
// iteration `it`: when more than S entries of a kind are present, the S
// taken start at a rank drawn from this hash, so that over the iterations
// every entry is sampled (the reference keeps the first S to win an LDS
// atomic, an effectively random choice); the choice stays deterministic.
__device__ __forceinline__ uint64_t sample_rotation(uint64_t key, int it) {
  return xorshift64star((key << 6) ^ (static_cast<uint64_t>(it + 1) * 0x9E3779B97F4A7C15ull));
}

__device__ __forceinline__ hdb_nnd_element key_to_elem(uint64_t key) {
  hdb_nnd_element e;
  if (key == kKeyMax) {
    e.distance = __uint_as_float(0x7F800000u);
    e.label = static_cast<int32_t>(kInvalidId);
  } else {
    const uint32_t id = key_id(key);
    e.distance = key_d2(key);
    e.label = key_new(key) ? static_cast<int32_t>(id) : -static_cast<int32_t>(id) - 1;
  }
  return e;
}

// Rows read as float4 when every row is 16-byte aligned (same summation
// order either way, so the same bits).
__device__ __forceinline__ float point_d2(const float* __restrict__ X, int d, uint32_t a, uint32_t b) {
  const float* ra = X + static_cast<int64_t>(a) * d;
  const float* rb = X + static_cast<int64_t>(b) * d;
  if ((d & 3) == 0 && (reinterpret_cast<uintptr_t>(X) & 15) == 0) return d2_vec4(ra, rb, d);
  return d2_any(ra, rb, d);
}
// The same distance from rows rs floats apart (the padded copy: zeros past
// d, read over the first d only, so the same bits).
__device__ __forceinline__ float row_d2(const float* __restrict__ R, int rs, int d, uint32_t a, uint32_t b) {
  const float* ra = R + static_cast<int64_t>(a) * rs;
  const float* rb = R + static_cast<int64_t>(b) * rs;
  if ((d & 3) == 0 && (rs & 3) == 0 && (reinterpret_cast<uintptr_t>(R) & 15) == 0) return d2_vec4(ra, rb, d);
  return d2_any(ra, rb, d);
}
// ------------------------------------------------------------------ init --
// InitKNNGraphIndexKernel (nndescent.cu:1673-1692) with the xorshift64* index
// path selected at :2118, then InitKNNGraphDistanceKernel (:1694-1726) and a
// sort of each list (SortEachBlockKernel :1728-1750).  Lane j of list p
// draws label = xorshift64star(p*K + j) mod n and steps +1 past p.  X holds
// rows rs floats apart: the points, or their padded copy when the join
// reads that (the same distances either way).
__global__ __launch_bounds__(256) void k_nnd_init_random(const float* __restrict__ X, int rs, int64_t n, int d,
                                                         hdb_nnd_element* __restrict__ lists,
                                                         float* __restrict__ worst, int ws) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t p = t >> 5;
  const int j = static_cast<int>(t & 31);
  uint64_t key = kKeyMax;
  if (p < n) {
    uint64_t lab = xorshift64star(static_cast<uint64_t>(p * kK + j)) % static_cast<uint64_t>(n);
    if (static_cast<int64_t>(lab) == p) lab = (lab + 1) % static_cast<uint64_t>(n);
    const float d2 = row_d2(X, rs, d, static_cast<uint32_t>(p), static_cast<uint32_t>(lab));
    key = make_key(d2, static_cast<uint32_t>(lab), 1u);
  }
  key = bitonic_group<32>(key);
  if (p < n) {
    lists[p * kK + j] = key_to_elem(key);
    if (j == kK - 1) worst[p * ws] = key_d2(key);
  }
}

// n <= K + 1: list p holds every other point (lane j takes j, or j + 1 past
// p), sorted; the remaining slots are empty.
__global__ __launch_bounds__(256) void k_nnd_exact_small(const float* __restrict__ X, int64_t n, int d,
                                                         hdb_nnd_element* __restrict__ lists) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t p = t >> 5;
  const int j = static_cast<int>(t & 31);
  uint64_t key = kKeyMax;
  const int64_t q = j < p ? j : j + 1;
  if (p < n && q < n) key = make_key(point_d2(X, d, static_cast<uint32_t>(p), static_cast<uint32_t>(q)),
                                     static_cast<uint32_t>(q), 1u);
  key = bitonic_group<32>(key);
  if (p < n) lists[p * kK + j] = key_to_elem(key);
}

// Recompute the distances of caller-supplied lists, sort them and mark
// every entry new (start of gpuknn::NNDescent from given lists).
__global__ __launch_bounds__(256) void k_nnd_init_given(const float* __restrict__ X, int64_t n, int d,
                                                        hdb_nnd_element* __restrict__ lists,
                                                        float* __restrict__ worst, int ws) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t p = t >> 5;
  const int j = static_cast<int>(t & 31);
  uint64_t key = kKeyMax;
  if (p < n) {
    const uint32_t id = label_id(lists[p * kK + j].label);
    if (id != kInvalidId && static_cast<int64_t>(id) < n && static_cast<int64_t>(id) != p) {
      key = make_key(point_d2(X, d, static_cast<uint32_t>(p), id), id, 1u);
    }
  }
  key = bitonic_group<32>(key);
  // duplicates: keep the first of equal keys
  uint32_t lo = static_cast<uint32_t>(key), hi = static_cast<uint32_t>(key >> 32);
  uint32_t plo = __shfl_up(lo, 1), phi = __shfl_up(hi, 1);
  const uint64_t prev = (static_cast<uint64_t>(phi) << 32) | plo;
  const bool keep = key != kKeyMax && (j == 0 || (prev >> 1) != (key >> 1));
  const uint64_t bal = __ballot(keep);
  const uint32_t half = static_cast<uint32_t>(bal >> (threadIdx.x & 32));
  const int pos = __popc(half & ((1u << j) - 1u));
  const int total = __popc(half);
  if (p < n) {
    if (keep) lists[p * kK + pos] = key_to_elem(key);
    if (j >= total) lists[p * kK + j] = key_to_elem(kKeyMax);
    if (keep && pos == kK - 1) worst[p * ws] = key_d2(key);
    if (j == 0 && total < kK) worst[p * ws] = __uint_as_float(0x7F800000u);
  }
}

// Lists already sorted, distinct and exact (as hdb_learned_init writes
// them): every entry is marked new and the list bound read off.
__global__ __launch_bounds__(256) void k_nnd_init_exact(hdb_nnd_element* __restrict__ lists, int64_t n,
                                                        float* __restrict__ worst, int ws) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= n * kK) return;
  hdb_nnd_element e = lists[t];
  if (e.label < 0) {
    e.label = -e.label - 1;
    lists[t] = e;
  }
  if ((t & (kK - 1)) == kK - 1) worst[(t / kK) * ws] = e.distance;
}

// knnmerge init: InitRandomBlockedKNNGraph (gpuknn/knnmerge.cu:80-185) after
// MarkAllToOld of both inputs (:487-503).  List p keeps the first 16 entries
// of its own graph (old; ids of graph 2 shifted by n1) and draws 16 new
// cross-half ids xorshift64star(local*16 + t) mod n_other (+ n1 for lists of
// graph 1), t = 0..15; distances are then recomputed and the list sorted
// (InitRandomKNNGraph with start_from_random_index = false, :2015).
__global__ __launch_bounds__(256) void k_nnd_init_merge(const float* __restrict__ X, int64_t n1, int64_t n2, int d,
                                                        const hdb_nnd_element* __restrict__ g1,
                                                        const hdb_nnd_element* __restrict__ g2,
                                                        hdb_nnd_element* __restrict__ lists,
                                                        float* __restrict__ worst, int ws) {
  const int64_t n = n1 + n2;
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t p = t >> 5;
  const int j = static_cast<int>(t & 31);
  uint64_t key = kKeyMax;
  if (p < n) {
    const bool first = p < n1;
    const int64_t local = first ? p : p - n1;
    uint32_t id;
    uint32_t is_new;
    if (j < kK / 2) {
      const hdb_nnd_element e = first ? g1[local * kK + j] : g2[local * kK + j];
      id = label_id(e.label);
      if (id != kInvalidId && static_cast<int64_t>(id) >= (first ? n1 : n2)) id = kInvalidId;
      if (id != kInvalidId && !first) id += static_cast<uint32_t>(n1);
      is_new = 0u;
    } else {
      const uint64_t r = xorshift64star(static_cast<uint64_t>(local * (kK / 2) + (j - kK / 2)));
      id = first ? static_cast<uint32_t>(r % static_cast<uint64_t>(n2) + static_cast<uint64_t>(n1))
                 : static_cast<uint32_t>(r % static_cast<uint64_t>(n1));
      is_new = 1u;
    }
    if (id != kInvalidId) key = make_key(point_d2(X, d, static_cast<uint32_t>(p), id), id, is_new);
  }
  key = bitonic_group<32>(key);
  if (p < n) {
    lists[p * kK + j] = key_to_elem(key);
    if (j == kK - 1) worst[p * ws] = (key == kKeyMax) ? __uint_as_float(0x7F800000u) : key_d2(key);
  }
}

// -------------------------------------------------------------- sampling --
// Forward samples: S new and S old entries of the list -- all of a kind
// when it has at most S, else S consecutive in list order (cyclically) from
// a rank rotated per point and iteration (the reference keeps the first S
// that win an LDS atomic); in merge mode old entries are kept only from the
// list's own half (PrepareGraphForMerge :100-166).  Every forward sample q of p becomes the
// reverse pair (2q + old, p) at slot 16n*old + 16p + rank; unused slots get
// the key 2n, past every real key, which the sort leaves out (half the slots
// of the first iteration, a quarter of the later ones).  New pairs all precede old
// ones, so a stable sort on the key without its low bit orders the pairs by
// the whole key (q, then new before old, then p).
template <bool MERGE>
__global__ __launch_bounds__(256) void k_nnd_sample(const hdb_nnd_element* __restrict__ lists, int64_t n, int S,
                                                    int64_t split, NndBufs b) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t p = t >> 5;
  const unsigned j = threadIdx.x & 31u;
  bool take_new = false, take_old = false;
  uint32_t id = kInvalidId;
  if (p < n) {
    const int32_t lab = lists[p * kK + j].label;
    id = label_id(lab);
    if (id != kInvalidId && static_cast<int64_t>(id) < n) {
      if (lab >= 0) take_new = true;
      else take_old = !MERGE || ((static_cast<int64_t>(id) < split) == (p < split));
    }
  }
  const unsigned sh = threadIdx.x & 32u;
  const uint32_t mnew = static_cast<uint32_t>(__ballot(take_new) >> sh);
  const uint32_t mold = static_cast<uint32_t>(__ballot(take_old) >> sh);
  if (p >= n) return;  // 32-lane halves are uniform in p
  const uint32_t lt = (1u << j) - 1u;
  const int cn = __popc(mnew), co = __popc(mold);
  const int nn = min(cn, S), no = min(co, S);
  int rot_n = 0, rot_o = 0;
  if (cn > S || co > S) {
    const uint64_t h = sample_rotation(static_cast<uint64_t>(p), b.iter);
    rot_n = cn > S ? static_cast<int>(static_cast<uint32_t>(h) % static_cast<uint32_t>(cn)) : 0;
    rot_o = co > S ? static_cast<int>(static_cast<uint32_t>(h >> 32) % static_cast<uint32_t>(co)) : 0;
  }
  const int64_t half = (j < 16 ? 0 : 16 * n) + p * 16;  // this lane's kind: new (j < 16) or old
  uint32_t* rk_new = b.rev_key + p * 16;
  uint32_t* rv_new = b.rev_val + p * 16;
  uint32_t* rk_old = b.rev_key + 16 * n + p * 16;
  uint32_t* rv_old = b.rev_val + 16 * n + p * 16;
  const uint32_t sentinel = static_cast<uint32_t>(2 * n);
  if (take_new) {
    int r = __popc(mnew & lt) - rot_n;  // rank in the rotated order
    if (r < 0) r += cn;
    if (r < S) {
      b.fwd_new[p * kSMax + r] = static_cast<int32_t>(id);
      rk_new[r] = 2u * id;
      rv_new[r] = static_cast<uint32_t>(p);
    }
  }
  if (take_old) {
    int r = __popc(mold & lt) - rot_o;
    if (r < 0) r += co;
    if (r < S) {
      b.fwd_old[p * kSMax + r] = static_cast<int32_t>(id);
      rk_old[r] = 2u * id + 1u;
      rv_old[r] = static_cast<uint32_t>(p);
    }
  }
  if ((j < 16 && static_cast<int>(j) >= nn) || (j >= 16 && static_cast<int>(j) - 16 >= no))
    b.rev_key[half + (j & 15u)] = sentinel;
  if (j == 0) {
    b.fwd_new_n[p] = nn;
    b.fwd_old_n[p] = no;
  }
}

// ------------------------------------------------------------ local join --
// Lanes below this one in the mask m.
__device__ __forceinline__ int lanes_below(uint64_t m) {
  return static_cast<int>(__builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(m >> 32),
                                                    __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(m), 0u)));
}

// Orders a wave's LDS writes before its later LDS reads by other lanes of
// the same wave: LDS instructions of a wave execute in order, so a compiler
// fence and scheduling barrier at wavefront scope are enough (the waves of a
// join block share no LDS data).
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Per point p (one wave): new = sort/dedup(fwd_new + rev_new), old =
// sort/dedup(fwd_old + rev_old), new -= old (ShrinkGraph :405-510).  The
// candidate ids land in s_cand (new first, each kind ascending), the wave's
// own 64-entry LDS row: waves run it independently.  All 64 slots go through
// one sort by (id, old before new), where an id's first slot is the one to
// keep: two sorts of 32, a search of every new id among the old ones and
// five-instruction sort steps took a third of the join's instructions.
__device__ __forceinline__ void join_candidates(const NndBufs& b, int64_t p, bool live, int S, uint32_t* s_cand,
                                                int* nn_out, int* nc_out, int* rev_drop_out) {
  const unsigned lane = __lane_id();
  uint32_t v = 0xFFFFFFFFu;
  int rev_drop = 0;
  if (live) {  // uniform: p is the wave's point
    // lanes 0-15 forward new, 16-31 reverse new, 32-47 forward old, 48-63
    // reverse old; the counts and the reverse segments' bounds are
    // wave-uniform (scalar loads)
    const int pu = __builtin_amdgcn_readfirstlane(static_cast<int>(p));
    const int part = lane >> 4, r = lane & 15;
    const bool rev = (part & 1) != 0, oldk = part >= 2;
    const int cn = b.fwd_new_n[pu], co = b.fwd_old_n[pu];
    const int s0n = b.rev_s[2 * pu], s0o = b.rev_s[2 * pu + 1];
    const int ln = b.rev_e[2 * pu] - s0n, lo = b.rev_e[2 * pu + 1] - s0o;
    // S evenly spaced entries of a longer reverse segment, rotated per
    // iteration so that every entry is sampled over the iterations:
    // entry (floor(r len / S) + rot) mod len, with floor(r len / S) =
    // r (len / S) + floor(r (len mod S) / S); the last term has r (len mod S)
    // < 256, where multiplying by ceil(65536 / S) and shifting is exact.
    const int len = oldk ? lo : ln;
    int off = r;
    if (ln > S || lo > S) {
      int rn = 0, ro = 0;
      if (ln > S)
        rn = static_cast<int>(static_cast<uint32_t>(sample_rotation(static_cast<uint64_t>(2 * pu), b.iter)) %
                              static_cast<uint32_t>(ln));
      if (lo > S)
        ro = static_cast<int>(static_cast<uint32_t>(sample_rotation(static_cast<uint64_t>(2 * pu + 1), b.iter)) %
                              static_cast<uint32_t>(lo));
      // both quotients on the scalar unit: x / S = x m >> 32 with m =
      // floor(2^32 / S) + 1, exact for x < 2^28 and 2 <= S <= 16
      const int qn = S == 1 ? ln : static_cast<int>(__umulhi(static_cast<uint32_t>(ln), b.s_recip));
      const int qo = S == 1 ? lo : static_cast<int>(__umulhi(static_cast<uint32_t>(lo), b.s_recip));
      const int q = oldk ? qo : qn, rem = oldk ? lo - qo * S : ln - qn * S, rot = oldk ? ro : rn;
      if (len > S) {
        off = r * q + static_cast<int>((static_cast<uint32_t>(r * rem) * b.s_recip16) >> 16) + rot;
        off = off >= len ? off - len : off;
      }
    }
    const int cnt = rev ? min(len, S) : (oldk ? co : cn);
    const uint32_t* src = rev ? b.rev_val + (oldk ? s0o : s0n)
                              : reinterpret_cast<const uint32_t*>(oldk ? b.fwd_old : b.fwd_new) + pu * kSMax;
    if (r < cnt) v = (src[rev ? off : r] << 1) | (oldk ? 0u : 1u);  // ids are below 2^26
    if (rev && r == 0 && len > S) rev_drop = len - S;
  }
  v = bitonic_group_u32<64>(v);
  const uint32_t prev = lane_below(v);
  const bool keep = v != 0xFFFFFFFFu && (lane == 0 || (v >> 1) != (prev >> 1));
  const uint64_t all = __ballot(keep), fresh = __ballot(keep && (v & 1u));
  const uint64_t old = all ^ fresh;
  const int nn = __popcll(fresh);
  if (keep) s_cand[(v & 1u) ? lanes_below(fresh) : nn + lanes_below(old)] = v >> 1;
  wave_sync();
  *nn_out = nn;
  *nc_out = nn + __popcll(old);
  *rev_drop_out = rev_drop;
}

// Filters each lane's proposals against its list bound lim, compacts the
// wave's proposals with one atomic and appends them; accumulates the wave's
// counters.  Waves run it independently: wave wid (the block's WPB waves
// numbered from blockIdx.x * WPB) appends to segment wid % kPropSegs and
// counts into part[4 wid ..]; a lane's offset among the wave's proposals is
// the number of valid slots in the lanes below it (ballot and mbcnt).
template <int WPB, int SLOTS>
__device__ __forceinline__ void join_emit(const NndBufs& b, uint64_t (&top)[SLOTS], bool active, uint32_t my_id,
                                          float lim, int nc, int rev_drop) {
  const unsigned lane = __lane_id();
  const int64_t wid = static_cast<int64_t>(blockIdx.x) * WPB + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int excl = 0, wcnt = 0;
#pragma unroll
  for (int s = 0; s < SLOTS; ++s) {
    const bool ok = active && top[s] != kKeyMax && key_d2(top[s]) < lim;
    if (!ok) top[s] = kKeyMax;
    const uint64_t m = __ballot(ok);
    excl += lanes_below(m);
    wcnt += __popcll(m);
  }
  // reverse-sample drops: lanes 16 and 48 hold them
  const int rd = __builtin_amdgcn_readlane(rev_drop, 16) + __builtin_amdgcn_readlane(rev_drop, 48);
  if (wcnt == 0 && rd == 0 && nc == 0) return;  // uniform: a wave past n, or a point without candidates
  const int seg = static_cast<int>(wid % kPropSegs);
  unsigned long long bs = 0;
  if (lane == 0) {
    bs = wcnt ? atomicAdd(b.prop_cnt + seg * kCtrStride, static_cast<unsigned long long>(wcnt)) : 0ull;
    unsigned long long* pp = b.part + 4 * wid;
    pp[0] += static_cast<unsigned long long>(wcnt);
    const int64_t over = static_cast<int64_t>(bs) + wcnt - b.seg_cap;
    if (over > 0) pp[1] += static_cast<unsigned long long>(over < wcnt ? over : wcnt);
    pp[2] += static_cast<unsigned long long>(rd);
    pp[3] += static_cast<unsigned long long>(nc);
  }
  const int64_t base = static_cast<int64_t>(__builtin_amdgcn_readfirstlane(static_cast<uint32_t>(bs))) |
                       (static_cast<int64_t>(__builtin_amdgcn_readfirstlane(static_cast<uint32_t>(bs >> 32))) << 32);
  // entries past the segment's capacity are dropped one by one, so each
  // segment holds exactly its first min(count, seg_cap) entries
  int64_t o = base + excl;
  const int64_t seg0 = static_cast<int64_t>(seg) * b.seg_cap;
#pragma unroll
  for (int s = 0; s < SLOTS; ++s) {
    if (top[s] != kKeyMax) {
      if (o < b.seg_cap) {
        b.prop_tgt[seg0 + o] = my_id;
        b.prop_key[seg0 + o] = top[s];
      }
      ++o;
    }
  }
}

// Keeps the SLOTS smallest keys (ascending) of a stream.
template <int SLOTS>
__device__ __forceinline__ void top_insert(uint64_t (&top)[SLOTS], uint64_t key) {
#pragma unroll
  for (int s = 0; s < SLOTS; ++s) {
    const uint64_t a = top[s];
    const bool sw = key < a;
    top[s] = sw ? key : a;
    key = sw ? a : key;
  }
}

// FP32 joins.  Candidate c (lane c) takes the squared distance to each
// partner -- the other new candidates and the old ones if c is new (NEWNEW),
// only the old ones if c is new in merge mode, the new ones if c is old --
// and proposes its nearest partners (GetMinElement/2/3 :852-961) to its own
// list unless they cannot beat the list's current 32nd entry.  KEEP == 0: the
// reference's two kernels -- a new candidate takes its nearest new partner
// (NewNeighborsCompareKernel) and its nearest old partner
// (TiledNewOldNeighborsCompareKernel), an old one its nearest new partner.
// KEEP > 0: every candidate proposes its nearest partners.  k_nnd_join2
// serves d = 12 and 32, k_nnd_join_rows the other d <= 31, k_nnd_join_wide
// d > 32.

// Order-preserving u32 image of a float of any sign (NaN excluded).
__device__ __forceinline__ uint32_t order_bits(float x) {
  const uint32_t b = __float_as_uint(x);
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}

template <int SLOTS>
__device__ __forceinline__ void top_insert32(uint32_t (&top)[SLOTS], uint32_t key) {
  top_insert_med3<SLOTS>(top, key);
}

// Ranking values of candidate `lane` against candidates 4 Q .. 4 Q + 3:
// |b|^2 + sum_k (-2 a_k) b_k + |a|^2, the additions in that order with one
// rounding each (the norms come in as products with 1).  The 4 x 4 x 1 matrix product works on 16 blocks of
// 4 x 4; with the A operand's block Q broadcast to all of them its rows are
// the four partners and its column is the lane's own candidate, so both
// operands are the lanes' own registers and the four results are the lane's.
template <int D, int Q, int DS>
__device__ __forceinline__ f32x4 join_quad(const float (&own)[DS], const float (&own2)[D], float own_norm) {
  const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
  f32x4 acc = __builtin_amdgcn_mfma_f32_4x4x1f32(own_norm, 1.0f, zero, 4, Q, 0);
#pragma unroll
  for (int k = 0; k < D; ++k) acc = __builtin_amdgcn_mfma_f32_4x4x1f32(own[k], own2[k], acc, 4, Q, 0);
  return __builtin_amdgcn_mfma_f32_4x4x1f32(1.0f, own_norm, acc, 4, Q, 0);
}

// f(integral_constant Q) for Q = Q0 .. Q1 - 1: the block selector of a matrix
// product is an immediate.
template <int Q0, int Q1, typename F>
__device__ __forceinline__ void join_quads(F f) {
  if constexpr (Q0 < Q1) {
    f(std::integral_constant<int, Q0>{});
    join_quads<Q0 + 1, Q1>(f);
  }
}

// Partner-split FP32 join for D <= 32.  Phase 1: every candidate ranks each
// new candidate by |a|^2 + |b|^2 - 2 a.b (so each old-new pair is evaluated
// once) and old candidates store that value in an LDS block; phase 2: new
// candidates read their old partners from that block.  Ranking uses 32-bit
// keys -- the bits of that value without the sign, with the low 6 bits
// replaced by the partner's index -- and the KEEP winners' exact squared
// distances are then recomputed from the same rows in the same operation
// order as the other joins, so proposals carry exactly its distances.  A
// ranking value carries the roundings of the norms and of D products, about
// 2^-22 (|a|^2 + |b|^2) and at most (D + 2) 2^-24 of it, and the key a relative
// 2^-17: partners whose distances differ by less may be chosen in either
// order.  Data far from the origin for its neighbour distances leaves nothing
// but that error (unit clusters 3000 off it: recall 0.33 at 300k x 12), so a
// wave whose last winners show it (below) ranks every partner by its
// distance.  The ranking values come from the matrix cores, four partners of
// all 64 candidates in D + 2 products (join_quad), where the vector unit took
// D multiply-adds per partner and each wave read the partners' rows from LDS
// again.  At D = 32 the kernel is bound by instruction issue: at 500k points
// and KEEP = 3 a launch takes 1.17 ms instead of 1.63 (the block and the rows
// in one buffer: five blocks on a CU, not four).  At D = 12 it is bound by the
// gathers of the candidates' rows, 42M L2 misses a launch of 1M points: with 744
// vector instructions per wave instead of 1034 a launch takes 1.44 ms at 1M (1.37
// before) and 13.5 at 10M (13.9).
template <int D, bool NEWNEW, int KEEP>
__global__ __launch_bounds__(kJoinWaves * 64, D <= 16 ? 8 : 5) void k_nnd_join2(const float* __restrict__ X, int64_t n, int d, int S,
                                                               NndBufs b) {
  static_assert(D > 0 && D <= 32, "register-resident rows only");
  constexpr int WPB = kJoinWaves;
  constexpr int kStride = (D + 3) & ~3;
  constexpr int kSlots = KEEP == 0 ? 2 : KEEP;
  // Old x new block, rows of kBst values (odd, so the old lanes' stores and
  // the new lanes' column reads spread over the banks); it holds every old-new
  // pair.  Its values add the old candidate's norm last; where no * (nn + 1)
  // passes kBlock, phase 2 forms them again with the new candidate's norm last.
  // kBlock is no capacity: it decides the order of additions, and with it the
  // choice between partners that the ranking cannot tell apart.  Taking every
  // value from the block changes 73 of 1M lists (d = 12, join_keep 3, six
  // iterations; the joins 8.54 -> 8.10 ms), so the limit stays.
  constexpr int kBlock = 384;
  constexpr int kBst = 33;
  // The block's space takes the candidates' rows afterwards, kCols columns
  // at a time (D = 32: two chunks, which lets five blocks share a CU).
  constexpr int kCols = D <= 16 ? kStride : 16;
  constexpr int kRow = kCols == 16 ? 20 : kCols;
  constexpr int kBuf = 64 * kRow > 32 * kBst ? 64 * kRow : 32 * kBst;
  constexpr uint32_t kNone = 0xFFFFFFFFu;
  __shared__ __attribute__((aligned(16))) float s_buf[WPB][kBuf];
  __shared__ uint32_t s_cand[WPB][64];
  (void)d;
  const unsigned lane = __lane_id();
  const unsigned w = threadIdx.x >> 6;
  const int64_t p = static_cast<int64_t>(blockIdx.x) * WPB + w;

  int nn, nc, rev_drop;
  join_candidates(b, p, p < n, S, s_cand[w], &nn, &nc, &rev_drop);
  const int no = nc - nn;
  const bool active = lane < static_cast<unsigned>(nc);
  const bool is_new = lane < static_cast<unsigned>(nn);
  const uint32_t my_id = active ? s_cand[w][lane] : 0u;
  // D <= 15: the candidate's padded row of 16 floats (one aligned 64-byte
  // read) holds its list bound in the last column
  constexpr bool kPadded = D <= 15;
  float own[kStride];
  float lim = 0.0f;
  if (active) {
    if (kPadded) {
      const float4* src = reinterpret_cast<const float4*>(b.rows + static_cast<int64_t>(my_id) * 16);
      float r[16];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float4 v = src[q];
        r[4 * q] = v.x;
        r[4 * q + 1] = v.y;
        r[4 * q + 2] = v.z;
        r[4 * q + 3] = v.w;
      }
#pragma unroll
      for (int k = 0; k < D; ++k) own[k] = r[k];
      lim = r[15];
    } else {
      const float* src = X + static_cast<int64_t>(my_id) * D;
#pragma unroll
      for (int k = 0; k < D; ++k) own[k] = src[k];
      lim = b.worst[static_cast<int64_t>(my_id) * b.wstride];
    }
  } else {
#pragma unroll
    for (int k = 0; k < D; ++k) own[k] = 0.0f;
  }
#pragma unroll
  for (int k = D; k < kStride; ++k) own[k] = 0.0f;
  float own_norm = 0.0f;
#pragma unroll
  for (int k = 0; k < D; ++k) own_norm = __builtin_fmaf(own[k], own[k], own_norm);

  // Ranking value |b|^2 + sum_k (-2 a_k) b_k + |a|^2 (-2 a_k is exact).
  // Cancellation can leave it slightly below 0; the key's mask drops the
  // sign, so such a value ranks as its magnitude, still next to 0.
  float own2[D];
#pragma unroll
  for (int k = 0; k < D; ++k) own2[k] = -2.0f * own[k];
  // Phase 1 ranks the lane's own row too (a new lane meets itself among the
  // new partners): one slot more is kept and the lane itself dropped at the
  // end, which leaves the KEEP nearest of the others.  KEEP == 0: slots 0-1
  // take the new partners (the lane itself included), slot 2 the old ones.
  constexpr int kRank = kSlots + 1;
  uint32_t top[kRank];
#pragma unroll
  for (int s = 0; s < kRank; ++s) top[s] = kNone;
  const bool blocked = no * (nn + 1) <= kBlock;  // uniform
  const bool store_old = active && !is_new && blocked;
  // row o: old candidate nn + o's values against the new candidates
  float* blk_row = s_buf[w] + (store_old ? (static_cast<int>(lane) - nn) * kBst : 0);  // + j
  // (bits & 0x7FFFFFC0) | j
  auto rank_key = [&](float acc, int j) { return (__float_as_uint(acc) & 0x7FFFFFC0u) | static_cast<uint32_t>(j); };
  auto rank_new = [&](int j, float acc) {
    const uint32_t key = rank_key(acc, j);
    if (KEEP == 0) {
      uint32_t t2[2] = {top[0], top[1]};
      top_insert32<2>(t2, key);
      top[0] = t2[0];
      top[1] = t2[1];
    } else {
      top_insert32<kRank>(top, key);
    }
  };
  // phase 1: partners among the new candidates (at most 32), four per step
  join_quads<0, 8>([&](auto quad) {
    constexpr int Q = decltype(quad)::value, j = 4 * Q;
    if (j >= nn) return;  // uniform, as are the conditions below
    const f32x4 v = join_quad<D, Q>(own, own2, own_norm);
    if (j + 4 <= nn) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float a = v[r];
        if (store_old) blk_row[j + r] = a;
        rank_new(j + r, a);
      }
    } else {
#pragma unroll
      for (int r = 0; r < 3; ++r) {
        if (j + r < nn) {
          const float a = v[r];
          if (store_old) blk_row[j + r] = a;
          rank_new(j + r, a);
        }
      }
    }
  });
  if (!NEWNEW && is_new) {  // merge mode: new candidates skip new partners
#pragma unroll
    for (int s = 0; s < kRank; ++s) top[s] = kNone;
  }
  wave_sync();
  // phase 2: new candidates take their old partners from the block; the
  // other lanes read a valid slot and keep their phase 1 result
  uint32_t keep_top[kRank];
#pragma unroll
  for (int s = 0; s < kRank; ++s) keep_top[s] = top[s];
  const float* blk_col = s_buf[w] + (is_new ? static_cast<int>(lane) : 0);
  auto rank_old = [&](float acc, int j) {
    const uint32_t key = rank_key(acc, j);
    if (KEEP == 0) top[2] = key < top[2] ? key : top[2];
    else top_insert32<kRank>(top, key);
  };
  int o = 0;
  if (blocked) {
    for (; o + 4 <= no; o += 4, blk_col += 4 * kBst) {  // four reads in flight a step
      const float a0 = blk_col[0], a1 = blk_col[kBst];
      const float a2 = blk_col[2 * kBst], a3 = blk_col[3 * kBst];
      rank_old(a0, nn + o);
      rank_old(a1, nn + o + 1);
      rank_old(a2, nn + o + 2);
      rank_old(a3, nn + o + 3);
    }
    for (; o < no; ++o, blk_col += kBst) rank_old(*blk_col, nn + o);
  } else {
    join_quads<0, 16>([&](auto quad) {  // the pairs themselves
      constexpr int Q = decltype(quad)::value, j = 4 * Q;
      if (j + 4 <= nn || j >= nc) return;
      const f32x4 v = join_quad<D, Q>(own, own2, own_norm);
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (j + r >= nn && j + r < nc) rank_old(v[r], j + r);
    });
  }
  if (!is_new) {
#pragma unroll
    for (int s = 0; s < kRank; ++s) top[s] = keep_top[s];
  }
  // drop the lane itself: it ranks at most once, in phase 1
  uint32_t fin[kSlots];
  if (KEEP == 0) {
    const bool self0 = top[0] != kNone && (top[0] & 63u) == lane;
    fin[0] = self0 ? top[1] : top[0];
    fin[1] = top[2];
  } else {
    bool seen = false;
#pragma unroll
    for (int s = 0; s < kSlots; ++s) {
      seen = seen || (top[s] != kNone && (top[s] & 63u) == lane);
      fin[s] = seen ? top[s + 1] : top[s];
    }
  }
  // exact keys of the winners
  float dist[kSlots];
#pragma unroll
  for (int s = 0; s < kSlots; ++s) dist[s] = 0.0f;
#pragma unroll
  for (int c = 0; c < D; c += kCols) {
    wave_sync();
#pragma unroll
    for (int k = 0; k < kCols; k += 4)
      *reinterpret_cast<float4*>(&s_buf[w][lane * kRow + k]) =
          make_float4(own[c + k], own[c + k + 1], own[c + k + 2], own[c + k + 3]);
    wave_sync();
#pragma unroll
    for (int s = 0; s < kSlots; ++s) {
      // a branch per slot, so that one row's reads are in flight at a time:
      // with all the slots' reads first the kernel spills
      if (active && fin[s] != kNone) {
        const float* row = s_buf[w] + (fin[s] & 63u) * kRow;
#pragma unroll
        for (int k = 0; k < kCols && c + k < D; ++k) {
          const float diff = own[c + k] - row[k];
          dist[s] = __builtin_fmaf(diff, diff, dist[s]);
        }
      }
    }
  }
  uint64_t top64[kSlots];
#pragma unroll
  for (int s = 0; s < kSlots; ++s) {
    top64[s] = kKeyMax;
    if (active && fin[s] != kNone) top64[s] = make_key(dist[s], s_cand[w][fin[s] & 63u], 1u);
  }
  // Far from the origin the ranking values are rounding errors: where the
  // last winner's is off by a sixteenth of its distance for most candidates,
  // the wave ranks every partner by its distance.  (Unit clusters at 300k x 12,
  // join_keep 4: 300 off the origin no wave does, recall 0.987 in 9.4 ms; 1000 off
  // 0.960 -> 0.987 for 12.2 ms, 3000 off 0.334 -> 0.988 for 12.7 ms.)
  constexpr int kLast = KEEP == 0 ? 0 : kSlots - 1;
  const float last = dist[kLast];
  const bool has = active && fin[kLast] != kNone && last > 0.0f && last < __uint_as_float(0x7F800000u);
  const bool off = !(16.0f * __builtin_fabsf(__uint_as_float(fin[kLast] & ~63u) - last) <= last);
  if (2 * __popcll(__ballot(has && off)) > __popcll(__ballot(has))) {  // uniform
    const int me = static_cast<int>(lane), jb = is_new && !NEWNEW ? nn : 0, je = is_new ? nc : nn;
#pragma unroll
    for (int s = 0; s < kSlots; ++s) top64[s] = kKeyMax;
#pragma unroll 1
    for (int j = 0; j < nc; ++j) {
      const uint32_t id = __builtin_amdgcn_readfirstlane(s_cand[w][j]);
      const float* row = kPadded ? b.rows + static_cast<int64_t>(id) * 16 : X + static_cast<int64_t>(id) * D;
      float acc = 0.0f;
#pragma unroll
      for (int k = 0; k < D; ++k) {
        const float diff = own[k] - row[k];
        acc = __builtin_fmaf(diff, diff, acc);
      }
      const uint64_t key = active && j >= jb && j < je && j != me ? make_key(acc, id, 1u) : kKeyMax;
      if (KEEP != 0) top_insert<kSlots>(top64, key);
      else if (j < nn) top64[0] = key < top64[0] ? key : top64[0];
      else top64[1] = key < top64[1] ? key : top64[1];
    }
  }
  join_emit<WPB, kSlots>(b, top64, active, my_id, lim, nc, rev_drop);
}

// Key of a ranking value with no sign: its bits, the low 6 replaced by the
// partner's index j, which is wave-uniform.
__device__ __forceinline__ uint32_t rank_key6(float acc, int j) {
  const uint32_t mask_v = 0xFFFFFFC0u;  // a VGPR operand: VOP3 takes no literal here
  uint32_t r;
  asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(__float_as_uint(acc)), "v"(mask_v), "s"(j));
  return r;
}

// The kept partners of one candidate from its smallest 26-bit ranking keys
// (ascending): top holds one slot more than the kept and the next one, for
// the lane itself, which ranks at most once and is dropped here; KEEP == 0
// has its old partners' two smallest in told.  The `keep` smallest are
// exactly the `keep` nearest unless the last of them and the next one share
// all their distance bits, and then the wave ranks its partners again by full
// (distance, id) keys: about one wave in a hundred on continuous data, nearly
// every one on rounded coordinates or repeated points (kNN graph of 200k x 20,
// join_keep 4: 7.5 and 10.3 ms; 12.0 and 11.6 with u64 keys throughout).
// dist(j): the exact distance to partner j.
template <bool NEWNEW, int KEEP, int SLOTS, int RANK, typename F>
__device__ __forceinline__ void join_choose(const uint32_t (&top)[RANK], const uint32_t (&told)[2], int nn, int nc,
                                            int keep, const uint32_t* s_cand, F dist, uint64_t (&top64)[SLOTS]) {
  constexpr uint32_t kNone = 0xFFFFFFFFu;
  static_assert(RANK == (KEEP == 0 ? 3 : KEEP + 2) && SLOTS == (KEEP == 0 ? 2 : KEEP), "slots of the join");
  const int lane = static_cast<int>(__lane_id());
  const bool active = lane < nc, is_new = lane < nn;
  uint32_t fin[SLOTS], f[RANK - 1];
  bool seen = false, tie = false;
#pragma unroll
  for (int s = 0; s < RANK - 1; ++s) {
    // values first, then the choice: a choice between elements would become
    // an index, and the array would go to scratch memory
    const uint32_t here = top[s], next = top[s + 1];
    seen = seen || (here != kNone && static_cast<int>(here & 63u) == lane);
    f[s] = here ^ ((here ^ next) & (seen ? 0xFFFFFFFFu : 0u));
  }
  if (KEEP == 0) {
    fin[0] = f[0];
    fin[1] = told[0];
    tie = (f[1] != kNone && ((f[0] ^ f[1]) >> 6) == 0) || (told[1] != kNone && ((told[0] ^ told[1]) >> 6) == 0);
  } else {
    // bit s: slots s and s + 1 agree (a bit mask, so that no slot is indexed
    // by keep and the arrays stay in registers)
    uint32_t same = 0;
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) {
      fin[s] = s < keep ? f[s] : kNone;
      same |= (f[s + 1] != kNone && ((f[s] ^ f[s + 1]) >> 6) == 0 ? 1u : 0u) << s;
    }
    tie = ((same >> (keep - 1)) & 1u) != 0;
  }
#pragma unroll
  for (int s = 0; s < SLOTS; ++s) {
    top64[s] = kKeyMax;
    if (active && fin[s] != kNone) {
      const int j = static_cast<int>(fin[s] & 63u);
      top64[s] = make_key(dist(j), s_cand[j], 1u);
    }
  }
  if (__ballot(active && tie)) {  // uniform: rank every partner by its full key
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) top64[s] = kKeyMax;
    const int jb = is_new ? (NEWNEW ? 0 : nn) : 0, je = is_new ? nc : nn;
    for (int j = 0; j < nc; ++j) {
      if (!(active && j >= jb && j < je && j != lane)) continue;
      const uint64_t key = make_key(dist(j), s_cand[j], 1u);
      if (KEEP == 0) {
        if (j < nn) top64[0] = key < top64[0] ? key : top64[0];
        else top64[1] = key < top64[1] ? key : top64[1];
      } else {
        top_insert<SLOTS>(top64, key);
      }
    }
    if (KEEP != 0) {
#pragma unroll
      for (int s = 0; s < SLOTS; ++s)
        if (s >= keep) top64[s] = kKeyMax;
    }
  }
}

// FP32 join for d <= 31 other than 12 (d = 12 and 32 have k_nnd_join2): exact
// distances, with the candidates' padded rows in LDS and the lane's own row
// in registers (DP: 4, 8, 12, 16, 20, 24 or 32 columns; the zeros past d add
// nothing to a distance, but d = 25 to 28 pay for 32: six launches at 200k and
// join_keep 4 take 4.5 ms at d = 25, 3.9 with 28 columns).  As in k_nnd_join2
// each old-new pair is evaluated once (a distance has the same bits both ways)
// and passed to the new lane through an LDS block.  Ranking uses 32-bit keys
// (rank_key6, join_choose).  KEEP is 0, or the largest join_keep the kernel
// serves: 4 or 8, as the spare slots cost little (d = 20, join_keep 1: 2.74 ms,
// 2.56 with a kernel of its own; from 3 on nothing).
// Bound by VALU issue (two instructions per dimension and pair): six launches
// at 200k points and join_keep 4 take 1.62 ms at d = 8, 2.31 at 16, 2.78 at
// 20 and 4.49 at 31, where u64 keys and the lane's own row read from LDS took
// 3.27, 4.19, 5.67 and 10.94.
template <int DP, bool NEWNEW, int KEEP>
__global__ __launch_bounds__(kJoinWaves * 64) void k_nnd_join_rows(int64_t n, int d, int S, int keep, NndBufs b) {
  constexpr int WPB = kJoinWaves;
  constexpr int kSlots = KEEP == 0 ? 2 : KEEP;
  constexpr int kRank = KEEP == 0 ? 3 : KEEP + 2;  // the kept, the next one, and the lane itself
  constexpr int kBlock = 384;                      // as in k_nnd_join2
  constexpr uint32_t kNone = 0xFFFFFFFFu;
  __shared__ __attribute__((aligned(16))) float s_vec[WPB][64 * DP];
  __shared__ float s_blk[WPB][kBlock];
  __shared__ uint32_t s_cand[WPB][64];
  const unsigned lane = __lane_id();
  const unsigned w = threadIdx.x >> 6;
  const int64_t p = static_cast<int64_t>(blockIdx.x) * WPB + w;

  int nn, nc, rev_drop;
  join_candidates(b, p, p < n, S, s_cand[w], &nn, &nc, &rev_drop);
  const int no = nc - nn;
  const bool active = lane < static_cast<unsigned>(nc);
  const bool is_new = lane < static_cast<unsigned>(nn);
  const uint32_t my_id = active ? s_cand[w][lane] : 0u;
  float own[DP];
  float lim = 0.0f;
#pragma unroll
  for (int k = 0; k < DP; ++k) own[k] = 0.0f;
  if (active) {
    // the row ends with the list bound; columns in [d, rstride - 1) are zero
    const float* src = b.rows + static_cast<int64_t>(my_id) * b.rstride;
#pragma unroll
    for (int q = 0; q < DP / 4; ++q) {
      const float4 v = reinterpret_cast<const float4*>(src)[q];
      own[4 * q] = v.x, own[4 * q + 1] = v.y, own[4 * q + 2] = v.z, own[4 * q + 3] = v.w;
    }
    lim = src[b.rstride - 1];
    if (DP == b.rstride) own[DP - 1] = 0.0f;
#pragma unroll
    for (int q = 0; q < DP / 4; ++q)
      *reinterpret_cast<float4*>(&s_vec[w][lane * DP + 4 * q]) =
          make_float4(own[4 * q], own[4 * q + 1], own[4 * q + 2], own[4 * q + 3]);
  }
  wave_sync();

  auto partner = [&](int j) {
    const float* row = s_vec[w] + j * DP;
    float acc = 0.0f;
#pragma unroll
    for (int q = 0; q < DP / 4; ++q) {
      const float4 v = *reinterpret_cast<const float4*>(row + 4 * q);
      float diff = own[4 * q] - v.x;
      acc = __builtin_fmaf(diff, diff, acc);
      diff = own[4 * q + 1] - v.y;
      acc = __builtin_fmaf(diff, diff, acc);
      diff = own[4 * q + 2] - v.z;
      acc = __builtin_fmaf(diff, diff, acc);
      diff = own[4 * q + 3] - v.w;
      acc = __builtin_fmaf(diff, diff, acc);
    }
    return acc;
  };
  // top: partners among the new candidates (phase 1), then for a new lane
  // the old ones too; KEEP == 0 ranks the old ones apart (told)
  uint32_t top[kRank], told[2] = {kNone, kNone};
#pragma unroll
  for (int s = 0; s < kRank; ++s) top[s] = kNone;
  const int bst = nn + 1;  // odd-or-padded row stride of the old x new block
  const bool blocked = no * bst <= kBlock;  // uniform
  const bool store_old = active && !is_new && blocked;
  float* blk_row = s_blk[w] + (store_old ? (static_cast<int>(lane) - nn) * bst : 0);  // + j
  int j = 0;
  for (; j + 2 <= nn; j += 2) {
    const float a0 = partner(j);
    const float a1 = partner(j + 1);
    if (store_old) {
      blk_row[j] = a0;
      blk_row[j + 1] = a1;
    }
    top_insert32<kRank>(top, rank_key6(a0, j));
    top_insert32<kRank>(top, rank_key6(a1, j + 1));
  }
  if (j < nn) {
    const float a0 = partner(j);
    if (store_old) blk_row[j] = a0;
    top_insert32<kRank>(top, rank_key6(a0, j));
  }
  if (!NEWNEW && is_new) {  // merge mode: new candidates skip new partners
#pragma unroll
    for (int s = 0; s < kRank; ++s) top[s] = kNone;
  }
  wave_sync();
  uint32_t keep_top[kRank];
#pragma unroll
  for (int s = 0; s < kRank; ++s) keep_top[s] = top[s];
  const float* blk_col = s_blk[w] + (is_new ? static_cast<int>(lane) : 0);
  auto rank_old = [&](float acc, int jj) {
    if (KEEP == 0) top_insert32<2>(told, rank_key6(acc, jj));
    else top_insert32<kRank>(top, rank_key6(acc, jj));
  };
  int o = 0;
  if (blocked) {
    for (; o + 4 <= no; o += 4) {  // four reads in flight a step
      const float a0 = blk_col[o * bst], a1 = blk_col[(o + 1) * bst];
      const float a2 = blk_col[(o + 2) * bst], a3 = blk_col[(o + 3) * bst];
      rank_old(a0, nn + o);
      rank_old(a1, nn + o + 1);
      rank_old(a2, nn + o + 2);
      rank_old(a3, nn + o + 3);
    }
    for (; o < no; ++o) rank_old(blk_col[o * bst], nn + o);
  } else {
    for (; o < no; ++o) rank_old(partner(nn + o), nn + o);
  }
  if (!is_new) {
#pragma unroll
    for (int s = 0; s < kRank; ++s) top[s] = keep_top[s];
    told[0] = told[1] = kNone;
  }
  uint64_t top64[kSlots];
  join_choose<NEWNEW, KEEP>(top, told, nn, nc, keep, s_cand[w], partner, top64);
  join_emit<WPB, kSlots>(b, top64, active, my_id, lim, nc, rev_drop);
}

// FP32 join for d > 32: exact distances, the dimensions taken 16 at a time.
// Per chunk the wave stages its candidates' 16 columns in LDS (quad q of row
// r at q ^ ((r >> 1) & 3), so that the lanes' 16-byte stores spread over the
// banks)
// and every lane adds the chunk to its distances to the new candidates, which
// stay in registers (at most 32); the additions run in dimension order, so
// the distances have the bits of the other forms.  The distances then go to
// LDS in place of the rows (entry (j, lane) at 65 j + lane), where the new
// lanes also find theirs to the old candidates.  Bound by VALU issue, two
// instructions per dimension and pair: six launches at join_keep 4 take 5.5 ms
// at 200k x 40, 6.7 at 200k x 64 and 5.7 at 100k x 128, where the lane's own row
// read from LDS and u64 keys took 11.5, 19.6 and 29.9.
template <bool NEWNEW, int KEEP>
__global__ __launch_bounds__(kJoinWaves * 64, 4) void k_nnd_join_wide(const float* __restrict__ X, int64_t n, int d,
                                                                   int S, int keep, NndBufs b) {
  constexpr int WPB = kJoinWaves;
  constexpr int kSlots = KEEP == 0 ? 2 : KEEP;
  constexpr int kRank = KEEP == 0 ? 3 : KEEP + 2;
  constexpr int kNew = 32;  // new candidates at most (join_candidates)
  constexpr int kC = 16;    // columns per chunk
  constexpr int kM = 65;    // stride of the distance block
  constexpr uint32_t kNone = 0xFFFFFFFFu;
  __shared__ __attribute__((aligned(16))) float s_buf[WPB][kNew * kM];
  static_assert(kNew * kM >= 64 * kC && (kNew * kM) % 4 == 0, "rows and distances share the buffer");
  __shared__ uint32_t s_cand[WPB][64];
  const unsigned lane = __lane_id();
  const unsigned w = threadIdx.x >> 6;
  const int64_t p = static_cast<int64_t>(blockIdx.x) * WPB + w;
  float* buf = s_buf[w];

  int nn, nc, rev_drop;
  join_candidates(b, p, p < n, S, s_cand[w], &nn, &nc, &rev_drop);
  const int no = nc - nn;
  const bool active = lane < static_cast<unsigned>(nc);
  const bool is_new = lane < static_cast<unsigned>(nn);
  const uint32_t my_id = active ? s_cand[w][lane] : 0u;
  const float lim = active ? b.worst[static_cast<int64_t>(my_id) * b.wstride] : 0.0f;
  const float* src = X + static_cast<int64_t>(my_id) * d;
  const bool vec4 = (d & 3) == 0 && (reinterpret_cast<uintptr_t>(X) & 15) == 0;  // uniform

  float acc[kNew];
#pragma unroll
  for (int j = 0; j < kNew; ++j) acc[j] = 0.0f;
  for (int c0 = 0; c0 < d; c0 += kC) {
    float own[kC];
#pragma unroll
    for (int k = 0; k < kC; ++k) own[k] = 0.0f;
    if (active) {
      if (vec4) {
#pragma unroll
        for (int q = 0; q < kC / 4; ++q)
          if (c0 + 4 * q < d) {
            const float4 v = *reinterpret_cast<const float4*>(src + c0 + 4 * q);
            own[4 * q] = v.x, own[4 * q + 1] = v.y, own[4 * q + 2] = v.z, own[4 * q + 3] = v.w;
          }
      } else {
#pragma unroll
        for (int k = 0; k < kC; ++k)
          if (c0 + k < d) own[k] = src[c0 + k];
      }
    }
    wave_sync();  // the previous chunk (and the candidate scratch) has been read
#pragma unroll
    for (int q = 0; q < kC / 4; ++q)
      *reinterpret_cast<float4*>(buf + lane * kC + 4 * (q ^ static_cast<int>((lane >> 1) & 3))) =
          make_float4(own[4 * q], own[4 * q + 1], own[4 * q + 2], own[4 * q + 3]);
    wave_sync();
#pragma unroll
    for (int j0 = 0; j0 < kNew; j0 += 4) {
      if (j0 < nn) {  // uniform
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int j = j0 + u;
          float a = acc[j];
#pragma unroll
          for (int q = 0; q < kC / 4; ++q) {
            const float4 v = *reinterpret_cast<const float4*>(buf + j * kC + 4 * (q ^ ((j >> 1) & 3)));
            float diff = own[4 * q] - v.x;
            a = __builtin_fmaf(diff, diff, a);
            diff = own[4 * q + 1] - v.y;
            a = __builtin_fmaf(diff, diff, a);
            diff = own[4 * q + 2] - v.z;
            a = __builtin_fmaf(diff, diff, a);
            diff = own[4 * q + 3] - v.w;
            a = __builtin_fmaf(diff, diff, a);
          }
          acc[j] = a;
        }
      }
    }
  }
  wave_sync();
  uint32_t top[kRank], told[2] = {kNone, kNone};
#pragma unroll
  for (int s = 0; s < kRank; ++s) top[s] = kNone;
#pragma unroll
  for (int j = 0; j < kNew; ++j) {
    if (j < nn) {  // uniform
      buf[j * kM + lane] = acc[j];
      top_insert32<kRank>(top, rank_key6(acc[j], j));
    }
  }
  if (!NEWNEW && is_new) {  // merge mode: new candidates skip new partners
#pragma unroll
    for (int s = 0; s < kRank; ++s) top[s] = kNone;
  }
  wave_sync();
  uint32_t keep_top[kRank];
#pragma unroll
  for (int s = 0; s < kRank; ++s) keep_top[s] = top[s];
  const float* to_old = buf + (is_new ? static_cast<int>(lane) : 0) * kM + nn;
  auto rank_old = [&](float a, int jj) {
    if (KEEP == 0) top_insert32<2>(told, rank_key6(a, jj));
    else top_insert32<kRank>(top, rank_key6(a, jj));
  };
  int o = 0;
  for (; o + 4 <= no; o += 4) {  // four reads in flight a step
    const float a0 = to_old[o], a1 = to_old[o + 1], a2 = to_old[o + 2], a3 = to_old[o + 3];
    rank_old(a0, nn + o);
    rank_old(a1, nn + o + 1);
    rank_old(a2, nn + o + 2);
    rank_old(a3, nn + o + 3);
  }
  for (; o < no; ++o) rank_old(to_old[o], nn + o);
  if (!is_new) {
#pragma unroll
    for (int s = 0; s < kRank; ++s) top[s] = keep_top[s];
    told[0] = told[1] = kNone;
  }
  uint64_t top64[kSlots];
  join_choose<NEWNEW, KEEP>(
      top, told, nn, nc, keep, s_cand[w],
      [&](int j) { return j < nn ? buf[j * kM + lane] : buf[lane * kM + j]; }, top64);
  join_emit<WPB, kSlots>(b, top64, active, my_id, lim, nc, rev_drop);
}

// BF16 join (distance_mode 1): the 64 x 64 Gram matrix of the candidates is
// computed with v_mfma_f32_16x16x32_bf16 (BF16 inputs, FP32 accumulation),
// with the operands swapped so that lane l holds row I*16 + (l % 16) and
// columns J*16 + 4*(l / 16) + q of tile (I, J).  Each lane ranks its rows'
// partners by the approximate |x|^2 + |y|^2 - 2 x.y (32-bit keys), the four
// lanes that share a row merge their shortlists, and each candidate's SHORT
// nearest partners are re-ranked with the exact FP32 formula, so proposals --
// and therefore lists, core distances and MST weights -- carry exact FP32
// distances only.
// Lane layout of the 16x16x32 instruction: A/B lane l holds row (l % 16),
// k = 8*(l/16) .. +7; the result lane l holds rows 4*(l/16) + q, column l % 16.
// The gather uses that layout: lane l loads 8 columns of its row of each
// tile, which are the tile's fragment once rounded (one for both operands),
// and all 16 tiles accumulate in registers.  The re-rank gathers the rows a
// second time, 32 columns at a time through LDS, and every lane adds each
// chunk to the distances of its whole shortlist: reading them again (from a
// cache, mostly) keeps the LDS of a wave at 10 KB and its chains in parallel,
// where holding 64 whole FP32 rows left four waves to a CU, each ranking one
// partner after the other.  A launch at 100k x 128 and join_keep 4 takes 0.77
// ms (2.19 in that form; 0.99 with the next chunk's columns in registers of
// their own, which spill).
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

template <int N>
__device__ __forceinline__ void merge_short(uint32_t (&a)[N], int xor_mask) {
  uint32_t o[N];
#pragma unroll
  for (int s = 0; s < N; ++s) o[s] = __shfl_xor(a[s], xor_mask);
#pragma unroll
  for (int s = 0; s < N; ++s) top_insert32<N>(a, o[s]);
}

template <bool NEWNEW, int KEEP, int SHORT>
__global__ __launch_bounds__(64, SHORT <= 6 ? 3 : 2) void k_nnd_join_mfma(const float* __restrict__ X, int64_t n, int d, int dp, int S,
                                                      NndBufs b) {
  constexpr int WPB = 1;
  constexpr int kSlots = KEEP == 0 ? 2 : KEEP;
  constexpr int kShort = SHORT;  // BF16 shortlist re-ranked in FP32 per candidate
  static_assert(KEEP == 0 ? SHORT == 2 : SHORT >= KEEP, "the shortlist holds the kept partners");
  constexpr uint32_t kNone = 0xFFFFFFFFu;
  constexpr int kRs = 36;  // LDS row stride of a 32-column chunk (16-byte aligned rows)
  __shared__ __attribute__((aligned(16))) float s_vec[64 * kRs];
  __shared__ uint32_t s_cand[WPB][64];
  __shared__ float s_norm[64];
  const unsigned lane = __lane_id();
  const int64_t p = blockIdx.x;

  int nn, nc, rev_drop;
  join_candidates(b, p, p < n, S, s_cand[0], &nn, &nc, &rev_drop);

  const bool active = lane < static_cast<unsigned>(nc);
  const uint32_t my_id = active ? s_cand[0][lane] : 0u;
  const float lim = active ? b.worst[static_cast<int64_t>(my_id) * b.wstride] : 0.0f;
  s_norm[lane] = active ? b.norms[my_id] : 0.0f;
  const int tiles = (nc + 15) >> 4;
  const int r16 = static_cast<int>(lane & 15), kq = static_cast<int>(lane >> 4);
  const bool vec4 = (d & 3) == 0 && (reinterpret_cast<uintptr_t>(X) & 15) == 0;  // uniform
  // this lane's row of tile I, from its first column 8 kq on
  const float* src[4];
  bool has[4];
#pragma unroll
  for (int I = 0; I < 4; ++I) {
    has[I] = I * 16 + r16 < nc;
    src[I] = X + static_cast<int64_t>(has[I] ? s_cand[0][I * 16 + r16] : 0u) * d + 8 * kq;
  }
  // columns [k0 + 8 kq, + 8) of those rows; zeros past d and past nc
  auto load = [&](int k0, float (&v)[4][8]) {
#pragma unroll
    for (int I = 0; I < 4; ++I) {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[I][e] = 0.0f;
      if (I < tiles && has[I]) {
        const int left = d - k0 - 8 * kq;
        if (vec4) {
          if (left >= 4) {
            const float4 x = *reinterpret_cast<const float4*>(src[I] + k0);
            v[I][0] = x.x, v[I][1] = x.y, v[I][2] = x.z, v[I][3] = x.w;
          }
          if (left >= 8) {
            const float4 x = *reinterpret_cast<const float4*>(src[I] + k0 + 4);
            v[I][4] = x.x, v[I][5] = x.y, v[I][6] = x.z, v[I][7] = x.w;
          }
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (e < left) v[I][e] = src[I][k0 + e];
        }
      }
    }
  };
  f32x4_t acc[4][4];
#pragma unroll
  for (int I = 0; I < 4; ++I)
#pragma unroll
    for (int J = 0; J < 4; ++J) acc[I][J] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  float cur[4][8];
  load(0, cur);
  for (int k0 = 0; k0 < dp; k0 += 32) {
    bf16x8_t f[4];
#pragma unroll
    for (int I = 0; I < 4; ++I) {
#pragma unroll
      for (int e = 0; e < 8; ++e) f[I][e] = static_cast<__bf16>(cur[I][e]);
    }
    if (k0 + 32 < dp) load(k0 + 32, cur);  // uniform: in flight during this chunk's products
#pragma unroll
    for (int I = 0; I < 4; ++I)
#pragma unroll
      for (int J = 0; J < 4; ++J)
        // uniform; old x old tiles are never joined
        if (I < tiles && J < tiles && !(I * 16 >= nn && J * 16 >= nn))
          acc[I][J] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f[J], f[I], acc[I][J], 0, 0, 0);
  }
  __syncthreads();

  uint32_t sl[4][kShort];
#pragma unroll
  for (int I = 0; I < 4; ++I) {
#pragma unroll
    for (int s = 0; s < kShort; ++s) sl[I][s] = kNone;
    if (I < tiles) {  // uniform across the wave
      const int row = I * 16 + r16;
      const bool row_new = row < nn, row_live = row < nc;
      const float nrow = s_norm[row];
#pragma unroll
      for (int J = 0; J < 4; ++J) {
        if (J >= tiles || (I * 16 >= nn && J * 16 >= nn)) continue;  // uniform
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int col = J * 16 + 4 * kq + q;
          const bool ok = row_live && col < nc && col != row &&
                          (row_new ? (NEWNEW || col >= nn) : (col < nn));
          const float a = nrow + s_norm[col] - 2.0f * acc[I][J][q];
          const uint32_t key = ok ? ((order_bits(a) & ~63u) | static_cast<uint32_t>(col)) : kNone;
          if (KEEP == 0) {
            if (col < nn) sl[I][0] = key < sl[I][0] ? key : sl[I][0];
            else sl[I][1] = key < sl[I][1] ? key : sl[I][1];
          } else {
            top_insert32<kShort>(sl[I], key);
          }
        }
      }
    }
  }
  // the four lanes holding one row (same l % 16) merge their shortlists
#pragma unroll
  for (int I = 0; I < 4; ++I) {
    if (KEEP == 0) {
#pragma unroll
      for (int m = 16; m <= 32; m <<= 1) {
        const uint32_t o0 = __shfl_xor(sl[I][0], m), o1 = __shfl_xor(sl[I][1], m);
        sl[I][0] = o0 < sl[I][0] ? o0 : sl[I][0];
        sl[I][1] = o1 < sl[I][1] ? o1 : sl[I][1];
      }
    } else {
      merge_short<kShort>(sl[I], 16);
      merge_short<kShort>(sl[I], 32);
    }
  }
  // lane c is candidate c: its row's shortlist is sl[c / 16]
  uint32_t mine[kShort];
#pragma unroll
  for (int s = 0; s < kShort; ++s) {
    const uint32_t v0 = sl[0][s], v1 = sl[1][s], v2 = sl[2][s], v3 = sl[3][s];
    mine[s] = kq == 0 ? v0 : (kq == 1 ? v1 : (kq == 2 ? v2 : v3));
  }

  // exact FP32 re-rank of the shortlist (zeros past d add nothing)
  int js[kShort];
  float e[kShort];
#pragma unroll
  for (int s = 0; s < kShort; ++s) {
    js[s] = mine[s] == kNone ? 0 : static_cast<int>(mine[s] & 63u);
    e[s] = 0.0f;
  }
  load(0, cur);
  for (int k0 = 0; k0 < dp; k0 += 32) {
    wave_sync();  // the previous chunk has been read
#pragma unroll
    for (int I = 0; I < 4; ++I) {
      float* dst = s_vec + (I * 16 + r16) * kRs + 8 * kq;
      *reinterpret_cast<float4*>(dst) = make_float4(cur[I][0], cur[I][1], cur[I][2], cur[I][3]);
      *reinterpret_cast<float4*>(dst + 4) = make_float4(cur[I][4], cur[I][5], cur[I][6], cur[I][7]);
    }
    wave_sync();
    if (k0 + 32 < dp) load(k0 + 32, cur);  // uniform: in flight during this chunk's sums
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const float4 x = *reinterpret_cast<const float4*>(s_vec + lane * kRs + 4 * q);
#pragma unroll
      for (int s = 0; s < kShort; ++s) {
        const float4 y = *reinterpret_cast<const float4*>(s_vec + js[s] * kRs + 4 * q);
        float diff = x.x - y.x;
        e[s] = __builtin_fmaf(diff, diff, e[s]);
        diff = x.y - y.y;
        e[s] = __builtin_fmaf(diff, diff, e[s]);
        diff = x.z - y.z;
        e[s] = __builtin_fmaf(diff, diff, e[s]);
        diff = x.w - y.w;
        e[s] = __builtin_fmaf(diff, diff, e[s]);
      }
    }
  }
  uint64_t top[kSlots];
#pragma unroll
  for (int s = 0; s < kSlots; ++s) top[s] = kKeyMax;
#pragma unroll
  for (int s = 0; s < kShort; ++s) {
    if (!active || mine[s] == kNone) continue;
    const uint64_t key = make_key(e[s], s_cand[0][js[s]], 1u);
    if (KEEP == 0) {
      if (js[s] < nn) top[0] = key < top[0] ? key : top[0];
      else top[1] = key < top[1] ? key : top[1];
    } else {
      top_insert<kSlots>(top, key);
    }
  }
  join_emit<WPB, kSlots>(b, top, active, my_id, lim, nc, rev_drop);
}

// |x|^2 of every point in dimension order (the BF16 join's ranking).
__global__ __launch_bounds__(256) void k_nnd_norms(const float* __restrict__ X, int64_t n, int d,
                                                   float* __restrict__ norms) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float* r = X + i * d;
  float s = 0.0f;
  for (int k = 0; k < d; ++k) s = __builtin_fmaf(r[k], r[k], s);
  norms[i] = s;
}

// ----------------------------------------------------------- list update --
// InsertToGlobalGraph (nndescent.cu:969-1028) without locks.  Proposals are
// sorted by target >> 4, so a block owns a group of 16 lists and their
// proposals: it stages the proposals in LDS tiles, buckets them by target
// (order inside a bucket does not matter), and each wave merges four
// buckets into their lists.
__device__ __forceinline__ uint64_t bitonic_merge64(uint64_t v) {
  const unsigned lane = __lane_id();
#pragma unroll
  for (int j = 32; j > 0; j >>= 1) v = bitonic_ce(v, lane_xor_u64(v, j), (lane & j) == 0);
  return v;
}

// Merges up to 64 proposals (one per lane, kKeyMax for none) into the list
// held in lanes 0..31 of cur (ascending keys; old entries carry flag 0) and
// returns it: the chunk is sorted across the wave and made unique, its 32
// smallest distinct keys are reversed into lanes 32..63 (no other proposal of
// the chunk can be among the 32 smallest of the union), and a 64-wide
// bitonic merge with the list keeps the 32 smallest distinct (distance, id)
// keys -- an existing entry wins over a proposal of the same id, so it stays
// old.  s_prop and s_top are this wave's 32-entry LDS rows.
__device__ __forceinline__ uint64_t merge_proposals(uint64_t cur, uint64_t pr, uint64_t* s_prop, uint64_t* s_top) {
  const unsigned lane = __lane_id();
  const uint64_t lt = lanemask_lt();
  pr = bitonic_group<64>(pr);
  const uint64_t pp = lane_below(pr);
  const bool kp = pr != kKeyMax && (lane == 0 || pp != pr);
  const uint64_t bp = __ballot(kp);
  const int ppos = __popcll(bp & lt);
  const int ptot = __popcll(bp);
  if (kp && ppos < 32) s_prop[ppos] = pr;
  if (static_cast<int>(lane) >= ptot && lane < 32u) s_prop[lane] = kKeyMax;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  const uint64_t pv = s_prop[(63u - lane) & 31u];
  uint64_t v = lane < 32 ? cur : pv;
  __builtin_amdgcn_wave_barrier();
  v = bitonic_merge64(v);
  const uint64_t prev = lane_below(v);
  const bool keep = v != kKeyMax && (lane == 0 || (prev >> 1) != (v >> 1));
  const uint64_t bal = __ballot(keep);
  const int pos = __popcll(bal & lt);
  const int total = __popcll(bal);
  if (keep && pos < kK) s_top[pos] = v;
  if (static_cast<int>(lane) >= total && lane < 32u) s_top[lane] = kKeyMax;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  const uint64_t tv = s_top[lane & 31u];
  __builtin_amdgcn_wave_barrier();
  return lane < 32 ? tv : kKeyMax;
}

// The list in lanes 0..31 (sorted, distinct) merged with the proposals
// (kKeyMax: none; each distinct from the list's entries, `pos` = # entries
// below it): every element's new position is counted, with no sort.  Of
// equal proposals one is kept: the step of the first takes the others out,
// so a step is two reads, three compares and two additions (about twice
// that with the repeated proposals found lane by lane: an update of 1M lists
// at join_keep 3 took 1.04 ms, now 0.85; of 10M at join_keep 2 6.5, now 5.4).
// Returns the new list in lanes 0..31; s_top is the wave's 32-entry LDS row.
__device__ __forceinline__ uint64_t insert_few(uint64_t cur, uint64_t pr, int pos, uint64_t* s_top) {
  const unsigned lane = __lane_id();
  const uint64_t live = __ballot(pr != kKeyMax);
  uint64_t first = 0;  // the lanes whose proposal enters
  int below_cur = 0, below_pr = 0;
  for (uint64_t m = live; m;) {  // uniform
    const int t = __builtin_ctzll(m);
    const uint64_t x = (static_cast<uint64_t>(__builtin_amdgcn_readlane(static_cast<uint32_t>(pr >> 32), t)) << 32) |
                       __builtin_amdgcn_readlane(static_cast<uint32_t>(pr), t);
    first |= 1ull << t;
    m &= ~__ballot(pr == x);
    below_cur += x < cur ? 1 : 0;
    below_pr += x < pr ? 1 : 0;
  }
  const int pc = static_cast<int>(lane) + below_cur;
  if (lane < 32u && pc < kK) s_top[pc] = cur;
  const int pp = pos + below_pr;
  if (((first >> lane) & 1u) && pp < kK) s_top[pp] = pr;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  const uint64_t tv = s_top[lane & 31u];
  __builtin_amdgcn_wave_barrier();
  return lane < 32 ? tv : kKeyMax;
}

constexpr int kGroupBits = 4;     // lists per update block: 16
constexpr int kGroupTile = 1024;  // proposals staged per LDS tile

constexpr int kUpdFull = 1;   // merge (and so deduplicate) every list, with or without proposals
constexpr int kUpdStrip = 2;  // write labels without the old flag (the last iteration)

// One block of 4 waves per group g of lists [16g, 16g + 16); prop_s/prop_e[g]
// bound the group's proposals; each wave merges four lists.  kUpdFull: merge
// (and so deduplicate) every list even without proposals (first iteration);
// otherwise a list without proposals is only marked old.
__global__ __launch_bounds__(256, 7) void k_nnd_update(hdb_nnd_element* __restrict__ lists, int64_t n, NndBufs b,
                                                    int flags) {
  const bool full = (flags & kUpdFull) != 0;
  constexpr int G = 1 << kGroupBits;
  __shared__ uint64_t s_cur[G][32];
  __shared__ uint64_t s_key[kGroupTile];
  __shared__ uint64_t s_prop[4][32];
  __shared__ uint64_t s_top[4][32];
  __shared__ int32_t s_cnt[G], s_start[G], s_hit[G];
  const unsigned lane = __lane_id();
  const unsigned w = threadIdx.x >> 6;
  const int64_t g = blockIdx.x;
  const int64_t t0 = g << kGroupBits;
  for (int idx = threadIdx.x; idx < G * 32; idx += 256) {
    const int q = idx >> 5, j = idx & 31;
    const int64_t t = t0 + q;
    uint64_t key = kKeyMax;
    if (t < n) {
      const hdb_nnd_element e = lists[t * kK + j];
      const uint32_t id = label_id(e.label);
      key = (id == kInvalidId) ? kKeyMax : make_key(e.distance, id, 0u);
    }
    s_cur[q][j] = key;
  }
  if (threadIdx.x < G) s_hit[threadIdx.x] = 0;
  const int64_t gs = b.prop_s[g], ge = b.prop_e[g];
  __syncthreads();
  for (int64_t base = gs; base < ge; base += kGroupTile) {
    const int cnt = static_cast<int>(ge - base < kGroupTile ? ge - base : kGroupTile);
    if (threadIdx.x < G) s_cnt[threadIdx.x] = 0;
    __syncthreads();
    int rb[kGroupTile / 256], rr[kGroupTile / 256];
    uint64_t rk[kGroupTile / 256];
#pragma unroll
    for (int u = 0; u < kGroupTile / 256; ++u) {
      const int i = static_cast<int>(threadIdx.x) + u * 256;
      rb[u] = -1;
      rr[u] = 0;
      rk[u] = kKeyMax;
      if (i < cnt) {
        rb[u] = static_cast<int>(b.prop_tgt[base + i] & (G - 1));
        rk[u] = b.prop_key[base + i];
        rr[u] = atomicAdd(&s_cnt[rb[u]], 1);
      }
    }
    __syncthreads();
    if (threadIdx.x < G) {
      int acc = 0;
      for (unsigned c = 0; c < threadIdx.x; ++c) acc += s_cnt[c];
      s_start[threadIdx.x] = acc;
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kGroupTile / 256; ++u)
      if (rb[u] >= 0) s_key[s_start[rb[u]] + rr[u]] = rk[u];
    __syncthreads();
    for (int q4 = 0; q4 < G / 4; ++q4) {
      const int q = static_cast<int>(w) * (G / 4) + q4;
      const int c = s_cnt[q];
      if (c == 0) continue;  // uniform across the wave
      uint64_t cur = s_cur[q][lane & 31u];
      cur = lane < 32 ? cur : kKeyMax;
      const uint64_t* lst = s_cur[q];  // the list as it stands, sorted, in LDS
      for (int c0 = 0; c0 < c; c0 += 64) {
        uint64_t pr = c0 + static_cast<int>(lane) < c ? s_key[s_start[q] + c0 + lane] : kKeyMax;
        if (!full) {
          // After the first iteration lists are distinct, so a proposal that
          // ranks past the 32nd entry, or equals an entry's (distance, id),
          // cannot change the list: drop it, and skip the merge when none is
          // left.
          // entries below the proposal, capped at 31, in three dependent
          // rounds of LDS reads (an 8-entry block, a pair within it, then
          // one entry) where a binary search takes five.  A proposal carries
          // flag 1, so an entry's (distance, id) is below its own exactly if
          // the entry is below the proposal's key with the flag clear.
          const uint64_t pk = pr & ~1ull;
          int pos = (lst[7] < pk ? 8 : 0) + (lst[15] < pk ? 8 : 0) + (lst[23] < pk ? 8 : 0);
          pos += (lst[pos + 1] < pk ? 2 : 0) + (lst[pos + 3] < pk ? 2 : 0) + (lst[pos + 5] < pk ? 2 : 0);
          if (lst[pos] < pk) pos += 1;
          // lst[pos] >= pk unless all 32 entries are below it (pos = 31)
          pr = lst[pos] > pr ? pr : kKeyMax;
          const bool keep = pr != kKeyMax;
          const uint64_t km = __ballot(keep);
          if (km == 0) continue;
          // counting costs a step per proposal; past about 32 the sort wins
          if (__popcll(km) <= 32) cur = insert_few(cur, pr, pos, s_top[w]);
          else cur = merge_proposals(cur, pr, s_prop[w], s_top[w]);
        } else {
          cur = merge_proposals(cur, pr, s_prop[w], s_top[w]);
        }
        lst = s_top[w];
      }
      if (lane < 32) s_cur[q][lane] = cur;
      if (lane == 0) s_hit[q] = 1;
    }
    __syncthreads();
  }
  for (int q4 = 0; q4 < G / 4; ++q4) {
    const int q = static_cast<int>(w) * (G / 4) + q4;
    const int64_t t = t0 + q;
    if (t >= n) break;  // uniform across the wave; later lists are past n too
    uint64_t cur = s_cur[q][lane & 31u];
    cur = lane < 32 ? cur : kKeyMax;
    if (full && !s_hit[q]) cur = merge_proposals(cur, kKeyMax, s_prop[w], s_top[w]);
    if (lane < 32) lists[t * kK + lane] = key_to_elem((flags & kUpdStrip) ? (cur | 1u) : cur);
    if (lane == 31) b.worst[t * b.wstride] = (cur == kKeyMax) ? __uint_as_float(0x7F800000u) : key_d2(cur);
  }
}

// Strip old flags so exported labels are >= 0.
__global__ void k_nnd_finalize(hdb_nnd_element* __restrict__ lists, int64_t total) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < total) {
    const int32_t lab = lists[i].label;
    if (lab < 0) lists[i].label = -lab - 1;
  }
}

__global__ __launch_bounds__(256) void k_sum_parts(const unsigned long long* __restrict__ part, int64_t blocks,
                                                   unsigned long long* __restrict__ out) {
  __shared__ unsigned long long acc[4][256];
  unsigned long long a[4] = {0, 0, 0, 0};
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; i < blocks;
       i += static_cast<int64_t>(gridDim.x) * 256)
    for (int q = 0; q < 4; ++q) a[q] += part[4 * i + q];
  for (int q = 0; q < 4; ++q) acc[q][threadIdx.x] = a[q];
  __syncthreads();
  for (int st = 128; st > 0; st >>= 1) {
    if (static_cast<int>(threadIdx.x) < st)
      for (int q = 0; q < 4; ++q) acc[q][threadIdx.x] += acc[q][threadIdx.x + st];
    __syncthreads();
  }
  if (threadIdx.x < 4 && acc[threadIdx.x][0]) atomicAdd(&out[threadIdx.x], acc[threadIdx.x][0]);
}

// Segment map of the proposal buffer: pre[g] = sum of min(count, seg_cap)
// over the segments before g (one block of kPropSegs threads).
__global__ void k_prop_segs(const unsigned long long* __restrict__ cnt, int64_t seg_cap, int64_t* __restrict__ pre) {
  __shared__ int64_t c[kPropSegs];
  const int g = static_cast<int>(threadIdx.x);
  const int64_t v = static_cast<int64_t>(cnt[g * kCtrStride]);
  c[g] = v < seg_cap ? v : seg_cap;
  __syncthreads();
  if (g == 0) {
    int64_t acc = 0;
    for (int q = 0; q < kPropSegs; ++q) {
      pre[q] = acc;
      acc += c[q];
    }
    pre[kPropSegs] = acc;
  }
}

// --------------------------------------------------------- unique merge --
// UpdateKNNGraphKernel / UniqueMergeSequential (gpuknn/gen_large_knngraph.cu:
// 136-213) with PreProcIDKernel (:215-228): running list = first 32 distinct
// of merge(running, pair result remapped to global ids).  Entries are written
// with plain (non-negative) ids: these lists are the exported result.
__global__ __launch_bounds__(256) void k_unique_merge(hdb_nnd_element* __restrict__ running,
                                                      const hdb_nnd_element* __restrict__ pair, int64_t n_first,
                                                      int64_t rows, int64_t row0_pair, int64_t off_a,
                                                      int64_t off_b) {
  const unsigned lane = __lane_id();
  const int64_t r = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (r >= rows) return;
  uint64_t key;
  if (lane < 32) {
    const hdb_nnd_element e = running[r * kK + lane];
    const uint32_t id = label_id(e.label);
    key = id == kInvalidId ? kKeyMax : make_key(e.distance, id, 1u);
  } else {
    const hdb_nnd_element e = pair[(row0_pair + r) * kK + (lane - 32)];
    uint32_t id = label_id(e.label);
    if (id == kInvalidId) {
      key = kKeyMax;
    } else {
      const int64_t g = (static_cast<int64_t>(id) < n_first) ? off_a + id : off_b + (id - n_first);
      key = make_key(e.distance, static_cast<uint32_t>(g), 1u);
    }
  }
  key = bitonic_group<64>(key);
  const uint64_t prev = shfl_u64(key, (lane + 63) & 63);
  const bool keep = key != kKeyMax && (lane == 0 || (prev >> 1) != (key >> 1));
  const uint64_t bal = __ballot(keep);
  const int pos = __popcll(bal & lanemask_lt());
  const int total = __popcll(bal);
  hdb_nnd_element* out = running + r * kK;
  if (keep && pos < kK) out[pos] = key_to_elem(key);
  if (total < kK && static_cast<int>(lane) >= total && lane < static_cast<unsigned>(kK)) out[lane] = key_to_elem(kKeyMax);
}

__global__ void k_offset_labels(const hdb_nnd_element* __restrict__ in, hdb_nnd_element* __restrict__ out,
                                int64_t total, int64_t off) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < total) {
    hdb_nnd_element e = in[i];
    const uint32_t id = label_id(e.label);
    e.label = id == kInvalidId ? static_cast<int32_t>(kInvalidId) : static_cast<int32_t>(id + off);
    out[i] = e;
  }
}

// Padded copy of the points for the FP32 join (d <= 31): rows of rs floats,
// zeros past d; the last column, the list bound, is left to the init kernel.
__global__ __launch_bounds__(256) void k_nnd_pad_rows(const float* __restrict__ X, int64_t n, int d, int rs,
                                                      float* __restrict__ rows) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t p = t / rs;
  const int c = static_cast<int>(t - p * rs);
  if (p >= n || c == rs - 1) return;
  rows[t] = c < d ? X[p * d + c] : 0.0f;
}

// ------------------------------------------------------------ host side --
static int get_bufs(hdb_ctx* ctx, const float* X, int64_t n, int d, const hdb_params& prm, NndBufs* b) {
  HDB_CALL(scratch_t(ctx, kSlotFwdNew, n * kSMax, &b->fwd_new));
  HDB_CALL(scratch_t(ctx, kSlotFwdOld, n * kSMax, &b->fwd_old));
  HDB_CALL(scratch_t(ctx, kSlotRevNew, n * 32, &b->rev_key));
  HDB_CALL(scratch_t(ctx, kSlotRevOld, n * 32, &b->rev_val));
  int32_t* c2;
  HDB_CALL(scratch_t(ctx, kSlotCounts4, 2 * n, &c2));
  b->fwd_new_n = c2;
  b->fwd_old_n = c2 + n;
  int32_t* rse;
  HDB_CALL(scratch_t(ctx, kSlotRevSE, 4 * n, &rse));
  b->rev_s = rse;
  b->rev_e = rse + 2 * n;
  // bucket_cap proposals per point on average, split into kPropSegs
  // segments; a segment holds at least 4096 (a join block emits at most
  // 4 waves x 64 lanes x 8 proposals = 2048)
  b->seg_cap = std::max<int64_t>(n * static_cast<int64_t>(prm.bucket_cap) / kPropSegs, 4096);
  b->prop_cap = b->seg_cap * kPropSegs;
  HDB_CALL(scratch_t(ctx, kSlotPropTgt, b->prop_cap, &b->prop_tgt));
  HDB_CALL(scratch_t(ctx, kSlotBucket, b->prop_cap, &b->prop_key));
  int64_t* pse;
  const int64_t ngroups = (n + (1 << kGroupBits) - 1) >> kGroupBits;
  HDB_CALL(scratch_t(ctx, kSlotPropSE, 2 * ngroups, &pse));
  b->prop_s = pse;
  b->prop_e = pse + ngroups;
  if (prm.distance_mode == 0 && d <= 31) {
    const int rs = d <= 15 ? 16 : 32;
    float* rows;
    HDB_CALL(scratch_t(ctx, kSlotNndRows, static_cast<size_t>(n) * rs, &rows));
    hipLaunchKernelGGL(k_nnd_pad_rows, dim3(grid_for(n * rs, 256)), dim3(256), 0, ctx->stream, X, n, d, rs, rows);
    HDB_LAUNCHED();
    b->rows = rows;
    b->rstride = rs;
    b->worst = rows + (rs - 1);
    b->wstride = rs;
  } else {
    HDB_CALL(scratch_t(ctx, kSlotWorst, n, &b->worst));
    if (prm.distance_mode >= 1) {
      float* norms;
      HDB_CALL(scratch_t(ctx, kSlotNndRows, n, &norms));
      hipLaunchKernelGGL(k_nnd_norms, dim3(grid_for(n, 256)), dim3(256), 0, ctx->stream, X, n, d, norms);
      HDB_LAUNCHED();
      b->norms = norms;
    }
    b->rows = X;
    b->rstride = d;
    b->wstride = 1;
  }
  unsigned long long* st;  // segment counters, then 4 totals, then the segment map
  HDB_CALL(scratch_t(ctx, kSlotStats, kPropSegs * kCtrStride + 8 + kPropSegs + 1, &st));
  b->prop_cnt = st;
  const int64_t blocks = n;  // one counter set per join wave, i.e. per point
  HDB_CALL(scratch_t(ctx, kSlotPart, 4 * blocks, &b->part));
  HDB_CALL(fill_u64(ctx, reinterpret_cast<uint64_t*>(b->part), 4 * blocks, 0));
  HDB_CALL(fill_u64(ctx, reinterpret_cast<uint64_t*>(st), kPropSegs * kCtrStride + 8, 0));
  b->join_keep = prm.join_keep;
  b->distance_mode = prm.distance_mode;
  b->iter = 0;
  if (prm.distance_mode == 0) b->norms = nullptr;
  b->rerank_deep = prm.rerank_keep == 16 ? 1 : 0;
  return HDB_OK;
}

static int read_stats(hdb_ctx* ctx, int64_t n, const NndBufs& b) {
  const int64_t blocks = n;  // one counter set per join wave, i.e. per point
  unsigned long long* tot = b.prop_cnt + kPropSegs * kCtrStride;
  HDB_CALL(fill_u64(ctx, reinterpret_cast<uint64_t*>(tot), 4, 0));
  hipLaunchKernelGGL(k_sum_parts, dim3(static_cast<unsigned>(std::min<int64_t>(grid_for(blocks, 256), 512))),
                     dim3(256), 0, ctx->stream, b.part, blocks, tot);
  HDB_LAUNCHED();
  unsigned long long s[4];
  HDB_HIP(hipMemcpyAsync(s, tot, sizeof(s), hipMemcpyDeviceToHost, ctx->stream));
  HDB_HIP(hipStreamSynchronize(ctx->stream));
  for (int i = 0; i < 4; ++i) ctx->stats_host[i] = static_cast<int64_t>(s[i]);
  return HDB_OK;
}

template <int D, bool NEWNEW, int KEEP>
static int launch_join_k(hdb_ctx* ctx, const float* X, int64_t n, int d, int S, const NndBufs& b) {
  hipLaunchKernelGGL((k_nnd_join2<D, NEWNEW, KEEP>), dim3(grid_for(n, kJoinWaves)), dim3(kJoinWaves * 64), 0,
                     ctx->stream, X, n, d, S, b);
  HDB_LAUNCHED();
  return HDB_OK;
}

template <int D, bool NEWNEW>
static int launch_join_t(hdb_ctx* ctx, const float* X, int64_t n, int d, int S, const NndBufs& b) {
  switch (b.join_keep) {
    case 0: return launch_join_k<D, NEWNEW, 0>(ctx, X, n, d, S, b);
    case 1: return launch_join_k<D, NEWNEW, 1>(ctx, X, n, d, S, b);
    case 2: return launch_join_k<D, NEWNEW, 2>(ctx, X, n, d, S, b);
    case 3: return launch_join_k<D, NEWNEW, 3>(ctx, X, n, d, S, b);
    case 4: return launch_join_k<D, NEWNEW, 4>(ctx, X, n, d, S, b);
    default: return launch_join_k<D, NEWNEW, 8>(ctx, X, n, d, S, b);
  }
}

template <int DP, bool NEWNEW>
static int launch_join_rows(hdb_ctx* ctx, int64_t n, int d, int S, const NndBufs& b) {
  const dim3 grid(grid_for(n, kJoinWaves)), block(kJoinWaves * 64);
  if (b.join_keep == 0)
    hipLaunchKernelGGL((k_nnd_join_rows<DP, NEWNEW, 0>), grid, block, 0, ctx->stream, n, d, S, 0, b);
  else if (b.join_keep <= 4)
    hipLaunchKernelGGL((k_nnd_join_rows<DP, NEWNEW, 4>), grid, block, 0, ctx->stream, n, d, S, b.join_keep, b);
  else
    hipLaunchKernelGGL((k_nnd_join_rows<DP, NEWNEW, 8>), grid, block, 0, ctx->stream, n, d, S, b.join_keep, b);
  HDB_LAUNCHED();
  return HDB_OK;
}

template <bool NEWNEW>
static int launch_join_wide(hdb_ctx* ctx, const float* X, int64_t n, int d, int S, const NndBufs& b) {
  const dim3 grid(grid_for(n, kJoinWaves)), block(kJoinWaves * 64);
  if (b.join_keep == 0)
    hipLaunchKernelGGL((k_nnd_join_wide<NEWNEW, 0>), grid, block, 0, ctx->stream, X, n, d, S, 0, b);
  else if (b.join_keep <= 4)
    hipLaunchKernelGGL((k_nnd_join_wide<NEWNEW, 4>), grid, block, 0, ctx->stream, X, n, d, S, b.join_keep, b);
  else
    hipLaunchKernelGGL((k_nnd_join_wide<NEWNEW, 8>), grid, block, 0, ctx->stream, X, n, d, S, b.join_keep, b);
  HDB_LAUNCHED();
  return HDB_OK;
}

// rerank_keep 0: the join_keep + 2 nearest partners by the BF16 Gram
// matrix are re-ranked in FP32; 16: the 16 nearest.
template <bool NEWNEW, int KEEP>
static int launch_join_mfma_k(hdb_ctx* ctx, const float* X, int64_t n, int d, int S, const NndBufs& b) {
  const int dp = (d + 31) & ~31;
  constexpr int kShort = KEEP == 0 ? 2 : KEEP + 2;
  constexpr int kDeep = KEEP == 0 ? 2 : 16;
  if (b.rerank_deep)
    hipLaunchKernelGGL((k_nnd_join_mfma<NEWNEW, KEEP, kDeep>), dim3(static_cast<unsigned>(n)), dim3(64), 0,
                       ctx->stream, X, n, d, dp, S, b);
  else
    hipLaunchKernelGGL((k_nnd_join_mfma<NEWNEW, KEEP, kShort>), dim3(static_cast<unsigned>(n)), dim3(64), 0,
                       ctx->stream, X, n, d, dp, S, b);
  HDB_LAUNCHED();
  return HDB_OK;
}

template <bool NEWNEW>
static int launch_join(hdb_ctx* ctx, const float* X, int64_t n, int d, int S, const NndBufs& b) {
  if (b.distance_mode >= 1) {  // 2: the same join, refined after the last iteration
    switch (b.join_keep) {
      case 0: return launch_join_mfma_k<NEWNEW, 0>(ctx, X, n, d, S, b);
      case 1: return launch_join_mfma_k<NEWNEW, 1>(ctx, X, n, d, S, b);
      case 2: return launch_join_mfma_k<NEWNEW, 2>(ctx, X, n, d, S, b);
      case 3: return launch_join_mfma_k<NEWNEW, 3>(ctx, X, n, d, S, b);
      case 4: return launch_join_mfma_k<NEWNEW, 4>(ctx, X, n, d, S, b);
      default: return launch_join_mfma_k<NEWNEW, 8>(ctx, X, n, d, S, b);
    }
  }
  if (d == 12) return launch_join_t<12, NEWNEW>(ctx, X, n, d, S, b);
  if (d == 32) return launch_join_t<32, NEWNEW>(ctx, X, n, d, S, b);
  if (d <= 4) return launch_join_rows<4, NEWNEW>(ctx, n, d, S, b);
  if (d <= 8) return launch_join_rows<8, NEWNEW>(ctx, n, d, S, b);
  if (d <= 12) return launch_join_rows<12, NEWNEW>(ctx, n, d, S, b);
  if (d <= 16) return launch_join_rows<16, NEWNEW>(ctx, n, d, S, b);
  if (d <= 20) return launch_join_rows<20, NEWNEW>(ctx, n, d, S, b);
  if (d <= 24) return launch_join_rows<24, NEWNEW>(ctx, n, d, S, b);
  if (d < 32) return launch_join_rows<32, NEWNEW>(ctx, n, d, S, b);
  return launch_join_wide<NEWNEW>(ctx, X, n, d, S, b);
}

// first_full: the first update merges every list, which also removes
// repeated ids (random and knnmerge starts may hold them); lists that start
// distinct skip that.
static int iterate(hdb_ctx* ctx, const float* X, int64_t n, int d, int S, bool merge, int64_t split, int iterations,
                   hdb_nnd_element* lists, NndBufs& b, bool first_full = true) {
  const int rev_bits = bits_for(2 * n);
  const int tgt_bits = bits_for(n - 1);
  const int64_t ngroups = (n + (1 << kGroupBits) - 1) >> kGroupBits;
  b.s_recip = S > 1 ? static_cast<uint32_t>((static_cast<uint64_t>(1) << 32) / static_cast<uint32_t>(S)) + 1u : 0u;
  b.s_recip16 = (65536u + static_cast<uint32_t>(S) - 1u) / static_cast<uint32_t>(S);
  for (int it = 0; it < iterations; ++it) {
    b.iter = it;
    {
      Stage st(ctx, merge ? "nnd_sample_merge" : "nnd_sample");
      if (merge)
        hipLaunchKernelGGL(k_nnd_sample<true>, dim3(grid_for(n * kK, 256)), dim3(256), 0, ctx->stream, lists, n, S,
                           split, b);
      else
        hipLaunchKernelGGL(k_nnd_sample<false>, dim3(grid_for(n * kK, 256)), dim3(256), 0, ctx->stream, lists, n, S,
                           split, b);
      HDB_LAUNCHED();
    }
    // the sorts leave their results where they end (input or scratch
    // buffers); the kernels that read them get those pointers
    NndBufs bj = b;
    {
      Stage st(ctx, "nnd_reverse_sort");
      uint32_t* rk = nullptr;
      // bit 0 (the kind) is already ordered: new pairs precede old ones
      const int64_t* pairs = nullptr;
      HDB_CALL(radix_sort_u32_u32_drop(ctx, b.rev_key, b.rev_val, n * 32, 1, rev_bits, static_cast<uint32_t>(2 * n),
                                       &rk, &bj.rev_val, &pairs));
      HDB_CALL(segment_bounds(ctx, rk, n * 32, 2 * n, b.rev_s, b.rev_e, 0, pairs));
      HDB_CALL(fill_u64(ctx, reinterpret_cast<uint64_t*>(b.prop_cnt), kPropSegs * kCtrStride, 0));
    }
    {
      Stage st(ctx, merge ? "nnd_join_merge" : "nnd_join");
      if (merge) HDB_CALL(launch_join<false>(ctx, X, n, d, S, bj));
      else HDB_CALL(launch_join<true>(ctx, X, n, d, S, bj));
    }
    int64_t* seg_pre = reinterpret_cast<int64_t*>(b.prop_cnt + kPropSegs * kCtrStride + 8);
    hipLaunchKernelGGL(k_prop_segs, dim3(1), dim3(kPropSegs), 0, ctx->stream, b.prop_cnt, b.seg_cap, seg_pre);
    HDB_LAUNCHED();
    int64_t m = 0;
    HDB_CALL(read_i64(ctx, seg_pre + kPropSegs, &m));
    NndBufs bu = b;
    {
      Stage st(ctx, "nnd_proposal_sort");
      // by list group (target >> kGroupBits); the update buckets each group
      HDB_CALL(radix_sort_u32_u64_segs(ctx, b.prop_tgt, b.prop_key, m, seg_pre, kPropSegs, b.seg_cap, kGroupBits,
                                       std::max(tgt_bits, kGroupBits), &bu.prop_tgt, &bu.prop_key));
      HDB_CALL(segment_bounds(ctx, bu.prop_tgt, m, ngroups, b.prop_s, b.prop_e, kGroupBits));
    }
    {
      Stage st(ctx, merge ? "nnd_update_merge" : "nnd_update");
      // the last iteration writes the lists with the old flags stripped
      // (what k_nnd_finalize does otherwise)
      const int flags = (it == 0 && first_full ? kUpdFull : 0) | (it == iterations - 1 ? kUpdStrip : 0);
      hipLaunchKernelGGL(k_nnd_update, dim3(static_cast<unsigned>(ngroups)), dim3(256), 0, ctx->stream, lists, n, bu,
                         flags);
      HDB_LAUNCHED();
    }
  }
  return HDB_OK;
}

static int check_params(hdb_ctx* ctx, const hdb_params& prm, int64_t n, int d) {
  if (prm.k != kK) return ctx->fail(HDB_EUNSUPPORTED, "k must be 32 (NEIGHB_NUM_PER_LIST)");
  if (prm.sample_num < 1 || prm.sample_num > kSMax) return ctx->fail(HDB_EINVAL, "sample_num must be in [1,16]");
  if (prm.merge_sample_num < 1 || prm.merge_sample_num > kSMax)
    return ctx->fail(HDB_EINVAL, "merge_sample_num must be in [1,16]");
  if (prm.bucket_cap < 8 || prm.bucket_cap > 1024) return ctx->fail(HDB_EINVAL, "bucket_cap must be in [8,1024]");
  if (prm.nnd_iteration < 0 || prm.merge_iteration < 0) return ctx->fail(HDB_EINVAL, "negative iteration count");
  if (prm.join_keep < 0 || (prm.join_keep > 4 && prm.join_keep != 8))
    return ctx->fail(HDB_EINVAL, "join_keep must be in [0,4] or 8");
  if (prm.distance_mode < 0 || prm.distance_mode > 2) return ctx->fail(HDB_EINVAL, "distance_mode must be 0, 1 or 2");
  if (prm.rerank_keep != 0 && prm.rerank_keep != 16) return ctx->fail(HDB_EINVAL, "rerank_keep must be 0 or 16");
  // the joins take any d in chunks of columns; these limits are the tested range
  if (prm.distance_mode == 1 && d > 160) return ctx->fail(HDB_EUNSUPPORTED, "BF16 join built for d <= 160");
  if (prm.distance_mode == 2 && d > 128) return ctx->fail(HDB_EUNSUPPORTED, "BF16 refinement built for d <= 128");
  if (n < 2) return ctx->fail(HDB_EINVAL, "need at least 2 points");
  // reverse-pair positions (n x 32 of them) are int32
  if (n >= kMaxPoints) return ctx->fail(HDB_EINVAL, "n must be below 2^26 (67,108,864)");
  if (d < 1) return ctx->fail(HDB_EINVAL, "d must be >= 1");
  if (d > 255) return ctx->fail(HDB_EUNSUPPORTED, "the FP32 join is built for d <= 255");
  return HDB_OK;
}

int nnd_run(hdb_ctx* ctx, const float* X, int64_t n, int d, const hdb_params& prm, hdb_nnd_element* lists,
            NndInit init, int iterations) {
  HDB_CALL(check_params(ctx, prm, n, d));
  if (!X || !lists) return ctx->fail(HDB_EINVAL, "null pointer");
  if (n <= kK + 1 && iterations > 0) {
    // every other point fits in each list: the exact graph, sorted
    Stage st(ctx, "nnd_exact_small");
    hipLaunchKernelGGL(k_nnd_exact_small, dim3(grid_for(n * kK, 256)), dim3(256), 0, ctx->stream, X, n, d, lists);
    HDB_LAUNCHED();
    ctx->stats_host[0] = ctx->stats_host[1] = ctx->stats_host[2] = ctx->stats_host[3] = 0;
    return HDB_OK;
  }
  NndBufs b;
  HDB_CALL(get_bufs(ctx, X, n, d, prm, &b));
  {
    Stage st(ctx, "nnd_init");
    if (init == NndInit::kRandom)
      hipLaunchKernelGGL(k_nnd_init_random, dim3(grid_for(n * kK, 256)), dim3(256), 0, ctx->stream, b.rows, b.rstride,
                         n, d, lists,
                         b.worst, b.wstride);
    else if (init == NndInit::kGiven)
      hipLaunchKernelGGL(k_nnd_init_given, dim3(grid_for(n * kK, 256)), dim3(256), 0, ctx->stream, X, n, d, lists,
                         b.worst, b.wstride);
    else
      hipLaunchKernelGGL(k_nnd_init_exact, dim3(grid_for(n * kK, 256)), dim3(256), 0, ctx->stream, lists, n, b.worst,
                         b.wstride);
    HDB_LAUNCHED();
  }
  HDB_CALL(iterate(ctx, X, n, d, prm.sample_num, false, 0, iterations, lists, b, init == NndInit::kRandom));
  if (iterations == 0) {  // otherwise the last update wrote the lists without old flags
    Stage st(ctx, "nnd_finalize");
    hipLaunchKernelGGL(k_nnd_finalize, dim3(grid_for(n * kK, 256)), dim3(256), 0, ctx->stream, lists, n * kK);
    HDB_LAUNCHED();
  }
  return read_stats(ctx, n, b);
}

int nnd_merge_pair(hdb_ctx* ctx, const float* X, int64_t n1, int64_t n2, int d, const hdb_nnd_element* g1,
                   const hdb_nnd_element* g2, const hdb_params& prm, hdb_nnd_element* out) {
  const int64_t n = n1 + n2;
  HDB_CALL(check_params(ctx, prm, n, d));
  if (n1 < 1 || n2 < 1) return ctx->fail(HDB_EINVAL, "both graphs must be non-empty");
  if (!X || !g1 || !g2 || !out) return ctx->fail(HDB_EINVAL, "null pointer");
  NndBufs b;
  HDB_CALL(get_bufs(ctx, X, n, d, prm, &b));
  {
    Stage st(ctx, "nnd_init_merge");
    hipLaunchKernelGGL(k_nnd_init_merge, dim3(grid_for(n * kK, 256)), dim3(256), 0, ctx->stream, X, n1, n2, d, g1, g2,
                       out, b.worst, b.wstride);
    HDB_LAUNCHED();
  }
  HDB_CALL(iterate(ctx, X, n, d, prm.merge_sample_num, true, n1, prm.merge_iteration, out, b));
  if (prm.merge_iteration == 0) {  // otherwise the last update wrote the lists without old flags
    Stage st(ctx, "nnd_finalize");
    hipLaunchKernelGGL(k_nnd_finalize, dim3(grid_for(n * kK, 256)), dim3(256), 0, ctx->stream, out, n * kK);
    HDB_LAUNCHED();
  }
  return read_stats(ctx, n, b);
}

std::vector<int64_t> shard_offsets(int64_t n, int shards) {
  std::vector<int64_t> off(shards + 1);
  const int64_t per = n / shards;
  for (int i = 0; i < shards; ++i) off[i] = per * i;
  off[shards] = n;
  return off;
}

int unique_merge(hdb_ctx* ctx, hdb_nnd_element* running, const hdb_nnd_element* pair, int64_t n_first, int64_t rows,
                 int64_t row0_pair, int64_t off_a, int64_t off_b) {
  if (rows <= 0) return HDB_OK;
  Stage st(ctx, "nnd_unique_merge");
  hipLaunchKernelGGL(k_unique_merge, dim3(grid_for(rows, 4)), dim3(256), 0, ctx->stream, running, pair, n_first, rows,
                     row0_pair, off_a, off_b);
  HDB_LAUNCHED();
  return HDB_OK;
}

int nnd_blocked(hdb_ctx* ctx, const float* X, int64_t n, int d, int blocks, const hdb_params& prm,
                hdb_nnd_element* out) {
  HDB_CALL(check_params(ctx, prm, n, d));
  if (blocks < 1 || static_cast<int64_t>(blocks) * 2 > n) return ctx->fail(HDB_EINVAL, "bad block count");
  const std::vector<int64_t> off = shard_offsets(n, blocks);
  for (int i = 0; i < blocks; ++i)
    if (off[i + 1] - off[i] < 2) return ctx->fail(HDB_EINVAL, "block smaller than 2 points");
  hdb_nnd_element* local;
  HDB_CALL(scratch_t(ctx, kSlotBlockLocal, n * kK, &local));
  int64_t stats[4] = {0, 0, 0, 0};
  // BuildEachShard (gen_large_knngraph.cu:47-92): NN-Descent per block with
  // local ids; the running lists start as the block graphs in global ids.
  for (int i = 0; i < blocks; ++i) {
    const int64_t ni = off[i + 1] - off[i];
    HDB_CALL(nnd_run(ctx, X + off[i] * d, ni, d, prm, local + off[i] * kK, NndInit::kRandom, prm.nnd_iteration));
    for (int s = 0; s < 4; ++s) stats[s] += ctx->stats_host[s];
    hipLaunchKernelGGL(k_offset_labels, dim3(grid_for(ni * kK, 256)), dim3(256), 0, ctx->stream, local + off[i] * kK,
                       out + off[i] * kK, ni * kK, off[i]);
    HDB_LAUNCHED();
  }
  if (blocks == 1) return HDB_OK;
  int64_t max_pair = 0;
  for (int i = 0; i < blocks; ++i)
    for (int j = i + 1; j < blocks; ++j) max_pair = std::max(max_pair, off[i + 1] - off[i] + off[j + 1] - off[j]);
  hdb_nnd_element* pair;
  float* xp;
  HDB_CALL(scratch_t(ctx, kSlotPairGraph, max_pair * kK, &pair));
  HDB_CALL(scratch_t(ctx, kSlotPairX, max_pair * d, &xp));
  // MultiMerge (gen_large_knngraph.cu:249-407): every pair i < j.
  for (int i = 0; i < blocks; ++i) {
    for (int j = i + 1; j < blocks; ++j) {
      const int64_t ni = off[i + 1] - off[i], nj = off[j + 1] - off[j];
      const float* xpair = X + off[i] * d;
      if (j != i + 1) {
        HDB_HIP(hipMemcpyAsync(xp, X + off[i] * d, ni * d * sizeof(float), hipMemcpyDeviceToDevice, ctx->stream));
        HDB_HIP(hipMemcpyAsync(xp + ni * d, X + off[j] * d, nj * d * sizeof(float), hipMemcpyDeviceToDevice,
                               ctx->stream));
        xpair = xp;
      }
      HDB_CALL(nnd_merge_pair(ctx, xpair, ni, nj, d, local + off[i] * kK, local + off[j] * kK, prm, pair));
      for (int s = 0; s < 4; ++s) stats[s] += ctx->stats_host[s];
      HDB_CALL(unique_merge(ctx, out + off[i] * kK, pair, ni, ni, 0, off[i], off[j]));
      HDB_CALL(unique_merge(ctx, out + off[j] * kK, pair, ni, nj, ni, off[i], off[j]));
    }
  }
  for (int s = 0; s < 4; ++s) ctx->stats_host[s] = stats[s];
  return HDB_OK;
}

// ------------------------------------------------------ brute-force kNN --
// One wave per query and point chunk (blockIdx.y); each lane scans a strided
// share of the chunk keeping a sorted top-kq (kq <= 32) in registers, then
// the wave pops the chunk's top-kq from the 64 lane lists.  With one chunk
// (part == nullptr) that is the result; otherwise it goes to
// part[(qi * chunks + y) * 32 + s] (kKeyMax past the last), which k_bf_merge
// merges.  Bound by the row reads (a lane per row, 16 bytes at a time where
// rows are 16-byte aligned): the chunks let a few queries fill the chip.  16
// queries against 100k x 128 took 25.4 ms with one wave each, 0.4 ms split.
__global__ __launch_bounds__(256) void k_bruteforce(const float* __restrict__ X, int64_t n, int d,
                                                    const int32_t* __restrict__ qids, int64_t m, int kq,
                                                    int64_t csize, uint64_t* __restrict__ part,
                                                    int32_t* __restrict__ out_ids, float* __restrict__ out_d2) {
  const unsigned lane = __lane_id();
  const int64_t qi = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (qi >= m) return;
  const uint32_t q = static_cast<uint32_t>(qids[qi]);
  const bool known = static_cast<int64_t>(q) < n;  // an id outside [0, n): no neighbours
  uint64_t top[32];
#pragma unroll
  for (int i = 0; i < 32; ++i) top[i] = kKeyMax;
  const int64_t c0 = static_cast<int64_t>(blockIdx.y) * csize;
  const int64_t c1 = !known ? c0 : c0 + csize < n ? c0 + csize : n;
  for (int64_t i = c0 + lane; i < c1; i += 64) {
    if (static_cast<uint32_t>(i) == q) continue;
    uint64_t key = (static_cast<uint64_t>(__float_as_uint(point_d2(X, d, q, static_cast<uint32_t>(i)))) << 32) |
                   static_cast<uint32_t>(i);
    if (key < top[31]) {
#pragma unroll
      for (int s = 0; s < 32; ++s) {
        const uint64_t a = top[s];
        const bool sw = key < a;
        top[s] = sw ? key : a;
        key = sw ? a : key;
      }
    }
  }
  // pop kq minima across lanes
  int head = 0;
  uint64_t mine = kKeyMax;  // lane r ends with the r-th smallest
  for (int r = 0; r < kq; ++r) {
    uint64_t h = kKeyMax;
#pragma unroll
    for (int s = 0; s < 32; ++s)
      if (s == head) h = top[s];
    uint64_t mn = h;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const uint64_t oth = shfl_xor_u64(mn, o);
      mn = oth < mn ? oth : mn;
    }
    if (h == mn && mn != kKeyMax) head++;
    if (static_cast<int>(lane) == r) mine = mn;
  }
  if (part) {
    if (lane < 32) part[(qi * gridDim.y + blockIdx.y) * 32 + lane] = mine;
  } else if (static_cast<int>(lane) < kq) {
    out_ids[qi * kq + lane] = mine == kKeyMax ? -1 : static_cast<int32_t>(static_cast<uint32_t>(mine));
    if (out_d2)
      out_d2[qi * kq + lane] = __uint_as_float(known ? static_cast<uint32_t>(mine >> 32) : 0x7F800000u);
  }
}

// Tiled brute force for D = 12 or 32: block (g, y) holds queries
// [64g, 64g + 64) -- lane l of every wave holds query 64g + l -- and scans
// point chunk y, staged through LDS kBfTile points at a time; wave w takes
// points w, w + 4, ... of each tile, so every LDS read is a broadcast and
// each point is read from HBM once per 64 queries.  Each lane keeps its
// sorted top-32 keys (d2 bits << 32 | id), written to
// part[((qi * chunks + y) * 4 + w) * 32 + s]; k_bf_merge takes the kq
// smallest of a query's chunks * 4 lists.
template <int D>
struct BfTile {
  static constexpr int kPts = D <= 16 ? 512 : 256;  // 24 KB (d = 12) or 32 KB (d = 32) of LDS
};

template <int D>
__global__ __launch_bounds__(256) void k_bf_tile(const float* __restrict__ X, int64_t n,
                                                 const int32_t* __restrict__ qids, int64_t m, int64_t csize,
                                                 int chunks, uint64_t* __restrict__ part) {
  constexpr int kBfTile = BfTile<D>::kPts;
  __shared__ float s_pts[kBfTile * D];
  const unsigned lane = __lane_id();
  const unsigned w = threadIdx.x >> 6;
  const int64_t qi = static_cast<int64_t>(blockIdx.x) * 64 + lane;
  const int64_t c0 = static_cast<int64_t>(blockIdx.y) * csize;
  const int64_t c1 = c0 + csize < n ? c0 + csize : n;
  const bool live = qi < m;
  int64_t q = -1;
  float xq[D];
  if (live) {
    q = qids[qi];
    if (q < 0 || q >= n) q = -1;
  }
#pragma unroll
  for (int k = 0; k < D; ++k) xq[k] = q >= 0 ? X[q * D + k] : 0.0f;
  uint64_t top[32];
#pragma unroll
  for (int s = 0; s < 32; ++s) top[s] = kKeyMax;
  for (int64_t t0 = c0; t0 < c1; t0 += kBfTile) {
    const int cnt = static_cast<int>(c1 - t0 < kBfTile ? c1 - t0 : kBfTile);
    __syncthreads();
    const float* src = X + t0 * D;
    for (int i = threadIdx.x; i < cnt * D; i += 256) s_pts[i] = src[i];
    __syncthreads();
    for (int j = static_cast<int>(w); j < cnt; j += 4) {
      const float* row = s_pts + j * D;
      float acc = 0.0f;
#pragma unroll
      for (int k = 0; k < D; ++k) {
        const float diff = xq[k] - row[k];
        acc = __builtin_fmaf(diff, diff, acc);
      }
      const int64_t id = t0 + j;
      uint64_t key = (static_cast<uint64_t>(__float_as_uint(acc)) << 32) | static_cast<uint32_t>(id);
      if (id == q) key = kKeyMax;
      if (key < top[31]) {
#pragma unroll
        for (int s = 0; s < 32; ++s) {
          const uint64_t a = top[s];
          const bool sw = key < a;
          top[s] = sw ? key : a;
          key = sw ? a : key;
        }
      }
    }
  }
  if (!live) return;
  if (q < 0) {  // an id outside [0, n): the merge reports no neighbours
#pragma unroll
    for (int s = 0; s < 32; ++s) top[s] = kKeyMax;
  }
  uint64_t* out = part + ((qi * chunks + blockIdx.y) * 4 + w) * 32;
#pragma unroll
  for (int s = 0; s < 32; ++s) out[s] = top[s];
}

// One wave per query: lane l merges lists l, l + 64, ... of the query's
// `lists` sorted 32-key lists into its own top-32, then the wave pops the
// kq smallest keys.  qids (optional): an id outside [0, n) gets infinite
// distances.
__global__ __launch_bounds__(256) void k_bf_merge(const uint64_t* __restrict__ part, int64_t m, int lists, int kq,
                                                  const int32_t* __restrict__ qids, int64_t n,
                                                  int32_t* __restrict__ out_ids, float* __restrict__ out_d2) {
  const unsigned lane = __lane_id();
  const int64_t qi = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (qi >= m) return;
  uint64_t top[32];
#pragma unroll
  for (int s = 0; s < 32; ++s) top[s] = kKeyMax;
  const uint64_t* base = part + qi * static_cast<int64_t>(lists) * 32;
  for (int li = static_cast<int>(lane); li < lists; li += 64) {
    for (int e = 0; e < 32; ++e) {
      uint64_t key = base[li * 32 + e];
      if (!(key < top[31])) break;  // the list is sorted: nothing after it can enter
#pragma unroll
      for (int s = 0; s < 32; ++s) {
        const uint64_t a = top[s];
        const bool sw = key < a;
        top[s] = sw ? key : a;
        key = sw ? a : key;
      }
    }
  }
  int head = 0;
  for (int r = 0; r < kq; ++r) {
    uint64_t h = kKeyMax;
#pragma unroll
    for (int s = 0; s < 32; ++s)
      if (s == head) h = top[s];
    uint64_t mn = h;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const uint64_t oth = shfl_xor_u64(mn, o);
      mn = oth < mn ? oth : mn;
    }
    if (h == mn && mn != kKeyMax) head++;
    if (lane == 0) {
      out_ids[qi * kq + r] = mn == kKeyMax ? -1 : static_cast<int32_t>(static_cast<uint32_t>(mn));
      const bool bad = qids && static_cast<int64_t>(static_cast<uint32_t>(qids[qi])) >= n;
      if (out_d2) out_d2[qi * kq + r] = __uint_as_float(bad ? 0x7F800000u : static_cast<uint32_t>(mn >> 32));
    }
  }
}

// Evaluate (tools/evaluate.hpp:13-52) for sampled queries: hits +=
// |first kq ids of lists[q] intersect gt[qi][0..kq)| (set semantics: lists
// and ground truth hold distinct ids), one wave per query.
__global__ __launch_bounds__(256) void k_recall_hits(const hdb_nnd_element* __restrict__ lists, int64_t n,
                                                     const int32_t* __restrict__ qids, int64_t m,
                                                     const int32_t* __restrict__ gt, int kq,
                                                     unsigned long long* __restrict__ hits) {
  const unsigned lane = __lane_id();
  const int64_t qi = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (qi >= m) return;
  const int64_t q = qids[qi];
  uint32_t mine = 0xFFFFFFFFu;  // lanes < kq: list entry; lanes 32 + j < 32 + kq: ground-truth entry
  if (q >= 0 && q < n) {
    if (static_cast<int>(lane) < kq) mine = label_id(lists[q * kK + lane].label);
    else if (lane >= 32 && static_cast<int>(lane) - 32 < kq) {
      const int32_t g = gt[qi * kq + (lane - 32)];
      mine = g >= 0 ? static_cast<uint32_t>(g) : 0xFFFFFFFEu;
    }
  }
  bool hit = false;
  for (int j = 0; j < kq; ++j) {
    const uint32_t g = __shfl(mine, 32 + j);
    hit = hit || (static_cast<int>(lane) < kq && mine != kInvalidId && mine == g);
  }
  const int cnt = __popcll(__ballot(hit));
  if (lane == 0 && cnt) atomicAdd(hits, static_cast<unsigned long long>(cnt));
}

int recall_hits(hdb_ctx* ctx, const hdb_nnd_element* lists, int64_t n, const int32_t* qids, int64_t m,
                const int32_t* gt, int kq, int64_t* hits_out) {
  if (kq < 1 || kq > 32) return ctx->fail(HDB_EINVAL, "kq must be in [1,32]");
  if (!lists || !hits_out || (m > 0 && (!qids || !gt)) || n < 1) return ctx->fail(HDB_EINVAL, "bad recall arguments");
  *hits_out = 0;
  if (m <= 0) return HDB_OK;
  unsigned long long* h;
  HDB_CALL(scratch_t(ctx, kSlotMisc2, 1, &h));
  HDB_CALL(fill_u64(ctx, reinterpret_cast<uint64_t*>(h), 1, 0));
  hipLaunchKernelGGL(k_recall_hits, dim3(grid_for(m, 4)), dim3(256), 0, ctx->stream, lists, n, qids, m, gt, kq, h);
  HDB_LAUNCHED();
  return read_i64(ctx, reinterpret_cast<const int64_t*>(h), hits_out);
}

template <int D>
static int bruteforce_tiled(hdb_ctx* ctx, const float* X, int64_t n, const int32_t* qids, int64_t m, int kq,
                            int32_t* out_ids, float* out_d2) {
  const int64_t groups = (m + 63) / 64;
  // enough blocks to fill the chip, chunks of at least one tile
  int64_t chunks = (2048 + groups - 1) / groups;
  chunks = std::max<int64_t>(1, std::min<int64_t>(chunks, (n + BfTile<D>::kPts - 1) / BfTile<D>::kPts));
  chunks = std::min<int64_t>(chunks, 1024);
  const int64_t csize = (n + chunks - 1) / chunks;
  chunks = (n + csize - 1) / csize;
  uint64_t* part;
  HDB_CALL(scratch_t(ctx, kSlotBfTmp, m * chunks * 4 * 32, &part));
  hipLaunchKernelGGL(k_bf_tile<D>, dim3(static_cast<unsigned>(groups), static_cast<unsigned>(chunks)), dim3(256), 0,
                     ctx->stream, X, n, qids, m, csize, static_cast<int>(chunks), part);
  HDB_LAUNCHED();
  hipLaunchKernelGGL(k_bf_merge, dim3(grid_for(m, 4)), dim3(256), 0, ctx->stream, part, m,
                     static_cast<int>(chunks * 4), kq, nullptr, n, out_ids, out_d2);
  HDB_LAUNCHED();
  return HDB_OK;
}

int bruteforce_knn(hdb_ctx* ctx, const float* X, int64_t n, int d, const int32_t* qids, int64_t m, int kq,
                   int32_t* out_ids, float* out_d2) {
  if (kq < 1 || kq > 32) return ctx->fail(HDB_EINVAL, "kq must be in [1,32]");
  if (!X || !qids || !out_ids || n < 1 || d < 1) return ctx->fail(HDB_EINVAL, "bad brute-force arguments");
  if (n >= (static_cast<int64_t>(1) << 31)) return ctx->fail(HDB_EINVAL, "n must be below 2^31");
  if (m <= 0) return HDB_OK;
  Stage st(ctx, "bruteforce_knn");
  if (d == 12) return bruteforce_tiled<12>(ctx, X, n, qids, m, kq, out_ids, out_d2);
  if (d == 32) return bruteforce_tiled<32>(ctx, X, n, qids, m, kq, out_ids, out_d2);
  // About 8192 waves, chunks of at least 512 points; one chunk, which needs no
  // scratch and no merge, where a wave's whole scan (in loads, and six loads'
  // time for the rest of a point) costs less than popping and merging the
  // chunks' lists.  One chunk / split: 100 queries of 3000 x 7 134 / 151 us, of
  // 3000 x 33 219 / 162; 1000 of 3000 x 33 225 / 255, of 10k x 7 356 / 273; 4096
  // of 10k x 20 468 / 657, of 10k x 128 3388 / 3067.
  const bool vec4 = (d & 3) == 0 && (reinterpret_cast<uintptr_t>(X) & 15) == 0;
  const bool split = n * (6 + (vec4 ? d / 4 : d)) >= 60000 + 60 * m;
  int64_t chunks = split ? std::max<int64_t>(1, std::min<int64_t>(8192 / m, (n + 511) / 512)) : 1;
  const int64_t csize = (n + chunks - 1) / chunks;
  chunks = (n + csize - 1) / csize;
  uint64_t* part = nullptr;
  if (chunks > 1) HDB_CALL(scratch_t(ctx, kSlotBfTmp, m * chunks * 32, &part));
  hipLaunchKernelGGL(k_bruteforce, dim3(grid_for(m, 4), static_cast<unsigned>(chunks)), dim3(256), 0, ctx->stream, X, n,
                     d, qids, m, kq, csize, part, out_ids, out_d2);
  HDB_LAUNCHED();
  if (!part) return HDB_OK;
  hipLaunchKernelGGL(k_bf_merge, dim3(grid_for(m, 4)), dim3(256), 0, ctx->stream, part, m, static_cast<int>(chunks), kq,
                     qids, n, out_ids, out_d2);
  HDB_LAUNCHED();
  return HDB_OK;
}

}  // namespace hdb
