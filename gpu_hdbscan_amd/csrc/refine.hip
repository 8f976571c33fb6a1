// Exact refinement of a kNN graph with BF16 MFMA distance tiles (the
// distance_mode 2 variant: candidate distances by BF16 matrix products with
// FP32 accumulation, survivors re-ranked in exact FP32).
//
// Input: lists whose entry 31 of point q holds a true squared distance
// tau_q (any 32 distinct points give such a list, NN-Descent's included):
// then q's true 32 nearest neighbours all lie within tau_q.  The pass
//   1. splits every coordinate x = xh + xl into two BF16 values
//      (xh = bf16(x), xl = bf16(x - xh)) and computes |x|^2 in FP32;
//   2. streams every point past every query in 64 x 64 tiles: the product
//      x.y ~ xh.yh + xh.yl + xl.yh comes from three v_mfma_f32_16x16x32_bf16
//      chains accumulated in FP32, and y survives when
//      |y|^2 - 2 x.y < tau_q + delta_q - |x|^2.  delta_q bounds the error of
//      that test for every y with |x - y|^2 <= tau_q (below), so every true
//      neighbour survives; typically 40-100 points do;
//   3. re-ranks each query's survivors with the exact FP32 distance of the
//      kNN path (d2_vec4 / d2_any) and keeps the first 32 by (d2, id).
// The result is the exact 32-NN under FP32 distances with ties broken by id:
// the same lists the brute-force kernels give.  A point with more than
// kRfCap survivors (a loose tau) stops collecting at the cap; its list
// becomes the 32 nearest of its kept survivors and old entries, a tighter
// tau, and it goes through the pass again (a round over those points only);
// what is still past the cap after kRfRounds rounds gets the exact FP32
// brute force.
//
// Error bound.  With u = 2^-8 (BF16 unit roundoff), |x - xh - xl| <= u^2 |x|
// per coordinate, and the three products omit xl.yl and the split residues:
// |x.y - (xh.yh + xh.yl + xl.yh)| <= 3.001 u^2 sum|x_i y_i| <= 4.6e-5 |x||y|.
// FP32 accumulation of the 3d exact products (d <= 128) adds at most
// 384 * 2^-24 * sum|terms| <= 2.3e-5 |x||y|; |y|^2 and |x|^2 carry at most
// 128 * 2^-24 relative error.  So the test's left side exceeds the exact
// |y|^2 - 2 x.y by at most 1.4e-4 |x||y| + 7.7e-6 |y|^2, and with
// |y| <= |x| + sqrt(tau_q) = yb for every candidate within tau_q,
//   delta_q = 1.5e-4 |x| yb + 1e-5 (yb^2 + |x|^2) + 2e-5 tau_q
// covers it, the roundings of the threshold itself and the FP32 rounding
// of tau_q (a distance of d <= 128 terms: relative error below 7.7e-6).
// Entry 31 bounds the 32nd distance when the list holds 32 distinct points
// sorted by distance, as every list of the kNN path does.
//
// For d <= 32 the tiles are FP32 products on the matrix cores instead
// (k_rf_scan32, its own bound below): there the split-BF16 bound, relative
// to |x| |y|, is loose against the small neighbour distances.
//
// The same pass answers a set of query points only (exact_knn_bounded):
// their lists are copied to rows of their own, the stream is split into
// chunks over blockIdx.y so that a few hundred queries still fill the chip,
// and the rows are written out as ids and distances.
//
// Layout in HBM: xh, xl as np x dp BF16 rows (dp = d rounded up to 32,
// np = n rounded up to 256, zero padding), pn = |x|^2 (+inf on padding
// rows, so they never survive); per query row: cnt, kRfCap survivor ids.
#include "hdb_internal.hpp"

namespace hdb {

namespace {

typedef __bf16 rf_bf16x8 __attribute__((ext_vector_type(8)));
typedef float rf_f32x4 __attribute__((ext_vector_type(4)));

constexpr int kRfCap = 128;    // survivors kept per query (two per lane in the re-rank)
constexpr int kRfQS = 2;       // 16-query sub-tiles per wave (the survivor masks' layout)
constexpr int kRfWaves = 8;    // waves per block: 8 x 32 = 256 queries share each tile
constexpr int kRfThreads = kRfWaves * 64;
constexpr int kRfBlockQ = kRfWaves * kRfQS * 16;
constexpr int kRfTile = 64;    // points per streamed tile
constexpr int kRfPad = 8;      // BF16 elements of padding per LDS row

// A sorted key (d2 bits, id, flag 0) as a list entry; kKeyMax is the
// invalid entry (infinite distance, id -1).
__device__ __forceinline__ hdb_nnd_element key_to_list_elem(uint64_t k) {
  hdb_nnd_element e;
  if (k == kKeyMax) {
    e.distance = __uint_as_float(0x7F800000u);
    e.label = static_cast<int32_t>(kInvalidId);
  } else {
    e.distance = key_d2(k);
    e.label = static_cast<int32_t>(key_id(k));
  }
  return e;
}

__global__ void k_rf_split(const float* __restrict__ X, int64_t n, int d, int dp, int64_t np,
                           __bf16* __restrict__ xh, __bf16* __restrict__ xl) {
  const int64_t e = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (e >= np * dp) return;
  const int64_t i = e / dp;
  const int k = static_cast<int>(e - i * dp);
  const float v = (i < n && k < d) ? X[i * d + k] : 0.0f;
  const __bf16 h = static_cast<__bf16>(v);
  xh[e] = h;
  xl[e] = static_cast<__bf16>(v - static_cast<float>(h));
}

__global__ void k_rf_norms(const float* __restrict__ X, int64_t n, int d, int64_t np, float* __restrict__ pn) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= np) return;
  if (i >= n) {
    pn[i] = __uint_as_float(0x7F800000u);
    return;
  }
  const float* r = X + i * d;
  float s = 0.0f;
  for (int k = 0; k < d; ++k) s = __builtin_fmaf(r[k], r[k], s);
  pn[i] = s;
}

// A wave's queue of survivors in LDS.  A survivor costs an atomic on its
// row's count, whose result the wave has to wait for; at 100k points every
// tile holds one or two, and a wait for each left the matrix cores idle most
// of the time.  Survivors are queued instead and 64 at a time take their
// atomics together, one wait for all.  An entry is (row | tag << 24, id):
// rows are below 2^24; the tag is the query's place in the wave (0..31), or
// kRfNoTag for a reverse survivor.
constexpr int kRfQueue = 128;
constexpr uint32_t kRfNoTag = 0xFFu;

struct RfQueue {
  uint32_t* row;   // this wave's kRfQueue entries
  int32_t* id;
  uint32_t* stop;  // this wave's queries past the cap, a bit each
  int len;         // wave-uniform, below 64 between pushes
};

__device__ __forceinline__ void rf_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Sends the first `k` (at most 64) entries to their rows' candidates and
// moves the rest to the front.  A row past the cap takes no more; its
// query's bit is set in `stop`.
__device__ __forceinline__ void rf_flush(RfQueue& qu, int k, int32_t* __restrict__ cnt, int32_t* __restrict__ cand) {
  const int lane = static_cast<int>(__lane_id());
  rf_wave_sync();
  if (lane < k) {
    const uint32_t e = qu.row[lane];
    const int64_t r = e & 0xFFFFFFu;
    const int slot = atomicAdd(cnt + r, 1);
    if (slot < kRfCap) cand[r * kRfCap + slot] = qu.id[lane];
    else if ((e >> 24) != kRfNoTag) atomicOr(qu.stop, 1u << (e >> 24));
  }
  const int rest = qu.len - k;
  uint32_t r = 0;
  int32_t i = 0;
  if (lane < rest) {
    r = qu.row[k + lane];
    i = qu.id[k + lane];
  }
  rf_wave_sync();
  if (lane < rest) {
    qu.row[lane] = r;
    qu.id[lane] = i;
  }
  qu.len = rest;
}

// Queues every set bit of each lane's mask; entry(bit, &row, &id) names it.
template <typename F>
__device__ __forceinline__ void rf_push(RfQueue& qu, uint32_t mask, F entry, int32_t* __restrict__ cnt,
                                        int32_t* __restrict__ cand) {
  while (true) {
    const uint64_t bal = __ballot(mask != 0);
    if (!bal) return;  // uniform
    if (mask) {
      uint32_t row;
      int32_t id;
      entry(__builtin_ctz(mask), &row, &id);
      const int at = qu.len + __popcll(bal & lanemask_lt());
      qu.row[at] = row;
      qu.id[at] = id;
      mask &= mask - 1;
    }
    qu.len += __popcll(bal);
    if (qu.len >= 64) rf_flush(qu, 64, cnt, cand);
  }
}

// Survivors of one 64-point tile t for the wave's 32 query rows: lane l
// holds |y|^2 - 2 x.y for points 16 r + 4 (l / 16) + q of the tile and query
// sub-tile s; bit 8 r + 4 s + q of a lane's mask is that pair.
__device__ __forceinline__ void rf_survivors(const rf_f32x4 (&acc)[4][kRfQS], const float* s_pn,
                                             const float (&thr)[kRfQS], const int64_t (&qrow)[kRfQS],
                                             const int64_t (&qpt)[kRfQS], int64_t t, int grp, int col, RfQueue& qu,
                                             int32_t* __restrict__ cnt, int32_t* __restrict__ cand) {
  float4 p4[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) p4[r] = *reinterpret_cast<const float4*>(&s_pn[r * 16 + grp * 4]);
  bool any = false;
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int s = 0; s < kRfQS; ++s) {
      any |= __builtin_fmaf(-2.0f, acc[r][s][0], p4[r].x) < thr[s];
      any |= __builtin_fmaf(-2.0f, acc[r][s][1], p4[r].y) < thr[s];
      any |= __builtin_fmaf(-2.0f, acc[r][s][2], p4[r].z) < thr[s];
      any |= __builtin_fmaf(-2.0f, acc[r][s][3], p4[r].w) < thr[s];
    }
  if (!__ballot(any)) return;  // wave-uniform
  uint32_t mask = 0;
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int s = 0; s < kRfQS; ++s)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float pq = q == 0 ? p4[r].x : q == 1 ? p4[r].y : q == 2 ? p4[r].z : p4[r].w;
        mask |= __builtin_fmaf(-2.0f, acc[r][s][q], pq) < thr[s] ? 1u << (8 * r + 4 * s + q) : 0u;
      }
  // the query itself is no neighbour: its bit is cleared
  const int64_t first = t * kRfTile + grp * 4;
#pragma unroll
  for (int s = 0; s < kRfQS; ++s) {
    const int64_t o = qpt[s] - first;  // 16 r + q for the lane that holds it
    if (o >= 0 && o < kRfTile && (o & 15) < 4) mask &= ~(1u << (8 * (o >> 4) + 4 * s + (o & 15)));
  }
  rf_push(
      qu, mask,
      [&](int bit, uint32_t* row, int32_t* id) {
        const int s = (bit >> 2) & 1;
        *row = static_cast<uint32_t>(s ? qrow[1] : qrow[0]) | (static_cast<uint32_t>(16 * s + col) << 24);
        *id = static_cast<int32_t>(first + 16 * (bit >> 3) + (bit & 3));
      },
      cnt, cand);
}

// The other direction of a tile (SYM): point y = 16 r + 4 (l / 16) + q of
// tile t gets query x when |x|^2 - 2 x.y is below y's own threshold.  Rows
// are points here (the first round over every point).
__device__ __forceinline__ void rf_reverse(const rf_f32x4 (&acc)[4][kRfQS], const float* s_thr,
                                           const float (&qn)[kRfQS], const int64_t (&qpt)[kRfQS], int64_t t,
                                           int grp, RfQueue& qu, int32_t* __restrict__ cnt,
                                           int32_t* __restrict__ cand) {
  float4 t4[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) t4[r] = *reinterpret_cast<const float4*>(&s_thr[r * 16 + grp * 4]);
  bool any = false;
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int s = 0; s < kRfQS; ++s) {
      any |= __builtin_fmaf(-2.0f, acc[r][s][0], qn[s]) < t4[r].x;
      any |= __builtin_fmaf(-2.0f, acc[r][s][1], qn[s]) < t4[r].y;
      any |= __builtin_fmaf(-2.0f, acc[r][s][2], qn[s]) < t4[r].z;
      any |= __builtin_fmaf(-2.0f, acc[r][s][3], qn[s]) < t4[r].w;
    }
  if (!__ballot(any)) return;
  uint32_t mask = 0;
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int s = 0; s < kRfQS; ++s)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float tq = q == 0 ? t4[r].x : q == 1 ? t4[r].y : q == 2 ? t4[r].z : t4[r].w;
        mask |= __builtin_fmaf(-2.0f, acc[r][s][q], qn[s]) < tq ? 1u << (8 * r + 4 * s + q) : 0u;
      }
  const int64_t first = t * kRfTile + grp * 4;
  rf_push(
      qu, mask,
      [&](int bit, uint32_t* row, int32_t* id) {
        *row = static_cast<uint32_t>(first + 16 * (bit >> 3) + (bit & 3)) | (kRfNoTag << 24);
        *id = static_cast<int32_t>(((bit >> 2) & 1) ? qpt[1] : qpt[0]);
      },
      cnt, cand);
}

// Threshold of every point as a query (SYM's reverse tests): tau + delta -
// |x|^2 as in the forward test; -inf past n.
__global__ void k_rf_thr(const hdb_nnd_element* __restrict__ lists, const float* __restrict__ pn, int64_t n,
                         int64_t np, float* __restrict__ thr) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= np) return;
  float t = -__uint_as_float(0x7F800000u);
  if (i < n) {
    const hdb_nnd_element e = lists[i * kK + (kK - 1)];
    float tau = (label_id(e.label) == kInvalidId) ? __uint_as_float(0x7F800000u) : e.distance;
    if (!(tau >= 0.0f)) tau = __uint_as_float(0x7F800000u);
    const float qn = pn[i];
    const float xn = sqrtf(qn);
    const float yb = xn + sqrtf(tau);
    const float delta = 1.5e-4f * xn * yb + 1e-5f * (yb * yb + qn) + 2e-5f * tau + 1e-30f;
    t = (tau + delta) - qn;
  }
  thr[i] = t;
}

// One block: 8 waves x 32 query rows; every tile of 64 points passes
// through LDS (double-buffered, the next tile's loads in flight during the
// current tile's products).  Lane l of a wave holds, for query sub-tile s,
// the B fragments of query qb + 16 s + (l % 16); a 16 x 16 result tile gives
// lane l the products of points 4 (l / 16) + q (q < 4) with that query.
// Query index qi < m is row act[qi] (qi without act), the point of row r is
// ptid[r] (r without ptid); blockIdx.y streams tiles [y tpc, (y + 1) tpc).
// SYM (the first round over every point): block b streams only the tiles
// from its own points on (chunk y: y tpc past them), and for tiles past its own points also tests the
// other direction (the tile's point y against query q, with y's threshold
// thr_y from k_rf_thr): each pair's products are formed once, which halves
// the matrix work.  Tiles before a block's points are covered by the
// earlier blocks' reverse tests.
template <int KS, bool SYM>
__global__ __launch_bounds__(kRfThreads) void k_rf_scan(const rf_bf16x8* __restrict__ xh, const rf_bf16x8* __restrict__ xl,
                                                    const float* __restrict__ pn,
                                                    const hdb_nnd_element* __restrict__ rows, int64_t n,
                                                    const int32_t* __restrict__ ptid, const int32_t* __restrict__ act,
                                                    int64_t m, int64_t ntiles, int64_t tpc,
                                                    const float* __restrict__ thr_pt,
                                                    int32_t* __restrict__ cnt, int32_t* __restrict__ cand) {
  constexpr int CH = KS * 4;                // 16-byte chunks per row
  constexpr int RS = KS * 32 + kRfPad;      // LDS row stride in BF16 elements
  constexpr int kLoads = 512 * KS / kRfThreads;  // 16-byte chunks per thread per tile (both halves)
  __shared__ __attribute__((aligned(16))) __bf16 s_h[2][kRfTile * RS];
  __shared__ __attribute__((aligned(16))) __bf16 s_l[2][kRfTile * RS];
  __shared__ __attribute__((aligned(16))) float s_pn[2][kRfTile];
  __shared__ __attribute__((aligned(16))) float s_thr[SYM ? 2 : 1][SYM ? kRfTile : 4];
  __shared__ uint32_t s_qrow[kRfWaves][kRfQueue], s_stop[kRfWaves];
  __shared__ int32_t s_qid[kRfWaves][kRfQueue];
  const unsigned lane = __lane_id();
  const unsigned w = threadIdx.x >> 6;
  RfQueue qu{s_qrow[w], s_qid[w], &s_stop[w], 0};
  if (threadIdx.x < kRfWaves) s_stop[threadIdx.x] = 0;
  const int col = static_cast<int>(lane & 15), grp = static_cast<int>(lane >> 4);
  const int64_t qb = static_cast<int64_t>(blockIdx.x) * kRfBlockQ + static_cast<int64_t>(w) * (kRfQS * 16);
  constexpr int kOwnTiles = kRfBlockQ / kRfTile;  // tiles holding the block's own points (SYM)
  const int64_t own0 = SYM ? static_cast<int64_t>(blockIdx.x) * kOwnTiles : 0;
  const int64_t t0 = own0 + static_cast<int64_t>(blockIdx.y) * tpc;
  const int64_t t1 = t0 + tpc < ntiles ? t0 + tpc : ntiles;
  if (t0 >= t1) return;  // uniform across the block: a stream that ends before this chunk

  // query fragments and thresholds; past m the thresholds are -inf
  rf_bf16x8 bh[kRfQS][KS], bl[kRfQS][KS];
  float thr[kRfQS], qn2[kRfQS];
  int64_t qrow[kRfQS], qpt[kRfQS];
#pragma unroll
  for (int s = 0; s < kRfQS; ++s) {
    const int64_t qi = qb + s * 16 + col;
    const int64_t r = qi < m ? (act ? static_cast<int64_t>(act[qi]) : qi) : -1;
    int64_t q = r >= 0 ? (ptid ? static_cast<int64_t>(ptid[r]) : r) : -1;
    if (q >= n) q = -1;  // a query id outside [0, n) collects nothing
    qrow[s] = r;
    qpt[s] = q;
    const int64_t xr = q >= 0 ? q : 0;
#pragma unroll
    for (int kk = 0; kk < KS; ++kk) {
      bh[s][kk] = xh[xr * CH + kk * 4 + grp];
      bl[s][kk] = xl[xr * CH + kk * 4 + grp];
    }
    qn2[s] = q >= 0 ? pn[q] : __uint_as_float(0x7F800000u);
    float t = -__uint_as_float(0x7F800000u);
    if (q >= 0) {
      const hdb_nnd_element e = rows[r * kK + (kK - 1)];
      float tau = (label_id(e.label) == kInvalidId) ? __uint_as_float(0x7F800000u) : e.distance;
      if (!(tau >= 0.0f)) tau = __uint_as_float(0x7F800000u);  // NaN: no bound
      const float qn = pn[q];
      const float xn = sqrtf(qn);
      const float yb = xn + sqrtf(tau);
      const float delta = 1.5e-4f * xn * yb + 1e-5f * (yb * yb + qn) + 2e-5f * tau + 1e-30f;
      t = (tau + delta) - qn;
    }
    thr[s] = t;
  }

  // tile loader: chunk c < 256 KS is row c / CH, chunk c % CH of the high
  // half, the rest the same of the low half; thread t takes t + 512 j
  auto load_tile = [&](int64_t t, rf_bf16x8 (&reg)[kLoads], float& pv, float& tv) {
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
      const int c = static_cast<int>(threadIdx.x) + kRfThreads * j;
      const int half = c / (256 * KS);
      const int wi = c - half * 256 * KS;
      const int row = wi / CH, ch = wi - (wi / CH) * CH;
      const int64_t src = (t * kRfTile + row) * CH + ch;
      reg[j] = half ? xl[src] : xh[src];
    }
    pv = threadIdx.x < kRfTile ? pn[t * kRfTile + threadIdx.x] : 0.0f;
    if (SYM) tv = threadIdx.x < kRfTile ? thr_pt[t * kRfTile + threadIdx.x] : 0.0f;
  };
  auto store_tile = [&](int buf, const rf_bf16x8 (&reg)[kLoads], float pv, float tv) {
    if (SYM && threadIdx.x < kRfTile) s_thr[buf][threadIdx.x] = tv;
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
      const int c = static_cast<int>(threadIdx.x) + kRfThreads * j;
      const int half = c / (256 * KS);
      const int wi = c - half * 256 * KS;
      const int row = wi / CH, ch = wi - (wi / CH) * CH;
      __bf16* dst = (half ? s_l[buf] : s_h[buf]) + row * RS + ch * 8;
      *reinterpret_cast<rf_bf16x8*>(dst) = reg[j];
    }
    if (threadIdx.x < kRfTile) s_pn[buf][threadIdx.x] = pv;
  };

  rf_bf16x8 nxt[kLoads];
  float npv = 0.0f, ntv = 0.0f;
  load_tile(t0, nxt, npv, ntv);
  store_tile(0, nxt, npv, ntv);
  __syncthreads();
  for (int64_t t = t0; t < t1; ++t) {
    const int buf = static_cast<int>((t - t0) & 1);
    const bool more = t + 1 < t1;
    if (more) load_tile(t + 1, nxt, npv, ntv);
    rf_f32x4 acc[4][kRfQS];
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int s = 0; s < kRfQS; ++s) acc[r][s] = rf_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int kk = 0; kk < KS; ++kk) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int off = (r * 16 + col) * RS + kk * 32 + grp * 8;
        const rf_bf16x8 ah = *reinterpret_cast<const rf_bf16x8*>(s_h[buf] + off);
        const rf_bf16x8 al = *reinterpret_cast<const rf_bf16x8*>(s_l[buf] + off);
#pragma unroll
        for (int s = 0; s < kRfQS; ++s)
          acc[r][s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bh[s][kk], acc[r][s], 0, 0, 0);
#pragma unroll
        for (int s = 0; s < kRfQS; ++s)
          acc[r][s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bl[s][kk], acc[r][s], 0, 0, 0);
#pragma unroll
        for (int s = 0; s < kRfQS; ++s)
          acc[r][s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, bh[s][kk], acc[r][s], 0, 0, 0);
      }
    }
    {  // queries past the cap stop collecting
      const uint32_t stop = s_stop[w];
#pragma unroll
      for (int s = 0; s < kRfQS; ++s)
        if ((stop >> (16 * s + col)) & 1u) thr[s] = -__uint_as_float(0x7F800000u);
    }
    rf_survivors(acc, s_pn[buf], thr, qrow, qpt, t, grp, col, qu, cnt, cand);
    if (SYM && t >= own0 + kOwnTiles) rf_reverse(acc, s_thr[buf], qn2, qpt, t, grp, qu, cnt, cand);
    if (more) store_tile(buf ^ 1, nxt, npv, ntv);
    __syncthreads();
  }
  rf_flush(qu, qu.len, cnt, cand);
}

// FP32 form for d <= 32, where the split-BF16 bound (relative to |x| |y|)
// is loose against small neighbour distances: v_mfma_f32_16x16x4f32 on the
// FP32 rows (padded to dp = d rounded up to 4), one product chain per
// tile.  Each product and each add rounds at most once, so the dot carries
// at most 2 dp 2^-24 sum|x_i y_i| and the norms dp 2^-24 |.|^2:
//   delta_q = (4 dp + 16) 2^-24 (|x| yb + |x|^2 + yb^2) + 2e-5 tau_q
// covers the test.  Lane l holds A[16 r + l % 16][4 kk + l / 16] and
// B[4 kk + l / 16][l % 16]; the result layout is that of the BF16 form.
__global__ void k_rf_pad32(const float* __restrict__ X, int64_t n, int d, int dp, int64_t np,
                           float* __restrict__ xp) {
  const int64_t e = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (e >= np * dp) return;
  const int64_t i = e / dp;
  const int k = static_cast<int>(e - i * dp);
  xp[e] = (i < n && k < d) ? X[i * d + k] : 0.0f;
}

template <int KS4>
__global__ __launch_bounds__(kRfThreads) void k_rf_scan32(const float* __restrict__ xp, const float* __restrict__ pn,
                                                      const hdb_nnd_element* __restrict__ rows, int64_t n,
                                                      const int32_t* __restrict__ ptid,
                                                      const int32_t* __restrict__ act, int64_t m, int64_t ntiles,
                                                      int64_t tpc, int32_t* __restrict__ cnt,
                                                      int32_t* __restrict__ cand) {
  constexpr int DP = KS4 * 4;
  constexpr int RSF = DP + 1;         // odd LDS row stride: the 16 rows of a read hit distinct banks
  constexpr int kChunks = 16 * DP;    // float4 chunks per tile (<= kRfThreads for DP <= 32)
  static_assert(kChunks <= kRfThreads, "one chunk per thread");
  __shared__ float s_x[2][kRfTile * RSF];
  __shared__ __attribute__((aligned(16))) float s_pn[2][kRfTile];
  __shared__ uint32_t s_qrow[kRfWaves][kRfQueue], s_stop[kRfWaves];
  __shared__ int32_t s_qid[kRfWaves][kRfQueue];
  const unsigned lane = __lane_id();
  const unsigned w = threadIdx.x >> 6;
  RfQueue qu{s_qrow[w], s_qid[w], &s_stop[w], 0};
  if (threadIdx.x < kRfWaves) s_stop[threadIdx.x] = 0;
  const int col = static_cast<int>(lane & 15), grp = static_cast<int>(lane >> 4);
  const int64_t qb = static_cast<int64_t>(blockIdx.x) * kRfBlockQ + static_cast<int64_t>(w) * (kRfQS * 16);
  const int64_t t0 = static_cast<int64_t>(blockIdx.y) * tpc;
  const int64_t t1 = t0 + tpc < ntiles ? t0 + tpc : ntiles;

  float bq[kRfQS][KS4];
  float thr[kRfQS];
  int64_t qrow[kRfQS], qpt[kRfQS];
#pragma unroll
  for (int s = 0; s < kRfQS; ++s) {
    const int64_t qi = qb + s * 16 + col;
    const int64_t r = qi < m ? (act ? static_cast<int64_t>(act[qi]) : qi) : -1;
    int64_t q = r >= 0 ? (ptid ? static_cast<int64_t>(ptid[r]) : r) : -1;
    if (q >= n) q = -1;
    qrow[s] = r;
    qpt[s] = q;
    const int64_t xr = q >= 0 ? q : 0;
#pragma unroll
    for (int kk = 0; kk < KS4; ++kk) bq[s][kk] = xp[xr * DP + kk * 4 + grp];
    float t = -__uint_as_float(0x7F800000u);
    if (q >= 0) {
      const hdb_nnd_element e = rows[r * kK + (kK - 1)];
      float tau = (label_id(e.label) == kInvalidId) ? __uint_as_float(0x7F800000u) : e.distance;
      if (!(tau >= 0.0f)) tau = __uint_as_float(0x7F800000u);
      const float qn = pn[q];
      const float xn = sqrtf(qn);
      const float yb = xn + sqrtf(tau);
      const float c = static_cast<float>(4 * DP + 16) * 5.9604645e-8f;  // 2^-24
      const float delta = c * (xn * yb + qn + yb * yb) + 2e-5f * tau + 1e-30f;
      t = (tau + delta) - qn;
    }
    thr[s] = t;
  }

  auto load_tile = [&](int64_t t, float4& reg, float& pv) {
    const int c = static_cast<int>(threadIdx.x);
    if (c < kChunks) {
      const int row = c / KS4, c4 = c - (c / KS4) * KS4;
      reg = *reinterpret_cast<const float4*>(xp + (t * kRfTile + row) * DP + c4 * 4);
    }
    pv = threadIdx.x < kRfTile ? pn[t * kRfTile + threadIdx.x] : 0.0f;
  };
  auto store_tile = [&](int buf, const float4& reg, float pv) {
    const int c = static_cast<int>(threadIdx.x);
    if (c < kChunks) {
      const int row = c / KS4, c4 = c - (c / KS4) * KS4;
      float* dst = s_x[buf] + row * RSF + c4 * 4;
      dst[0] = reg.x;
      dst[1] = reg.y;
      dst[2] = reg.z;
      dst[3] = reg.w;
    }
    if (threadIdx.x < kRfTile) s_pn[buf][threadIdx.x] = pv;
  };

  if (t0 >= t1) return;  // uniform across the block
  float4 nxt = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  float npv = 0.0f;
  load_tile(t0, nxt, npv);
  store_tile(0, nxt, npv);
  __syncthreads();
  for (int64_t t = t0; t < t1; ++t) {
    const int buf = static_cast<int>((t - t0) & 1);
    const bool more = t + 1 < t1;
    if (more) load_tile(t + 1, nxt, npv);
    rf_f32x4 acc[4][kRfQS];
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int s = 0; s < kRfQS; ++s) acc[r][s] = rf_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int kk = 0; kk < KS4; ++kk) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float a = s_x[buf][(r * 16 + col) * RSF + kk * 4 + grp];
#pragma unroll
        for (int s = 0; s < kRfQS; ++s) acc[r][s] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, bq[s][kk], acc[r][s], 0, 0, 0);
      }
    }
    {  // queries past the cap stop collecting
      const uint32_t stop = s_stop[w];
#pragma unroll
      for (int s = 0; s < kRfQS; ++s)
        if ((stop >> (16 * s + col)) & 1u) thr[s] = -__uint_as_float(0x7F800000u);
    }
    rf_survivors(acc, s_pn[buf], thr, qrow, qpt, t, grp, col, qu, cnt, cand);
    if (more) store_tile(buf ^ 1, nxt, npv);
    __syncthreads();
  }
  rf_flush(qu, qu.len, cnt, cand);
}

// One wave per query index qi < m (row act[qi], point ptid[row]): its kept
// survivors -> exact FP32 keys -> bitonic sort of 128.  With at most kRfCap
// survivors the first 32 are the exact list.  Past the cap, the 32 nearest
// kept survivors merged with the row's current list (repeated keys dropped)
// give 32 distinct points whose entry 31 is a tighter bound, and the row is
// queued (next) for another round.
__global__ __launch_bounds__(256) void k_rf_select(const float* __restrict__ X, int64_t n, int d,
                                                   const int32_t* __restrict__ ptid, const int32_t* __restrict__ act,
                                                   int64_t m, const int32_t* __restrict__ cnt,
                                                   const int32_t* __restrict__ cand, hdb_nnd_element* __restrict__ rows,
                                                   int32_t* __restrict__ next, unsigned long long* __restrict__ stats) {
  const unsigned lane = __lane_id();
  const int64_t qi = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (qi >= m) return;
  const int64_t r = act ? static_cast<int64_t>(act[qi]) : qi;
  const int64_t q = ptid ? static_cast<int64_t>(ptid[r]) : r;
  hdb_nnd_element* row = rows + r * kK;
  if (q < 0 || q >= n) {  // no neighbours for an id outside [0, n)
    if (lane < kK) row[lane] = key_to_list_elem(kKeyMax);
    return;
  }
  const int c = cnt[r];
  const int cc = c < kRfCap ? c : kRfCap;
  if (lane == 0) atomicAdd(stats, static_cast<unsigned long long>(c));
  const bool vec4 = (d & 3) == 0 && (reinterpret_cast<uintptr_t>(X) & 15) == 0;
  const float* xq = X + q * d;
  uint64_t k0 = kKeyMax, k1 = kKeyMax;
  if (static_cast<int>(lane) < cc) {
    const uint32_t id = static_cast<uint32_t>(cand[r * kRfCap + lane]);
    const float* y = X + static_cast<int64_t>(id) * d;
    k0 = make_key(vec4 ? d2_vec4(xq, y, d) : d2_any(xq, y, d), id, 0u);
  }
  if (static_cast<int>(lane) + 64 < cc) {
    const uint32_t id = static_cast<uint32_t>(cand[r * kRfCap + 64 + lane]);
    const float* y = X + static_cast<int64_t>(id) * d;
    k1 = make_key(vec4 ? d2_vec4(xq, y, d) : d2_any(xq, y, d), id, 0u);
  }
  bitonic128(k0, k1);
  if (c <= kRfCap) {
    if (lane < kK) row[lane] = key_to_list_elem(k0);
    return;
  }
  uint64_t v = k0;  // lanes 0..31: the 32 nearest kept survivors
  if (lane >= 32) {
    const hdb_nnd_element e = row[lane - 32];
    const uint32_t id = label_id(e.label);
    v = (id == kInvalidId || static_cast<int64_t>(id) >= n) ? kKeyMax : make_key(e.distance, id, 0u);
  }
  v = bitonic_group<64>(v);
  const uint64_t prev = shfl_u64(v, lane == 0 ? 0 : static_cast<int>(lane) - 1);
  const bool keep = v != kKeyMax && (lane == 0 || v != prev);
  const uint64_t bal = __ballot(keep);
  const int pos = __popcll(bal & lanemask_lt());
  const int distinct = __popcll(bal);
  if (keep && pos < kK) row[pos] = key_to_list_elem(v);
  if (lane < kK && static_cast<int>(lane) >= distinct) row[lane] = key_to_list_elem(kKeyMax);
  if (lane == 0) {
    const unsigned long long slot = atomicAdd(stats + 1, 1ull);
    next[slot] = static_cast<int32_t>(r);
  }
}

__global__ void k_rf_zero(const int32_t* __restrict__ act, int64_t m, int32_t* __restrict__ cnt) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < m) cnt[act[i]] = 0;
}

// Points of the rows still past the cap (for the exact brute force).
__global__ void k_rf_points(const int32_t* __restrict__ ptid, const int32_t* __restrict__ act, int64_t m,
                            int32_t* __restrict__ pts) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < m) pts[i] = ptid ? ptid[act[i]] : act[i];
}

__global__ void k_rf_scatter(const int32_t* __restrict__ act, int64_t m, const int32_t* __restrict__ ids,
                             const float* __restrict__ d2, hdb_nnd_element* __restrict__ rows) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= m * kK) return;
  const int64_t i = t / kK;
  const int j = static_cast<int>(t - i * kK);
  hdb_nnd_element e;
  e.label = ids[t];
  e.distance = ids[t] < 0 ? __uint_as_float(0x7F800000u) : d2[t];
  rows[static_cast<int64_t>(act[i]) * kK + j] = e;
}

// rows[i] = lists[qids[i]] (bounded query mode), and the rows back out as
// ids and distances.
__global__ void k_rf_gather_rows(const hdb_nnd_element* __restrict__ lists, int64_t n,
                                 const int32_t* __restrict__ qids, int64_t m, hdb_nnd_element* __restrict__ rows) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= m * kK) return;
  const int64_t i = t / kK;
  const int64_t q = qids[i];
  hdb_nnd_element e;
  if (q >= 0 && q < n) {
    e = lists[q * kK + (t - i * kK)];
  } else {
    e.distance = __uint_as_float(0x7F800000u);
    e.label = static_cast<int32_t>(kInvalidId);
  }
  rows[t] = e;
}

__global__ void k_rf_rows_out(const hdb_nnd_element* __restrict__ rows, int64_t m, int kq,
                              int32_t* __restrict__ out_ids, float* __restrict__ out_d2) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= m * kq) return;
  const int64_t i = t / kq;
  const hdb_nnd_element e = rows[i * kK + (t - i * kq)];
  const uint32_t id = label_id(e.label);
  out_ids[t] = id == kInvalidId ? -1 : static_cast<int32_t>(id);
  if (out_d2) out_d2[t] = e.distance;
}

// thr_pt != nullptr: the symmetric first round over every point (rows are
// the points, no active list).  Its streams shrink from all tiles to none, so
// the longest alone would set the time while the point blocks are few (100k
// points: 391 blocks): they are cut into equal chunks for about
// kRfSymBlocks blocks, eight for each that a CU holds at once.  From 2M
// points on one or two chunks take the whole stream (scan at 30k x 128: 3.45 ->
// 1.11 ms, at 100k x 128 8.9 -> 7.6 ms).
constexpr int64_t kRfSymBlocks = 4096;

template <int KS>
int launch_scan(hdb_ctx* ctx, const __bf16* xh, const __bf16* xl, const float* pn, const hdb_nnd_element* rows,
                int64_t n, const int32_t* ptid, const int32_t* act, int64_t m, int64_t ntiles, const float* thr_pt,
                int32_t* cnt, int32_t* cand) {
  const int64_t qblocks = (m + kRfBlockQ - 1) / kRfBlockQ;
  if (thr_pt) {
    const int64_t steps = qblocks * (ntiles + 1) / 2;
    const int64_t cut = std::min<int64_t>(ntiles, std::max<int64_t>(32, (steps + kRfSymBlocks - 1) / kRfSymBlocks));
    hipLaunchKernelGGL((k_rf_scan<KS, true>),
                       dim3(static_cast<unsigned>(qblocks), static_cast<unsigned>((ntiles + cut - 1) / cut)),
                       dim3(kRfThreads), 0, ctx->stream, reinterpret_cast<const rf_bf16x8*>(xh),
                       reinterpret_cast<const rf_bf16x8*>(xl), pn, rows, n, ptid, act, m, ntiles, cut, thr_pt, cnt,
                       cand);
    HDB_LAUNCHED();
    return HDB_OK;
  }
  // stream chunks so that the grid has at least 512 blocks (two per CU)
  int64_t chunks = std::max<int64_t>(1, std::min<int64_t>((512 + qblocks - 1) / qblocks, ntiles));
  chunks = std::min<int64_t>(chunks, 65535);
  const int64_t tpc = (ntiles + chunks - 1) / chunks;
  chunks = (ntiles + tpc - 1) / tpc;
  hipLaunchKernelGGL((k_rf_scan<KS, false>), dim3(static_cast<unsigned>(qblocks), static_cast<unsigned>(chunks)),
                     dim3(kRfThreads), 0, ctx->stream, reinterpret_cast<const rf_bf16x8*>(xh),
                     reinterpret_cast<const rf_bf16x8*>(xl), pn, rows, n, ptid, act, m, ntiles, tpc, nullptr, cnt,
                     cand);
  HDB_LAUNCHED();
  return HDB_OK;
}

template <int KS4>
int launch_scan32(hdb_ctx* ctx, const float* xp, const float* pn, const hdb_nnd_element* rows, int64_t n,
                  const int32_t* ptid, const int32_t* act, int64_t m, int64_t ntiles, int32_t* cnt, int32_t* cand) {
  const int64_t qblocks = (m + kRfBlockQ - 1) / kRfBlockQ;
  int64_t chunks = std::max<int64_t>(1, std::min<int64_t>((512 + qblocks - 1) / qblocks, ntiles));
  chunks = std::min<int64_t>(chunks, 65535);
  const int64_t tpc = (ntiles + chunks - 1) / chunks;
  chunks = (ntiles + tpc - 1) / tpc;
  hipLaunchKernelGGL(k_rf_scan32<KS4>, dim3(static_cast<unsigned>(qblocks), static_cast<unsigned>(chunks)),
                     dim3(kRfThreads), 0, ctx->stream, xp, pn, rows, n, ptid, act, m, ntiles, tpc, cnt, cand);
  HDB_LAUNCHED();
  return HDB_OK;
}

constexpr int kRfRounds = 6;  // survivor rounds before the exact brute force takes the rest

// The pass over m0 rows (row r: point ptid[r], or r): rounds of scan and
// select until no row is past the cap, then the exact brute force for the
// rest.  stats_out: survivors and rows past the cap in the first round,
// rows left to the brute force.
int refine_rows(hdb_ctx* ctx, const float* X, int64_t n, int d, hdb_nnd_element* rows, const int32_t* ptid,
                int64_t m0, int64_t* stats_out) {
  const bool f32 = d <= 32;  // FP32 MFMA tiles (else split BF16)
  const int ks = f32 ? (d + 3) / 4 : (d + 31) / 32;
  const int dp = f32 ? ks * 4 : ks * 32;
  const int64_t np = (n + 255) / 256 * 256;
  __bf16 *xh = nullptr, *xl = nullptr;
  float *xp = nullptr, *pn;
  int32_t *cnt, *cand, *qbuf[2];
  unsigned long long* stats;
  if (f32) {
    HDB_CALL(scratch_t(ctx, kSlotRefineXh, np * dp * 2, &xh));  // np x dp floats in the same slot
    xp = reinterpret_cast<float*>(xh);
    xh = nullptr;
  } else {
    HDB_CALL(scratch_t(ctx, kSlotRefineXh, np * dp, &xh));
    HDB_CALL(scratch_t(ctx, kSlotRefineXl, np * dp, &xl));
  }
  HDB_CALL(scratch_t(ctx, kSlotRefineNorm, np, &pn));
  HDB_CALL(scratch_t(ctx, kSlotRefineCand, m0 * kRfCap, &cand));
  HDB_CALL(scratch_t(ctx, kSlotRefineCnt, 3 * m0 + 8, &cnt));
  qbuf[0] = cnt + m0;
  qbuf[1] = cnt + 2 * m0;
  stats = reinterpret_cast<unsigned long long*>(cnt + 3 * m0 + (m0 & 1));  // 8-byte aligned
  if (f32)
    hipLaunchKernelGGL(k_rf_pad32, dim3(grid_for(np * dp, 256)), dim3(256), 0, ctx->stream, X, n, d, dp, np, xp);
  else
    hipLaunchKernelGGL(k_rf_split, dim3(grid_for(np * dp, 256)), dim3(256), 0, ctx->stream, X, n, d, dp, np, xh, xl);
  HDB_LAUNCHED();
  hipLaunchKernelGGL(k_rf_norms, dim3(grid_for(np, 256)), dim3(256), 0, ctx->stream, X, n, d, np, pn);
  HDB_LAUNCHED();
  const int64_t ntiles = (n + kRfTile - 1) / kRfTile;  // padding rows past n up to np exist
  const int32_t* act = nullptr;                         // round 0: every row
  int64_t m = m0;
  // the first round over every point takes the symmetric scan (BF16 form)
  float* thr_all = nullptr;
  if (!f32 && !ptid && m0 == n) {
    HDB_CALL(scratch_t(ctx, kSlotRefineThr, np, &thr_all));
    hipLaunchKernelGGL(k_rf_thr, dim3(grid_for(np, 256)), dim3(256), 0, ctx->stream, rows, pn, n, np, thr_all);
    HDB_LAUNCHED();
  }
  for (int round = 0; round < kRfRounds && m > 0; ++round) {
    const float* thr_pt = round == 0 ? thr_all : nullptr;
    if (act) {
      hipLaunchKernelGGL(k_rf_zero, dim3(grid_for(m, 256)), dim3(256), 0, ctx->stream, act, m, cnt);
      HDB_LAUNCHED();
    } else {
      HDB_CALL(fill_i32(ctx, cnt, m0, 0));
    }
    HDB_CALL(fill_u64(ctx, reinterpret_cast<uint64_t*>(stats), 2, 0));
    {
      Stage s2(ctx, "refine_scan");
      if (f32) {
        switch (ks) {
          case 1: HDB_CALL(launch_scan32<1>(ctx, xp, pn, rows, n, ptid, act, m, ntiles, cnt, cand)); break;
          case 2: HDB_CALL(launch_scan32<2>(ctx, xp, pn, rows, n, ptid, act, m, ntiles, cnt, cand)); break;
          case 3: HDB_CALL(launch_scan32<3>(ctx, xp, pn, rows, n, ptid, act, m, ntiles, cnt, cand)); break;
          case 4: HDB_CALL(launch_scan32<4>(ctx, xp, pn, rows, n, ptid, act, m, ntiles, cnt, cand)); break;
          case 5: HDB_CALL(launch_scan32<5>(ctx, xp, pn, rows, n, ptid, act, m, ntiles, cnt, cand)); break;
          case 6: HDB_CALL(launch_scan32<6>(ctx, xp, pn, rows, n, ptid, act, m, ntiles, cnt, cand)); break;
          case 7: HDB_CALL(launch_scan32<7>(ctx, xp, pn, rows, n, ptid, act, m, ntiles, cnt, cand)); break;
          default: HDB_CALL(launch_scan32<8>(ctx, xp, pn, rows, n, ptid, act, m, ntiles, cnt, cand)); break;
        }
      } else {
        switch (ks) {
          case 1: HDB_CALL(launch_scan<1>(ctx, xh, xl, pn, rows, n, ptid, act, m, ntiles, thr_pt, cnt, cand)); break;
          case 2: HDB_CALL(launch_scan<2>(ctx, xh, xl, pn, rows, n, ptid, act, m, ntiles, thr_pt, cnt, cand)); break;
          case 3: HDB_CALL(launch_scan<3>(ctx, xh, xl, pn, rows, n, ptid, act, m, ntiles, thr_pt, cnt, cand)); break;
          default: HDB_CALL(launch_scan<4>(ctx, xh, xl, pn, rows, n, ptid, act, m, ntiles, thr_pt, cnt, cand)); break;
        }
      }
    }
    int32_t* next = qbuf[round & 1];
    {
      Stage s3(ctx, "refine_select");
      hipLaunchKernelGGL(k_rf_select, dim3(grid_for(m, 4)), dim3(256), 0, ctx->stream, X, n, d, ptid, act, m, cnt,
                         cand, rows, next, stats);
      HDB_LAUNCHED();
    }
    unsigned long long h[2];
    HDB_HIP(hipMemcpyAsync(h, stats, sizeof(h), hipMemcpyDeviceToHost, ctx->stream));
    HDB_HIP(hipStreamSynchronize(ctx->stream));
    if (round == 0) {
      stats_out[0] = static_cast<int64_t>(h[0]);
      stats_out[1] = static_cast<int64_t>(h[1]);
    }
    m = static_cast<int64_t>(h[1]);
    act = next;
  }
  stats_out[2] = m;
  if (m > 0) {  // still past the cap after every round: exact FP32 brute force
    Stage s4(ctx, "refine_overflow");
    int32_t *ids, *pts;
    float* dd;
    HDB_CALL(scratch_t(ctx, kSlotRefineOvfIds, m * (kK + 1), &ids));
    HDB_CALL(scratch_t(ctx, kSlotRefineOvfD2, m * kK, &dd));
    pts = ids + m * kK;
    hipLaunchKernelGGL(k_rf_points, dim3(grid_for(m, 256)), dim3(256), 0, ctx->stream, ptid, act, m, pts);
    HDB_LAUNCHED();
    HDB_CALL(bruteforce_knn(ctx, X, n, d, pts, m, kK, ids, dd));
    hipLaunchKernelGGL(k_rf_scatter, dim3(grid_for(m * kK, 256)), dim3(256), 0, ctx->stream, act, m, ids, dd, rows);
    HDB_LAUNCHED();
  }
  return HDB_OK;
}

}  // namespace

int refine_knng(hdb_ctx* ctx, const float* X, int64_t n, int d, hdb_nnd_element* lists, int64_t* candidates_out,
                int64_t* overflow_out) {
  if (!X || !lists || n < 2 || d < 1) return ctx->fail(HDB_EINVAL, "bad refine arguments");
  if (d > 128) return ctx->fail(HDB_EUNSUPPORTED, "the BF16 refinement is built for d <= 128");
  if (n >= (static_cast<int64_t>(1) << 31) / kRfCap) return ctx->fail(HDB_EINVAL, "n too large for the refinement");
  Stage st(ctx, "refine_knng");
  int64_t s[3] = {0, 0, 0};
  HDB_CALL(refine_rows(ctx, X, n, d, lists, nullptr, n, s));
  if (candidates_out) *candidates_out = s[0];
  if (overflow_out) *overflow_out = s[1];
  for (int i = 0; i < 3; ++i) ctx->refine_stats[i] = s[i];
  return HDB_OK;
}

int exact_knn_bounded(hdb_ctx* ctx, const float* X, int64_t n, int d, const hdb_nnd_element* lists,
                      const int32_t* qids, int64_t m, int kq, int32_t* out_ids, float* out_d2) {
  if (!X || !lists || !qids || !out_ids || n < 2 || d < 1 || m < 0) return ctx->fail(HDB_EINVAL, "bad arguments");
  if (kq < 1 || kq > kK) return ctx->fail(HDB_EINVAL, "kq must be in [1,32]");
  if (d > 128) return ctx->fail(HDB_EUNSUPPORTED, "the BF16 refinement is built for d <= 128");
  if (n >= (static_cast<int64_t>(1) << 31)) return ctx->fail(HDB_EINVAL, "n must be below 2^31");
  if (m == 0) return HDB_OK;
  if (m >= (static_cast<int64_t>(1) << 31) / kRfCap) return ctx->fail(HDB_EINVAL, "too many queries");
  Stage st(ctx, "exact_knn_bounded");
  hdb_nnd_element* rows;
  HDB_CALL(scratch_t(ctx, kSlotRefineRows, m * kK, &rows));
  hipLaunchKernelGGL(k_rf_gather_rows, dim3(grid_for(m * kK, 256)), dim3(256), 0, ctx->stream, lists, n, qids, m,
                     rows);
  HDB_LAUNCHED();
  int64_t s[3] = {0, 0, 0};
  HDB_CALL(refine_rows(ctx, X, n, d, rows, qids, m, s));
  hipLaunchKernelGGL(k_rf_rows_out, dim3(grid_for(m * kq, 256)), dim3(256), 0, ctx->stream, rows, m, kq, out_ids,
                     out_d2);
  HDB_LAUNCHED();
  for (int i = 0; i < 3; ++i) ctx->refine_stats[i] = s[i];
  return HDB_OK;
}

}  // namespace hdb
