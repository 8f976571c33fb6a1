// Device primitives for gfx950: fills, int32->int64 exclusive scan and a
// stable LSD radix sort (8-bit digits, wave64 match-based ranking).
#include <utility>

#include "hdb_internal.hpp"

namespace hdb {

// ---------------------------------------------------------------- fills --
template <typename T>
__global__ void k_fill(T* __restrict__ p, int64_t n, T v) {
  int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  for (; i < n; i += stride) p[i] = v;
}

template <typename T>
static int fill_t(hdb_ctx* ctx, T* p, int64_t n, T v) {
  if (n <= 0) return HDB_OK;
  unsigned grid = grid_for(n, 256);
  if (grid > 65536u) grid = 65536u;
  hipLaunchKernelGGL(k_fill<T>, dim3(grid), dim3(256), 0, ctx->stream, p, n, v);
  HDB_LAUNCHED();
  return HDB_OK;
}
int fill_i32(hdb_ctx* ctx, int32_t* p, int64_t n, int32_t v) { return fill_t(ctx, p, n, v); }
int fill_u64(hdb_ctx* ctx, uint64_t* p, int64_t n, uint64_t v) { return fill_t(ctx, p, n, v); }

int read_i64(hdb_ctx* ctx, const int64_t* p, int64_t* out) {
  HDB_HIP(hipMemcpyAsync(out, p, sizeof(int64_t), hipMemcpyDeviceToHost, ctx->stream));
  HDB_HIP(hipStreamSynchronize(ctx->stream));
  return HDB_OK;
}
int read_i64_async(hdb_ctx* ctx, const int64_t* p, int slot) {
  if (!ctx->pinned || slot < 0 || slot > 1) return ctx->fail(HDB_EINVAL, "bad readback slot");
  HDB_HIP(hipMemcpyAsync(ctx->pinned + slot, p, sizeof(int64_t), hipMemcpyDeviceToHost, ctx->stream));
  HDB_HIP(hipEventRecord(ctx->ready[slot], ctx->stream));
  return HDB_OK;
}
int wait_i64(hdb_ctx* ctx, int slot, int64_t* out) {
  if (!ctx->pinned || slot < 0 || slot > 1) return ctx->fail(HDB_EINVAL, "bad readback slot");
  HDB_HIP(hipEventSynchronize(ctx->ready[slot]));
  *out = ctx->pinned[slot];
  return HDB_OK;
}
int read_i32(hdb_ctx* ctx, const int32_t* p, int32_t* out) {
  HDB_HIP(hipMemcpyAsync(out, p, sizeof(int32_t), hipMemcpyDeviceToHost, ctx->stream));
  HDB_HIP(hipStreamSynchronize(ctx->stream));
  return HDB_OK;
}

// ----------------------------------------------------------------- scan --
constexpr int kScanBlock = 256;
constexpr int kScanItems = 8;
constexpr int kScanTile = kScanBlock * kScanItems;

__device__ __forceinline__ int64_t wave_incl_scan(int64_t v) {
  const unsigned lane = __lane_id();
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    int64_t u = __shfl_up(v, o);
    if (lane >= static_cast<unsigned>(o)) v += u;
  }
  return v;
}

// Block-wide exclusive scan of one value per thread (256 threads); returns
// the exclusive prefix and writes the block total to *total.
__device__ __forceinline__ int64_t block_excl_scan(int64_t v, int64_t* total) {
  __shared__ int64_t wsum[kScanBlock / 64];
  const unsigned lane = __lane_id();
  const unsigned w = threadIdx.x >> 6;
  int64_t incl = wave_incl_scan(v);
  if (lane == 63) wsum[w] = incl;
  __syncthreads();
  int64_t off = 0, tot = 0;
#pragma unroll
  for (unsigned i = 0; i < kScanBlock / 64; ++i) {
    if (i < w) off += wsum[i];
    tot += wsum[i];
  }
  __syncthreads();
  *total = tot;
  return off + incl - v;
}

__global__ void k_scan_tiles(const int32_t* __restrict__ in, int64_t n, int64_t* __restrict__ tile_sum) {
  const int64_t base = static_cast<int64_t>(blockIdx.x) * kScanTile + threadIdx.x * kScanItems;
  int64_t s = 0;
#pragma unroll
  for (int i = 0; i < kScanItems; ++i) {
    int64_t idx = base + i;
    if (idx < n) s += in[idx];
  }
  int64_t total;
  block_excl_scan(s, &total);
  if (threadIdx.x == 0) tile_sum[blockIdx.x] = total;
}

// Single-block exclusive scan of the tile sums in place.
__global__ void k_scan_sums(int64_t* __restrict__ sums, int64_t m) {
  __shared__ int64_t carry_s;
  if (threadIdx.x == 0) carry_s = 0;
  __syncthreads();
  for (int64_t start = 0; start < m; start += kScanBlock) {
    int64_t idx = start + threadIdx.x;
    int64_t v = idx < m ? sums[idx] : 0;
    int64_t total;
    int64_t ex = block_excl_scan(v, &total);
    int64_t carry = carry_s;
    if (idx < m) sums[idx] = carry + ex;
    __syncthreads();
    if (threadIdx.x == 0) carry_s = carry + total;
    __syncthreads();
  }
}

__global__ void k_scan_apply(const int32_t* __restrict__ in, int64_t n, const int64_t* __restrict__ tile_off,
                             int64_t* __restrict__ out) {
  const int64_t base = static_cast<int64_t>(blockIdx.x) * kScanTile + threadIdx.x * kScanItems;
  int32_t v[kScanItems];
  int64_t s = 0;
#pragma unroll
  for (int i = 0; i < kScanItems; ++i) {
    int64_t idx = base + i;
    v[i] = idx < n ? in[idx] : 0;
    s += v[i];
  }
  int64_t total;
  int64_t ex = block_excl_scan(s, &total) + tile_off[blockIdx.x];
#pragma unroll
  for (int i = 0; i < kScanItems; ++i) {
    int64_t idx = base + i;
    if (idx < n) out[idx] = ex;
    ex += v[i];
  }
  if (blockIdx.x == gridDim.x - 1 && threadIdx.x == kScanBlock - 1) out[n] = ex;
}

int scan_i32_to_i64(hdb_ctx* ctx, const int32_t* in, int64_t n, int64_t* out) {
  if (n <= 0) {
    HDB_CALL(fill_t<int64_t>(ctx, out, 1, 0));
    return HDB_OK;
  }
  const int64_t tiles = (n + kScanTile - 1) / kScanTile;
  int64_t* sums;
  HDB_CALL(scratch_t(ctx, kSlotScanTmp, tiles, &sums));
  hipLaunchKernelGGL(k_scan_tiles, dim3(tiles), dim3(kScanBlock), 0, ctx->stream, in, n, sums);
  HDB_LAUNCHED();
  hipLaunchKernelGGL(k_scan_sums, dim3(1), dim3(kScanBlock), 0, ctx->stream, sums, tiles);
  HDB_LAUNCHED();
  hipLaunchKernelGGL(k_scan_apply, dim3(tiles), dim3(kScanBlock), 0, ctx->stream, in, n, sums, out);
  HDB_LAUNCHED();
  return HDB_OK;
}

// ----------------------------------------------------------- radix sort --
// A tile is WAVES waves x CH chunks x 64 lanes.  Within a wave, chunk c
// holds keys [wave_base + 64c, wave_base + 64c + 64), one per lane, so the
// rank order (chunk, lane) is the input order and the sort is stable.
constexpr int kRsBins = 256;
constexpr int64_t kRsSmallKeys = 400000;

// Input read through a segment map: logical index i lives in segment g with
// pre[g] <= i < pre[g+1], at physical index g * seg_cap + (i - pre[g]).
// pre == nullptr: identity.  At most kRsMaxSegs segments.
constexpr int kRsMaxSegs = 64;

struct RsSegs {
  const int64_t* pre;
  int nseg;
  int64_t seg_cap;
};

__device__ __forceinline__ void rs_load_segs(const RsSegs& sg, int64_t* s_pre) {
  if (sg.pre)
    for (int i = threadIdx.x; i <= sg.nseg; i += blockDim.x) s_pre[i] = sg.pre[i];
}

__device__ __forceinline__ int64_t rs_phys(const RsSegs& sg, const int64_t* s_pre, int64_t i) {
  if (!sg.pre) return i;
  int lo = 0, hi = sg.nseg;  // largest g with s_pre[g] <= i
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (s_pre[mid] <= i) lo = mid; else hi = mid;
  }
  return static_cast<int64_t>(lo) * sg.seg_cap + (i - s_pre[lo]);
}

// Segment walk over one wave's consecutive chunks: the segment of the
// wave's first key is found once (wave-uniform binary search); each chunk
// then advances past the boundaries it has crossed (segments hold far more
// than a chunk, so this rarely loops), and a lane past its chunk's segment
// end searches on its own.
struct RsWalk {
  int seg;       // segment of the current chunk's first key
  int64_t next;  // start of the following segment (INT64_MAX past the last)
};

__device__ __forceinline__ RsWalk rs_walk_begin(const RsSegs& sg, const int64_t* s_pre, int64_t c0) {
  RsWalk wk{0, INT64_MAX};
  if (!sg.pre) return wk;
  int lo = 0, hi = sg.nseg;  // largest g with s_pre[g] <= c0
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (s_pre[mid] <= c0) lo = mid; else hi = mid;
  }
  wk.seg = lo;
  wk.next = lo + 1 < sg.nseg ? s_pre[lo + 1] : INT64_MAX;
  return wk;
}

__device__ __forceinline__ int64_t rs_walk_phys(const RsSegs& sg, const int64_t* s_pre, RsWalk& wk, int64_t c0,
                                                unsigned lane) {
  const int64_t i = c0 + lane;
  if (!sg.pre) return i;
  while (c0 >= wk.next) {  // uniform
    ++wk.seg;
    wk.next = wk.seg + 1 < sg.nseg ? s_pre[wk.seg + 1] : INT64_MAX;
  }
  if (i >= wk.next) return rs_phys(sg, s_pre, i);
  return static_cast<int64_t>(wk.seg) * sg.seg_cap + (i - s_pre[wk.seg]);
}

// Keys equal to `drop` leave the sort in its first pass (DROP kernels),
// which leaves the number of the others at *count; the later passes read it
// there.  count == nullptr: a plain sort.  (The reverse pairs of the kNN graph
// fill half to nine tenths of their slots: path at 1M x 12 32.8 -> 32.1 ms, at
// 10M 393 -> 387 ms.)
template <typename K>
struct RsDrop {
  int64_t* count;
  K drop;
};

// SEG: the input is read through a segment map (the first pass of a
// segmented sort); otherwise logical and physical indices agree and the
// chunk addresses are not kept in registers.
template <typename K, bool SEG, bool DROP, int WAVES, int CH>
__global__ __launch_bounds__(WAVES * 64) void k_rs_hist(const K* __restrict__ keys, int64_t n, int shift,
                                                        int32_t* __restrict__ hist, RsSegs sg, RsDrop<K> dr) {
  constexpr int kBlock = WAVES * 64;
  if (!SEG && !DROP && dr.count) n = *dr.count;  // tiles past it count nothing
  __shared__ int32_t h[kRsBins];
  __shared__ int64_t s_pre[SEG ? kRsMaxSegs + 1 : 1];
  for (int i = threadIdx.x; i < kRsBins; i += kBlock) h[i] = 0;
  if (SEG) rs_load_segs(sg, s_pre);
  __syncthreads();
  const unsigned lane = __lane_id();
  const int64_t wbase = (static_cast<int64_t>(blockIdx.x) * WAVES + (threadIdx.x >> 6)) * (64 * CH);
  // every chunk's load is issued before the first is used
  K kv[CH];
  if (SEG) {
    int64_t ph[CH];
    RsWalk wk = rs_walk_begin(sg, s_pre, wbase < n ? wbase : 0);
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int64_t c0 = wbase + c * 64;
      ph[c] = c0 + lane < n ? rs_walk_phys(sg, s_pre, wk, c0, lane) : 0;
    }
#pragma unroll
    for (int c = 0; c < CH; ++c) kv[c] = keys[ph[c]];
  } else {
    const K* kw = keys + wbase + lane;
#pragma unroll
    for (int c = 0; c < CH; ++c) kv[c] = wbase + c * 64 + lane < n ? kw[c * 64] : K(0);
  }
#pragma unroll
  for (int c = 0; c < CH; ++c)
    if (wbase + c * 64 + lane < n && !(DROP && kv[c] == dr.drop)) atomicAdd(&h[static_cast<unsigned>(kv[c] >> shift) & 0xFFu], 1);
  __syncthreads();
  // tile-major: the block's 256 counts are one contiguous 1 KB row
  for (int i = threadIdx.x; i < kRsBins; i += kBlock) hist[static_cast<int64_t>(blockIdx.x) * kRsBins + i] = h[i];
}

// Digit offsets from the tile-major counts H[t][d] (ntiles x 256): tiles are
// taken in ranges; H[t][d] is replaced by the sum over the earlier tiles of
// its range (32 bits), base[b][d] is the sum over the earlier ranges, tot[d]
// the digit's total.  The scatter adds the three (the digits' starts are a
// scan of tot).  Every access but the transposed writes of base is a
// contiguous row, and a tile costs 4 KB of traffic.
//
// Up to kRsColTiles tiles are one range and one launch: a block per 16
// digits (a 64-byte piece of every row), thread (r, d) takes a run of tiles
// and the runs' sums are scanned in LDS.
constexpr int64_t kRsColTiles = 2048;
constexpr int kRsColDigits = 16;

__global__ __launch_bounds__(1024) void k_rs_col_small(int32_t* __restrict__ hist, int ntiles,
                                                       int64_t* __restrict__ base, int64_t* __restrict__ tot) {
  __shared__ int32_t s_sum[64][kRsColDigits + 1];
  const int dl = static_cast<int>(threadIdx.x) & (kRsColDigits - 1);
  const int d = static_cast<int>(blockIdx.x) * kRsColDigits + dl;
  const int r = static_cast<int>(threadIdx.x) / kRsColDigits;  // run 0..63
  const int per = (ntiles + 63) / 64;
  const int t0 = r * per, t1 = t0 + per < ntiles ? t0 + per : ntiles;
  int32_t s = 0;  // 2048 tiles of at most 5120 keys fit
#pragma unroll 4
  for (int t = t0; t < t1; ++t) s += hist[t * kRsBins + d];
  s_sum[r][dl] = s;
  __syncthreads();
  // wave w scans digit w of the block: lane = run
  const int lane = static_cast<int>(__lane_id()), w = static_cast<int>(threadIdx.x >> 6);
  const int32_t v = s_sum[lane][w];
  int32_t incl = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int32_t y = __shfl_up(incl, o);
    if (lane >= o) incl += y;
  }
  s_sum[lane][w] = incl - v;
  if (lane == 63) {
    tot[blockIdx.x * kRsColDigits + w] = incl;
    base[blockIdx.x * kRsColDigits + w] = 0;
  }
  __syncthreads();
  int32_t run = s_sum[r][dl];
#pragma unroll 4
  for (int t = t0; t < t1; ++t) {
    const int32_t h = hist[t * kRsBins + d];
    hist[t * kRsBins + d] = run;
    run += h;
  }
}

// More tiles: ranges of kRsColRows.
constexpr int kRsColRows = 32;
static_assert(kRsBins == kScanBlock, "one thread per digit in the column scans");

// H of range b to running sums; Q[d][b] = the range's total of digit d.
__global__ __launch_bounds__(kRsBins) void k_rs_col_sum(int32_t* __restrict__ hist, int64_t ntiles, int64_t nrange,
                                                        int32_t* __restrict__ q) {
  const int d = static_cast<int>(threadIdx.x);
  const int64_t t0 = static_cast<int64_t>(blockIdx.x) * kRsColRows;
  int32_t h[kRsColRows];
#pragma unroll
  for (int r = 0; r < kRsColRows; ++r) h[r] = t0 + r < ntiles ? hist[(t0 + r) * kRsBins + d] : 0;
  int32_t run = 0;
#pragma unroll
  for (int r = 0; r < kRsColRows; ++r) {
    if (t0 + r < ntiles) hist[(t0 + r) * kRsBins + d] = run;
    run += h[r];
  }
  q[static_cast<int64_t>(d) * nrange + blockIdx.x] = run;
}

// One block per digit: base[.][d] = the exclusive prefix of Q[d][.] over
// ranges; tot[d] receives the digit's total.
__global__ __launch_bounds__(kScanBlock) void k_rs_col_scan(const int32_t* __restrict__ q, int64_t nrange,
                                                            int64_t* __restrict__ base, int64_t* __restrict__ tot) {
  __shared__ int64_t carry_s;
  const int32_t* row = q + static_cast<int64_t>(blockIdx.x) * nrange;
  if (threadIdx.x == 0) carry_s = 0;
  __syncthreads();
  for (int64_t start = 0; start < nrange; start += kScanBlock) {
    const int64_t idx = start + threadIdx.x;
    const int64_t v = idx < nrange ? row[idx] : 0;
    int64_t total;
    const int64_t ex = block_excl_scan(v, &total);
    const int64_t carry = carry_s;
    if (idx < nrange) base[idx * kRsBins + blockIdx.x] = carry + ex;
    __syncthreads();
    if (threadIdx.x == 0) carry_s = carry + total;
    __syncthreads();
  }
  if (threadIdx.x == 0) tot[blockIdx.x] = carry_s;
}

// Lanes of the wave whose digit equals this lane's (active lanes only).
__device__ __forceinline__ uint64_t rs_match(unsigned dg, bool act) {
  uint64_t m = __ballot(act);
#pragma unroll
  for (int b = 0; b < 8; ++b) {
    const bool bit = (dg >> b) & 1u;
    const uint64_t bal = __ballot(bit);
    m &= bit ? bal : ~bal;
  }
  return m;
}

// Stable ranks of one wave's CH chunks: rank[c] = keys of the same digit
// before this one in the wave; wcnt (the wave's 256 counters, zero on entry)
// ends as the wave's digit counts.
template <typename K, bool DROP, int CH>
__device__ __forceinline__ void rs_wave_ranks(const K (&key)[CH], int64_t wbase, int64_t n, int shift, K drop,
                                              uint16_t* wcnt, uint8_t (&dig)[CH], int32_t (&rank)[CH]) {
  const unsigned lane = __lane_id();
  const uint64_t lt = lanemask_lt();
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const bool act = wbase + c * 64 + lane < n && !(DROP && key[c] == drop);
    const unsigned dg = static_cast<unsigned>(key[c] >> shift) & 0xFFu;
    dig[c] = static_cast<uint8_t>(dg);
    const uint64_t m = rs_match(dg, act);
    // Lanes of one digit: the lowest one advances the wave's digit counter.
    const int leader = act ? __builtin_ctzll(m) : static_cast<int>(lane);
    int32_t base = 0;
    if (act && static_cast<int>(lane) == leader) {
      base = wcnt[dg];
      wcnt[dg] = static_cast<uint16_t>(base + __popcll(m));
    }
    base = __shfl(base, leader);
    rank[c] = act ? base + __popcll(m & lt) : 0;
  }
}

// Per digit (the block's first 256 threads): the waves' counts become their
// exclusive prefix in wave order; dstart[d] = the tile's start of digit d,
// dstart[256] = its keys.
// Every thread of the block calls it, after a barrier; wsum is LDS.
template <int WAVES>
__device__ __forceinline__ void rs_digit_starts(uint16_t (*wcnt)[kRsBins], int32_t* dstart, int32_t* wsum) {
  const unsigned lane = __lane_id();
  const unsigned w = threadIdx.x >> 6;
  const int dgt = static_cast<int>(threadIdx.x);
  int32_t tot = 0, incl = 0;
  if (dgt < kRsBins) {
#pragma unroll
    for (int ww = 0; ww < WAVES; ++ww) {
      const int32_t c = wcnt[ww][dgt];
      wcnt[ww][dgt] = static_cast<uint16_t>(tot);
      tot += c;
    }
    incl = tot;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int32_t y = __shfl_up(incl, o);
      if (static_cast<int>(lane) >= o) incl += y;
    }
    if (lane == 63) wsum[w] = incl;
  }
  __syncthreads();
  if (dgt < kRsBins) {
    int32_t wpre = 0;
    for (unsigned ww = 0; ww < w; ++ww) wpre += wsum[ww];
    dstart[dgt] = wpre + incl - tot;
    if (dgt == kRsBins - 1) dstart[kRsBins] = wpre + incl;
  }
  __syncthreads();
}

// Exclusive scan of tot over the 256 digits into s (first 256 threads).
__device__ __forceinline__ void rs_digit_base(const int64_t* __restrict__ tot, int64_t* s, int64_t* wsum64) {
  const unsigned lane = __lane_id();
  const unsigned w = threadIdx.x >> 6;
  int64_t v = 0, incl = 0;
  if (threadIdx.x < kRsBins) {
    v = tot[threadIdx.x];
    incl = wave_incl_scan(v);
    if (lane == 63) wsum64[w] = incl;
  }
  __syncthreads();
  if (threadIdx.x < kRsBins) {
    int64_t pre = 0;
    for (unsigned ww = 0; ww < w; ++ww) pre += wsum64[ww];
    s[threadIdx.x] = pre + incl - v;
  }
}

template <typename K, typename V, bool HAS_V, bool SEG, bool DROP, int WAVES, int CH>
__global__ __launch_bounds__(WAVES * 64) void k_rs_scatter(const K* __restrict__ kin, const V* __restrict__ vin,
                                                           K* __restrict__ kout, V* __restrict__ vout, int64_t n,
                                                           int shift, const int32_t* __restrict__ hist,
                                                           const int64_t* __restrict__ base,
                                                           const int64_t* __restrict__ tot, int range_shift, RsSegs sg,
                                                           int64_t ntiles, int64_t per, RsDrop<K> dr) {
  constexpr int kBlock = WAVES * 64;
  constexpr int kTile = kBlock * CH;
  // Workgroups go to the eight XCDs in turn, so blocks b, b + 8, b + 16, ...
  // share an L2: they take consecutive tiles (per of them for each XCD), and
  // the runs consecutive tiles write for a digit, which continue each other
  // in memory, fill their common cache lines in one L2.
  const int64_t tile = (static_cast<int64_t>(blockIdx.x) & 7) * per + (blockIdx.x >> 3);
  if (tile >= ntiles) return;  // uniform across the block
  if (!SEG && !DROP && dr.count) {
    n = *dr.count;
    if (tile * kTile >= n) return;
  }
  static_assert(kBlock >= kRsBins, "one thread per digit");
  static_assert(kTile <= 65535, "tile counts fit 16 bits");
  __shared__ uint16_t wcnt[WAVES][kRsBins];
  __shared__ int64_t goff[kRsBins];  // global position of the tile's first key of a digit, less its tile start
  __shared__ int32_t dstart[kRsBins + 1];
  __shared__ int32_t wsum[4];
  __shared__ int64_t wsum64[4];
  __shared__ int64_t s_pre[SEG ? kRsMaxSegs + 1 : 1];
  // staging: keys first, then values, through one buffer
  __shared__ uint64_t s_stage[kTile * (sizeof(K) > sizeof(V) || !HAS_V ? sizeof(K) : sizeof(V)) / 8];
  K* skey = reinterpret_cast<K*>(s_stage);
  V* sval = reinterpret_cast<V*>(s_stage);
  const unsigned lane = __lane_id();
  const unsigned w = threadIdx.x >> 6;
  for (int i = threadIdx.x; i < WAVES * kRsBins / 2; i += kBlock) reinterpret_cast<uint32_t*>(&wcnt[0][0])[i] = 0;
  if (SEG) rs_load_segs(sg, s_pre);
  rs_digit_base(tot, goff, wsum64);
  if (DROP && tile == 0 && threadIdx.x == kRsBins - 1) *dr.count = goff[kRsBins - 1] + tot[kRsBins - 1];
  if (threadIdx.x < kRsBins)
    goff[threadIdx.x] += base[(tile >> range_shift) * kRsBins + threadIdx.x] + hist[tile * kRsBins + threadIdx.x];
  __syncthreads();
  const int64_t wbase = (tile * WAVES + w) * (64 * CH);
  K key[CH];
  V val[CH];
  int32_t rank[CH];
  uint8_t dig[CH];
  // addresses first, then every chunk's loads back to back (no branch
  // between them), so their latencies overlap
  if (SEG) {
    int64_t ph[CH];
    RsWalk wk = rs_walk_begin(sg, s_pre, wbase < n ? wbase : 0);
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int64_t c0 = wbase + c * 64;
      ph[c] = c0 + lane < n ? rs_walk_phys(sg, s_pre, wk, c0, lane) : 0;
    }
#pragma unroll
    for (int c = 0; c < CH; ++c) key[c] = kin[ph[c]];
    if (HAS_V) {
#pragma unroll
      for (int c = 0; c < CH; ++c) val[c] = vin[ph[c]];
    }
  } else {
    // past n a lane reloads key n - 1 (never used); that also holds for a
    // wave that starts past n (the last tile's later waves), whose loads
    // would otherwise run past the end of the input
    const int64_t last = n - 1 - wbase;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int64_t o = c * 64 + lane;
      key[c] = kin[wbase + (o <= last ? o : last)];
    }
    if (HAS_V) {
#pragma unroll
      for (int c = 0; c < CH; ++c) {
        const int64_t o = c * 64 + lane;
        val[c] = vin[wbase + (o <= last ? o : last)];
      }
    }
  }
  rs_wave_ranks<K, DROP, CH>(key, wbase, n, shift, dr.drop, wcnt[w], dig, rank);
  __syncthreads();
  rs_digit_starts<WAVES>(wcnt, dstart, wsum);
  if (threadIdx.x < kRsBins) goff[threadIdx.x] -= dstart[threadIdx.x];
  // Stage the tile in LDS in digit order (keys, then values, through one
  // buffer) and write each digit's run to consecutive global positions.
  int32_t lp[CH];
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int64_t idx = wbase + c * 64 + lane;
    lp[c] = idx < n && !(DROP && key[c] == dr.drop) ? dstart[dig[c]] + wcnt[w][dig[c]] + rank[c] : -1;
    if (lp[c] >= 0) skey[lp[c]] = key[c];
  }
  __syncthreads();
  const int32_t cnt = dstart[kRsBins];
  // each thread keeps the digits of the staged positions it writes
  // (threadIdx.x + kBlock t), for the values' pass
  uint8_t dpos[CH];
#pragma unroll
  for (int t = 0; t < CH; ++t) {
    const int32_t i = static_cast<int32_t>(threadIdx.x) + t * kBlock;
    dpos[t] = 0;
    if (i < cnt) {
      const K k = skey[i];
      const unsigned dd = static_cast<unsigned>(k >> shift) & 0xFFu;
      kout[goff[dd] + i] = k;
      dpos[t] = static_cast<uint8_t>(dd);
    }
  }
  if (HAS_V) {
    __syncthreads();
#pragma unroll
    for (int c = 0; c < CH; ++c)
      if (lp[c] >= 0) sval[lp[c]] = val[c];
    __syncthreads();
#pragma unroll
    for (int t = 0; t < CH; ++t) {
      const int32_t i = static_cast<int32_t>(threadIdx.x) + t * kBlock;
      if (i < cnt) vout[goff[dpos[t]] + i] = sval[i];
    }
  }
}

// Up to kRsOne keys: every pass in one block and one launch, the keys and
// values in registers and reordered through LDS (a pass in three launches
// costs 10 us at any such size).
constexpr int kRsOneWaves = 16, kRsOneCh = 8;
constexpr int64_t kRsOne = kRsOneWaves * 64 * kRsOneCh;

template <typename K, typename V, bool HAS_V>
__global__ __launch_bounds__(kRsOneWaves * 64) void k_rs_one(K* __restrict__ keys, V* __restrict__ vals, int n,
                                                             int bit0, int bit1) {
  constexpr int CH = kRsOneCh;
  __shared__ uint16_t wcnt[kRsOneWaves][kRsBins];
  __shared__ int32_t dstart[kRsBins + 1];
  __shared__ int32_t wsum[4];
  __shared__ uint64_t s_stage[kRsOne * (sizeof(K) > sizeof(V) || !HAS_V ? sizeof(K) : sizeof(V)) / 8];
  K* skey = reinterpret_cast<K*>(s_stage);
  V* sval = reinterpret_cast<V*>(s_stage);
  const int lane = static_cast<int>(__lane_id());
  const unsigned w = threadIdx.x >> 6;
  const int wbase = static_cast<int>(w) * 64 * CH;
  K key[CH];
  V val[CH];
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int i = wbase + c * 64 + lane;
    key[c] = i < n ? keys[i] : K(0);
    if (HAS_V) val[c] = i < n ? vals[i] : V(0);
  }
  for (int shift = bit0; shift < bit1; shift += 8) {
    for (int i = threadIdx.x; i < kRsOneWaves * kRsBins / 2; i += kRsOneWaves * 64)
      reinterpret_cast<uint32_t*>(&wcnt[0][0])[i] = 0;
    __syncthreads();
    uint8_t dig[CH];
    int32_t rank[CH];
    rs_wave_ranks<K, false, CH>(key, wbase, n, shift, K(0), wcnt[w], dig, rank);
    __syncthreads();
    rs_digit_starts<kRsOneWaves>(wcnt, dstart, wsum);
    int32_t lp[CH];
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      lp[c] = wbase + c * 64 + lane < n ? dstart[dig[c]] + wcnt[w][dig[c]] + rank[c] : -1;
      if (lp[c] >= 0) skey[lp[c]] = key[c];
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < CH; ++c)
      if (wbase + c * 64 + lane < n) key[c] = skey[wbase + c * 64 + lane];
    if (HAS_V) {
      __syncthreads();
#pragma unroll
      for (int c = 0; c < CH; ++c)
        if (lp[c] >= 0) sval[lp[c]] = val[c];
      __syncthreads();
#pragma unroll
      for (int c = 0; c < CH; ++c)
        if (wbase + c * 64 + lane < n) val[c] = sval[wbase + c * 64 + lane];
    }
    __syncthreads();
  }
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int i = wbase + c * 64 + lane;
    if (i < n) {
      keys[i] = key[c];
      if (HAS_V) vals[i] = val[c];
    }
  }
}

// Scratch of one pass: tile counts, range bases, digit totals, range totals.
struct RsWork {
  int32_t* hist;
  int64_t *base, *tot;
  int32_t* q;
};

// One pass (digit at `shift`) from (ka, va) to (kb, vb).
template <typename K, typename V, bool HAS_V, int WAVES, int CH>
static int radix_pass(hdb_ctx* ctx, const K* ka, const V* va, K* kb, V* vb, int64_t n, int shift, const RsSegs& sp,
                      const RsDrop<K>& dr, bool first, const RsWork& wk) {
  constexpr int kTile = WAVES * 64 * CH;
  const int64_t ntiles = (n + kTile - 1) / kTile;
  const dim3 grid(static_cast<unsigned>(ntiles)), block(WAVES * 64);
  constexpr bool kDrops = HAS_V && sizeof(K) == 4 && sizeof(V) == 4;  // the one sort that drops keys
  if (sp.pre)
    hipLaunchKernelGGL((k_rs_hist<K, true, false, WAVES, CH>), grid, block, 0, ctx->stream, ka, n, shift, wk.hist, sp,
                       dr);
  else if (kDrops && dr.count && first)
    hipLaunchKernelGGL((k_rs_hist<K, false, kDrops, WAVES, CH>), grid, block, 0, ctx->stream, ka, n, shift, wk.hist,
                       sp, dr);
  else
    hipLaunchKernelGGL((k_rs_hist<K, false, false, WAVES, CH>), grid, block, 0, ctx->stream, ka, n, shift, wk.hist,
                       sp, dr);
  HDB_LAUNCHED();
  int range_shift = 62;  // one range
  if (ntiles <= kRsColTiles) {
    hipLaunchKernelGGL(k_rs_col_small, dim3(kRsBins / kRsColDigits), dim3(1024), 0, ctx->stream, wk.hist,
                       static_cast<int>(ntiles), wk.base, wk.tot);
    HDB_LAUNCHED();
  } else {
    static_assert(kRsColRows == 32, "range_shift");
    range_shift = 5;
    const int64_t nrange = (ntiles + kRsColRows - 1) / kRsColRows;
    hipLaunchKernelGGL(k_rs_col_sum, dim3(nrange), dim3(kRsBins), 0, ctx->stream, wk.hist, ntiles, nrange, wk.q);
    HDB_LAUNCHED();
    hipLaunchKernelGGL(k_rs_col_scan, dim3(kRsBins), dim3(kScanBlock), 0, ctx->stream, wk.q, nrange, wk.base, wk.tot);
    HDB_LAUNCHED();
  }
  const int64_t per = (ntiles + 7) / 8;  // tiles per XCD
  const dim3 sgrid(static_cast<unsigned>(8 * per));
  if (sp.pre)
    hipLaunchKernelGGL((k_rs_scatter<K, V, HAS_V, true, false, WAVES, CH>), sgrid, block, 0, ctx->stream, ka, va, kb,
                       vb, n, shift, wk.hist, wk.base, wk.tot, range_shift, sp, ntiles, per, dr);
  else if (kDrops && dr.count && first)
    hipLaunchKernelGGL((k_rs_scatter<K, V, HAS_V, false, kDrops, WAVES, CH>), sgrid, block, 0, ctx->stream, ka, va,
                       kb, vb, n, shift, wk.hist, wk.base, wk.tot, range_shift, sp, ntiles, per, dr);
  else
    hipLaunchKernelGGL((k_rs_scatter<K, V, HAS_V, false, false, WAVES, CH>), sgrid, block, 0, ctx->stream, ka, va, kb,
                       vb, n, shift, wk.hist, wk.base, wk.tot, range_shift, sp, ntiles, per, dr);
  HDB_LAUNCHED();
  return HDB_OK;
}

// LSD radix sort of (keys, vals) by bits [bit0, bit1).  seg != nullptr: the
// input is read through that segment map (see RsSegs).  kout == nullptr: the
// result ends in keys/vals; otherwise *kout/*vout receive the buffers that
// hold it (keys/vals or the sort's own scratch), which saves a copy.
// drop != nullptr (u32 keys and values only): keys equal to *drop, which sort
// last, are left out; *count receives a device pointer to the number of the
// others, in the sort's scratch (valid until the next sort), or nullptr where
// they were kept.
template <typename K, typename V, bool HAS_V>
static int radix_sort_t(hdb_ctx* ctx, K* keys, V* vals, int64_t n, int bit0, int bit1, const RsSegs* seg,
                        K** kout, V** vout, const K* drop = nullptr, const int64_t** count = nullptr) {
  RsSegs sg{nullptr, 0, 0};
  if (seg) {
    if (seg->nseg < 1 || seg->nseg > kRsMaxSegs) return ctx->fail(HDB_EINVAL, "bad segment map");
    sg = *seg;
    if (bit1 < bit0 + 8) bit1 = bit0 + 8;  // at least one pass gathers the segments
  }
  if (n <= 1 && !seg) bit1 = bit0;
  if (kout) *kout = keys;
  if (vout) *vout = vals;
  if (count) *count = nullptr;
  if (n <= 0 || bit1 <= bit0) return HDB_OK;
  if (!seg && n <= kRsOne) {
    hipLaunchKernelGGL((k_rs_one<K, V, HAS_V>), dim3(1), dim3(kRsOneWaves * 64), 0, ctx->stream, keys, vals,
                       static_cast<int>(n), bit0, bit1);
    HDB_LAUNCHED();
    return HDB_OK;
  }
  // Blocks of 8 waves; tiles of 4096 keys, of 5120 with u64 values, which
  // leave three or four blocks to a CU's LDS.  With the XCD-aware tile order
  // runs of that length fill their cache lines: a pass over 320M u32 keys
  // with u32 / u64 values takes 1.54 / 2.10 ms (4.2 / 4.3 TB/s; tiles of 8192
  // from 4 waves in plain order 2.16 / 3.43, of 8192 from 16 waves 2.03 /
  // 2.28, of 16384 1.77 / 3.04).  Up to kRsSmallKeys tiles of 2048, which
  // spread few keys over more CUs (160k keys: 11.5 / 11.8 us against 13.5 /
  // 14.4 with 4096; at 600k 15.0 / 15.4 against 15.0 / 16.1).
  constexpr int kCh = sizeof(V) == 8 && HAS_V ? 10 : 8;
  constexpr int64_t kTile = 8 * 64 * kCh;
  const bool small = n <= kRsSmallKeys;
  const int64_t ntiles = small ? (n + 2047) / 2048 : (n + kTile - 1) / kTile;
  K* k2;
  V* v2 = nullptr;
  RsWork wk;
  HDB_CALL(scratch_t(ctx, kSlotSortKeys, static_cast<size_t>(n), &k2));
  if (HAS_V) HDB_CALL(scratch_t(ctx, kSlotSortVals, static_cast<size_t>(n), &v2));
  HDB_CALL(scratch_t(ctx, kSlotSortHist, static_cast<size_t>(kRsBins * ntiles), &wk.hist));
  const int64_t nrange = (ntiles + kRsColRows - 1) / kRsColRows;
  HDB_CALL(scratch_t(ctx, kSlotSortAux, static_cast<size_t>(kRsBins * (1 + nrange + (nrange + 1) / 2) + 1), &wk.tot));
  wk.base = wk.tot + kRsBins;
  wk.q = reinterpret_cast<int32_t*>(wk.base + kRsBins * nrange);
  // the count of a sort that drops keys follows the range totals
  const RsDrop<K> dr{drop ? wk.tot + kRsBins * (1 + nrange + (nrange + 1) / 2) : nullptr, drop ? *drop : K(0)};
  if (count) *count = dr.count;
  K* ka = keys;
  K* kb = k2;
  V* va = vals;
  V* vb = v2;
  int passes = 0;
  for (int shift = bit0; shift < bit1; shift += 8, ++passes) {
    const RsSegs sp = passes == 0 ? sg : RsSegs{nullptr, 0, 0};
    if (small)
      HDB_CALL((radix_pass<K, V, HAS_V, 8, 4>(ctx, ka, va, kb, vb, n, shift, sp, dr, passes == 0, wk)));
    else
      HDB_CALL((radix_pass<K, V, HAS_V, 8, kCh>(ctx, ka, va, kb, vb, n, shift, sp, dr, passes == 0, wk)));
    std::swap(ka, kb);
    std::swap(va, vb);
  }
  if (kout) {
    *kout = ka;
    if (vout) *vout = va;
    return HDB_OK;
  }
  if (passes & 1) {
    HDB_HIP(hipMemcpyAsync(keys, ka, static_cast<size_t>(n) * sizeof(K), hipMemcpyDeviceToDevice, ctx->stream));
    if (HAS_V) HDB_HIP(hipMemcpyAsync(vals, va, static_cast<size_t>(n) * sizeof(V), hipMemcpyDeviceToDevice, ctx->stream));
  }
  return HDB_OK;
}

int radix_sort_u32_u64(hdb_ctx* ctx, uint32_t* keys, uint64_t* vals, int64_t n, int bit0, int bit1) {
  return radix_sort_t<uint32_t, uint64_t, true>(ctx, keys, vals, n, bit0, bit1, nullptr, nullptr, nullptr);
}
int radix_sort_u64_u32(hdb_ctx* ctx, uint64_t* keys, uint32_t* vals, int64_t n, int bit0, int bit1) {
  return radix_sort_t<uint64_t, uint32_t, true>(ctx, keys, vals, n, bit0, bit1, nullptr, nullptr, nullptr);
}
int radix_sort_u64(hdb_ctx* ctx, uint64_t* keys, int64_t n, int bit0, int bit1) {
  return radix_sort_t<uint64_t, uint64_t, false>(ctx, keys, static_cast<uint64_t*>(nullptr), n, bit0, bit1, nullptr,
                                                 nullptr, nullptr);
}
int radix_sort_u32_u64_segs(hdb_ctx* ctx, uint32_t* keys, uint64_t* vals, int64_t n, const int64_t* seg_pre,
                            int nseg, int64_t seg_cap, int bit0, int bit1, uint32_t** kout, uint64_t** vout) {
  const RsSegs sg{seg_pre, nseg, seg_cap};
  return radix_sort_t<uint32_t, uint64_t, true>(ctx, keys, vals, n, bit0, bit1, &sg, kout, vout);
}
int radix_sort_u32_u32_out(hdb_ctx* ctx, uint32_t* keys, uint32_t* vals, int64_t n, int bit0, int bit1,
                           uint32_t** kout, uint32_t** vout) {
  return radix_sort_t<uint32_t, uint32_t, true>(ctx, keys, vals, n, bit0, bit1, nullptr, kout, vout);
}
int radix_sort_u32_u32_drop(hdb_ctx* ctx, uint32_t* keys, uint32_t* vals, int64_t n, int bit0, int bit1, uint32_t drop,
                            uint32_t** kout, uint32_t** vout, const int64_t** count) {
  return radix_sort_t<uint32_t, uint32_t, true>(ctx, keys, vals, n, bit0, bit1, nullptr, kout, vout, &drop, count);
}

}  // namespace hdb

namespace hdb {

// -------------------------------------------------------- segment bounds --
template <typename P>
__global__ void k_seg_bounds(const uint32_t* __restrict__ keys, int64_t m, int64_t nseg, int shift,
                             P* __restrict__ s, P* __restrict__ e, const int64_t* __restrict__ count) {
  if (count) m = *count;
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= m) return;
  const uint32_t k = keys[i] >> shift;
  if (static_cast<int64_t>(k) >= nseg) return;
  if (i == 0 || (keys[i - 1] >> shift) != k) s[k] = static_cast<P>(i);
  if (i == m - 1 || (keys[i + 1] >> shift) != k) e[k] = static_cast<P>(i + 1);
}

// Four keys per lane from one 16-byte load; the neighbours across lanes
// come by shuffle, and only the wave's first and last lanes read the keys
// just outside their four.  keys must be 16-byte aligned.
template <typename P>
__global__ void k_seg_bounds4(const uint32_t* __restrict__ keys, int64_t m, int64_t nseg, int shift,
                              P* __restrict__ s, P* __restrict__ e, const int64_t* __restrict__ count) {
  if (count) m = *count;
  const int64_t i0 = (static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x) * 4;
  const unsigned lane = __lane_id();
  uint32_t k[4];
  if (i0 + 3 < m) {
    const uint4 v = *reinterpret_cast<const uint4*>(keys + i0);
    k[0] = v.x, k[1] = v.y, k[2] = v.z, k[3] = v.w;
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j) k[j] = i0 + j < m ? keys[i0 + j] : 0u;
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) k[j] >>= shift;
  uint32_t prev = __shfl_up(k[3], 1);
  uint32_t next = __shfl_down(k[0], 1);
  if (lane == 0 && i0 > 0 && i0 - 1 < m) prev = keys[i0 - 1] >> shift;
  if (lane == 63 && i0 + 4 < m) next = keys[i0 + 4] >> shift;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int64_t i = i0 + j;
    if (i >= m || static_cast<int64_t>(k[j]) >= nseg) continue;
    const uint32_t before = j == 0 ? prev : k[j - 1];
    const uint32_t after = j == 3 ? next : k[j + 1];
    if (i == 0 || before != k[j]) s[k[j]] = static_cast<P>(i);
    if (i == m - 1 || after != k[j]) e[k[j]] = static_cast<P>(i + 1);
  }
}

template <typename P>
static int segment_bounds_t(hdb_ctx* ctx, const uint32_t* keys, int64_t m, int64_t nseg, P* s, P* e, int shift,
                            const int64_t* count) {
  if (sizeof(P) == 4 && m > INT32_MAX) return ctx->fail(HDB_EUNSUPPORTED, "int32 segment bounds past 2^31 keys");
  if (sizeof(P) == 8) {
    HDB_CALL(fill_u64(ctx, reinterpret_cast<uint64_t*>(s), nseg, 0));
    HDB_CALL(fill_u64(ctx, reinterpret_cast<uint64_t*>(e), nseg, 0));
  } else {
    HDB_CALL(fill_i32(ctx, reinterpret_cast<int32_t*>(s), nseg, 0));
    HDB_CALL(fill_i32(ctx, reinterpret_cast<int32_t*>(e), nseg, 0));
  }
  if (m <= 0) return HDB_OK;
  if ((reinterpret_cast<uintptr_t>(keys) & 15) == 0)
    hipLaunchKernelGGL(k_seg_bounds4<P>, dim3(grid_for((m + 3) / 4, 256)), dim3(256), 0, ctx->stream, keys, m, nseg,
                       shift, s, e, count);
  else
    hipLaunchKernelGGL(k_seg_bounds<P>, dim3(grid_for(m, 256)), dim3(256), 0, ctx->stream, keys, m, nseg, shift, s,
                       e, count);
  HDB_LAUNCHED();
  return HDB_OK;
}

int segment_bounds(hdb_ctx* ctx, const uint32_t* keys, int64_t m, int64_t nseg, int32_t* s, int32_t* e, int shift,
                   const int64_t* count) {
  return segment_bounds_t(ctx, keys, m, nseg, s, e, shift, count);
}
int segment_bounds(hdb_ctx* ctx, const uint32_t* keys, int64_t m, int64_t nseg, int64_t* s, int64_t* e, int shift) {
  return segment_bounds_t(ctx, keys, m, nseg, s, e, shift, nullptr);
}

int bits_for(int64_t max_key) {
  int b = 0;
  while (b < 63 && (static_cast<int64_t>(1) << b) <= max_key) ++b;
  return b;
}

}  // namespace hdb
