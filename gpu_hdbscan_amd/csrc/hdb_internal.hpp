// Internal declarations shared by the gfx950 translation units of
// libhdbscan_mi355x.so: the context, scratch arena, stage timer, error
// plumbing, wave64 helpers and the launch wrappers of each kernel family.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <map>
#include <string>
#include <vector>

#include "../../include/hdbscan_mi355x.h"

namespace hdb {

constexpr int kK = 32;                       // NEIGHB_NUM_PER_LIST
constexpr uint32_t kInvalidId = 0x7FFFFFFFu;  // empty list slot label
constexpr uint64_t kKeyMax = ~0ull;
// No-allocation entry point (hdb_sort_edges_noalloc): its scratch array
// size, the edge count it takes at most, and the devices it serves.
constexpr size_t kNoAllocBytes = static_cast<size_t>(28) << 20;
constexpr int64_t kNoAllocMaxEdges = static_cast<int64_t>(1) << 20;
constexpr int kNoAllocMaxDevices = 64;

// Scratch arena slots owned by a context (grown on demand, never shrunk).
enum Slot : int {
  kSlotFwdNew, kSlotFwdOld, kSlotRevNew, kSlotRevOld, kSlotCounts4,  // sampling
  kSlotBucket, kSlotBucketCnt, kSlotWorst, kSlotStats,                // list update
  kSlotBlockLocal, kSlotPairGraph, kSlotPairX, kSlotPairG1, kSlotPairG2,  // blocked build
  kSlotScanTmp, kSlotRowCnt, kSlotRowCursor, kSlotRowTmp, kSlotRowUniq,  // CSR build
  kSlotAhFlag, kSlotAhAux, kSlotAhKeys, kSlotAhKeys2,                 // anti-hubs
  kSlotMstParent, kSlotMstMin, kSlotMstWl1, kSlotMstWl2, kSlotMstFlag, kSlotMstCnt,
  kSlotMstSrc, kSlotMstPos, kSlotMstCw, kSlotSeedX, kSlotSeedCand, kSlotMlpPack,
  kSlotSortKeys, kSlotSortVals, kSlotSortHist, kSlotSortAux,          // radix sort
  kSlotPipeNindex, kSlotPipeNlist, kSlotPipeW, kSlotPipeAh,  // pipeline
  kSlotBfTmp, kSlotMisc0, kSlotMisc1, kSlotMisc2,
  kSlotPropTgt, kSlotPropSE, kSlotRevSE, kSlotPart,                     // sort-routed NN-Descent
  // second set of the per-table learned-init slots (keys, sort, packed
  // weights), used by the work on the context's second stream
  kSlotAlt0, kSlotAlt1, kSlotAlt2, kSlotAlt3, kSlotAlt4, kSlotAlt5, kSlotAlt6, kSlotAlt7, kSlotAlt8,
  kSlotRefineXh, kSlotRefineXl, kSlotRefineNorm, kSlotRefineCand, kSlotRefineCnt,  // BF16 refinement
  kSlotRefineOvfIds, kSlotRefineOvfD2, kSlotRefineRows, kSlotRefineThr,
  kSlotTreeAddCnt, kSlotTreeAddOff, kSlotTreeAdd,  // GPU labels: stability addends
  kSlotNndRows,  // NN-Descent: padded point rows with the list bound
  kSlotMstRows, kSlotMstCur,  // Boruvka: weight-sorted rows and their cursors
  kSlotGatherFlag,  // hdb_gather_rows: bad-row flag
  kSlotCount
};

struct TimerAcc {
  double ms = 0.0;
  int64_t launches = 0;
};

struct PendingEvent {
  std::string name;
  hipEvent_t a, b;
};

}  // namespace hdb

struct hdb_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  std::string err;
  void* slot_ptr[hdb::kSlotCount] = {};
  size_t slot_bytes[hdb::kSlotCount] = {};
  bool timing = false;
  std::vector<hdb::PendingEvent> pending;
  std::map<std::string, hdb::TimerAcc> timers;
  std::vector<std::string> timer_names;  // stable storage for hdb_timer_read
  int64_t stats_host[4] = {0, 0, 0, 0};
  // last refinement: survivors in its first round, points past the cap in
  // that round, points left to the exact brute force after every round
  int64_t refine_stats[3] = {0, 0, 0};
  // Pinned host words and events for readbacks that overlap later work.
  int64_t* pinned = nullptr;  // kPinnedWords, from hipHostMalloc
  hipEvent_t ready[2] = {nullptr, nullptr};
  // A second stream (default priority) for independent work inside one call;
  // every call joins it back into `stream` before returning.
  hipStream_t stream2 = nullptr;
  hipEvent_t fork_ev = nullptr, join_ev = nullptr;
  // Pipeline CSR (kept when requested, for tests).
  int64_t csr_edges = 0;
  // This device's copy of the no-allocation scratch array (noalloc.hip),
  // resolved at context creation; null when unavailable.
  void* noalloc_base = nullptr;
  // Fixed-arena mode (set only inside a no-allocation entry point): scratch()
  // carves each slot from [fixed_base, fixed_base + fixed_bytes) and never
  // calls hipMalloc.
  unsigned char* fixed_base = nullptr;
  size_t fixed_bytes = 0, fixed_used = 0;
  void* fixed_slot_ptr[hdb::kSlotCount] = {};
  size_t fixed_slot_bytes[hdb::kSlotCount] = {};

  int fail(int code, const std::string& msg) {
    err = msg;
    return code;
  }
};

namespace hdb {

int hip_fail(hdb_ctx* ctx, hipError_t e, const char* what, const char* file, int line);

#define HDB_HIP(expr)                                                    \
  do {                                                                   \
    hipError_t e_ = (expr);                                              \
    if (e_ != hipSuccess) return hdb::hip_fail(ctx, e_, #expr, __FILE__, __LINE__); \
  } while (0)

#define HDB_LAUNCHED()                                                   \
  do {                                                                   \
    hipError_t e_ = hipGetLastError();                                   \
    if (e_ != hipSuccess) return hdb::hip_fail(ctx, e_, "kernel launch", __FILE__, __LINE__); \
  } while (0)

#define HDB_CALL(expr)             \
  do {                             \
    int s_ = (expr);               \
    if (s_ != HDB_OK) return s_;   \
  } while (0)

// Scratch buffer of at least `bytes` for `slot`; contents are undefined.
int scratch(hdb_ctx* ctx, Slot slot, size_t bytes, void** out);
// Exchange two slots' buffers (e.g. to keep a sort's output where its
// input lived, without a copy).
void scratch_swap(hdb_ctx* ctx, Slot a, Slot b);
template <typename T>
inline int scratch_t(hdb_ctx* ctx, Slot slot, size_t count, T** out) {
  return scratch(ctx, slot, count * sizeof(T), reinterpret_cast<void**>(out));
}
// Device address of this device's no-allocation scratch array (the device
// must be current); resolved with hipGetSymbolAddress once per device.
int noalloc_scratch(int device, void** out);
// While alive: the context's scratch slots come from [base, base + bytes)
// (fixed-arena mode, no hipMalloc) and the stage timer is off (it creates
// events).
struct FixedArena {
  hdb_ctx* ctx;
  bool timing;
  FixedArena(hdb_ctx* c, void* base, size_t bytes);
  ~FixedArena();
};

// Stage timer: records a HIP event pair around the enclosed launches.
struct Stage {
  hdb_ctx* ctx;
  PendingEvent ev;
  bool on;
  Stage(hdb_ctx* c, const char* name);
  ~Stage();
};

inline unsigned grid_for(int64_t threads, int block) {
  return static_cast<unsigned>((threads + block - 1) / block);
}

// ---- device helpers ------------------------------------------------------

// xorshift64* as used by the reference init (gpuknn/knncuda_tools.cu:126-132):
// Vigna's xorshift64* step applied to (x + 42).
__host__ __device__ inline uint64_t xorshift64star(uint64_t x) {
  x += 42ull;
  x ^= x >> 12;
  x ^= x << 25;
  x ^= x >> 27;
  return x * 0x2545F4914F6CDD1Dull;
}

// Bits of max(x, 0) for a ranking key: a negative float (sign bit set) is a
// negative int, so one integer max clamps it, -0 included, to +0.
__device__ __forceinline__ uint32_t nonneg_bits(float x) {
  const int32_t b = __float_as_int(x);
  return static_cast<uint32_t>(b > 0 ? b : 0);
}

// top[j] = median of (lo, key, top[j]) in place, in one instruction.
__device__ __forceinline__ void med3_into_u32(uint32_t& top_j, uint32_t lo, uint32_t key) {
  asm("v_med3_u32 %0, %1, %2, %0" : "+v"(top_j) : "v"(lo), "v"(key));
}

// Insert key into the ascending list top[0..K) and drop the largest: slot 0
// takes min(top[0], key) and slot j the median of top[j-1], key and top[j]
// (the key clamped to [top[j-1], top[j]]).  Slots are rewritten from the
// last down, so each reads the old top[j-1], and each result stays in its
// own register (no copies in a rolled loop).
template <int K>
__device__ __forceinline__ void top_insert_med3(uint32_t (&top)[K], uint32_t key) {
#pragma unroll
  for (int j = K - 1; j >= 1; --j) med3_into_u32(top[j], top[j - 1], key);
  top[0] = top[0] < key ? top[0] : key;
}

// Squared L2 distance in FP32, accumulated in dimension order with fused
// multiply-add.  Every distance of the kNN path goes through this one
// formula, so the same pair always yields the same bits (the oracle uses the
// identical formula with C fmaf).
__device__ __forceinline__ float d2_any(const float* __restrict__ a, const float* __restrict__ b, int d) {
  float acc = 0.0f;
  for (int k = 0; k < d; ++k) {
    float diff = a[k] - b[k];
    acc = __builtin_fmaf(diff, diff, acc);
  }
  return acc;
}

// d2_any over 16-byte aligned rows with d % 4 == 0, read as float4: the
// accumulation order is the same, so the bits are too.
__device__ __forceinline__ float d2_vec4(const float* __restrict__ a, const float* __restrict__ b, int d) {
  float acc = 0.0f;
  for (int k = 0; k < d; k += 4) {
    const float4 x = *reinterpret_cast<const float4*>(a + k);
    const float4 y = *reinterpret_cast<const float4*>(b + k);
    float diff = x.x - y.x;
    acc = __builtin_fmaf(diff, diff, acc);
    diff = x.y - y.y;
    acc = __builtin_fmaf(diff, diff, acc);
    diff = x.z - y.z;
    acc = __builtin_fmaf(diff, diff, acc);
    diff = x.w - y.w;
    acc = __builtin_fmaf(diff, diff, acc);
  }
  return acc;
}

// Euclidean distance accumulated in FP64, rounded once: diff = a - b and
// acc = acc + diff * diff with the product rounded before the add (no fused
// multiply-add, as the oracle's C with -ffp-contract=off).  Loads are issued
// four dimensions at a time ahead of the arithmetic.
__device__ __forceinline__ float dist_fp64(const float* __restrict__ a, const float* __restrict__ b, int d) {
#pragma clang fp contract(off)
  double acc = 0.0;
  int k = 0;
  for (; k + 4 <= d; k += 4) {
    float x[4], y[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      x[t] = a[k + t];
      y[t] = b[k + t];
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const double diff = static_cast<double>(x[t]) - static_cast<double>(y[t]);
      acc = acc + diff * diff;
    }
  }
  for (; k < d; ++k) {
    const double diff = static_cast<double>(a[k]) - static_cast<double>(b[k]);
    acc = acc + diff * diff;
  }
  return static_cast<float>(__dsqrt_rn(acc));
}

// List key: (squared distance bits, id, new flag).  Non-negative floats order
// like their bit patterns, so an unsigned compare orders by distance, then
// id, then old-before-new.
__device__ __forceinline__ uint64_t make_key(float d2, uint32_t id, uint32_t is_new) {
  return (static_cast<uint64_t>(__float_as_uint(d2)) << 32) | (static_cast<uint64_t>(id) << 1) | is_new;
}
__device__ __forceinline__ float key_d2(uint64_t k) { return __uint_as_float(static_cast<uint32_t>(k >> 32)); }
__device__ __forceinline__ uint32_t key_id(uint64_t k) { return static_cast<uint32_t>(k) >> 1; }
__device__ __forceinline__ uint32_t key_new(uint64_t k) { return static_cast<uint32_t>(k) & 1u; }

__device__ __forceinline__ uint32_t label_id(int32_t label) {
  return label >= 0 ? static_cast<uint32_t>(label) : static_cast<uint32_t>(-label - 1);
}

__device__ __forceinline__ uint64_t shfl_xor_u64(uint64_t v, int mask) {
  uint32_t lo = static_cast<uint32_t>(v), hi = static_cast<uint32_t>(v >> 32);
  lo = __shfl_xor(lo, mask);
  hi = __shfl_xor(hi, mask);
  return (static_cast<uint64_t>(hi) << 32) | lo;
}
__device__ __forceinline__ uint64_t shfl_u64(uint64_t v, int src) {
  uint32_t lo = static_cast<uint32_t>(v), hi = static_cast<uint32_t>(v >> 32);
  lo = __shfl(lo, src);
  hi = __shfl(hi, src);
  return (static_cast<uint64_t>(hi) << 32) | lo;
}
__device__ __forceinline__ uint64_t lanemask_lt() {
  const unsigned lane = __lane_id();
  return lane == 0 ? 0ull : (~0ull >> (64 - lane));
}

// One DPP move (a lane without a source lane gets 0).
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t v) {
  return static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(v), CTRL, 0xF, 0xF, true));
}

// The value of the lane below (lane 0: unspecified), one DPP move each word.
__device__ __forceinline__ uint32_t lane_below(uint32_t v) { return dpp_u32<0x138>(v); }  // wave_shr:1
__device__ __forceinline__ uint64_t lane_below(uint64_t v) {
  return (static_cast<uint64_t>(lane_below(static_cast<uint32_t>(v >> 32))) << 32) | lane_below(static_cast<uint32_t>(v));
}

// The value of lane (lane ^ j), for a full wave.  j = 1, 2: one DPP
// quad_perm; j = 4: half-row mirror (i <- 7 - i) then quad reversal
// (i <- 3 - i), two DPP moves; j = 8: DPP row rotation by 8; j = 16, 32:
// a swap of rows (halves) between two copies and a select.  All are ALU
// operations, free of the LDS round trip of a swizzle.
__device__ __forceinline__ uint32_t lane_xor_u32(uint32_t v, int j) {
  switch (j) {
    case 1: return dpp_u32<0xB1>(v);                  // quad_perm(1, 0, 3, 2)
    case 2: return dpp_u32<0x4E>(v);                  // quad_perm(2, 3, 0, 1)
    case 4: return dpp_u32<0x1B>(dpp_u32<0x141>(v));  // quad_perm(3, 2, 1, 0) of row_half_mirror
    case 8: return dpp_u32<0x128>(v);                 // row_ror:8
    case 16: {
      const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
      return __builtin_amdgcn_inverse_ballot_w64(0x0000FFFF0000FFFFull) ? r[1] : r[0];
    }
    default: {
      const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
      return __builtin_amdgcn_inverse_ballot_w64(0x00000000FFFFFFFFull) ? r[1] : r[0];
    }
  }
}
__device__ __forceinline__ uint64_t lane_xor_u64(uint64_t v, int j) {
  const uint32_t lo = lane_xor_u32(static_cast<uint32_t>(v), j);
  const uint32_t hi = lane_xor_u32(static_cast<uint32_t>(v >> 32), j);
  return (static_cast<uint64_t>(hi) << 32) | lo;
}

// One compare-exchange of a bitonic network: the lane keeps the smaller of
// (v, o) when want_min, else the larger, i.e. it takes o exactly when
// (o < v) == want_min -- one compare and one select.
template <typename T>
__device__ __forceinline__ T bitonic_ce(T v, T o, bool want_min) {
  return ((o < v) == want_min) ? o : v;
}

// Lanes whose index has bit j clear (j a power of two below 64).
__device__ __forceinline__ constexpr uint64_t lanes_without(int j) {
  return j == 1    ? 0x5555555555555555ull
         : j == 2  ? 0x3333333333333333ull
         : j == 4  ? 0x0F0F0F0F0F0F0F0Full
         : j == 8  ? 0x00FF00FF00FF00FFull
         : j == 16 ? 0x0000FFFF0000FFFFull
                   : 0x00000000FFFFFFFFull;
}
// Lanes that keep the smaller value in step j of stage k of a bitonic sort
// of groups of `group` lanes.
__device__ __forceinline__ constexpr uint64_t bitonic_min_lanes(int group, int k, int j) {
  return k == group ? lanes_without(j) : ~(lanes_without(j) ^ lanes_without(k));
}

// The two values of a lane pair (lane, lane ^ j), in either order.
__device__ __forceinline__ void lane_pair_u32(uint32_t v, int j, uint32_t& a, uint32_t& b) {
  if (j >= 16) {
    // rows (halves) of the two copies swapped: both lanes of a pair then
    // hold both values, without an LDS round trip
    const auto r = j == 16 ? __builtin_amdgcn_permlane16_swap(v, v, false, false)
                           : __builtin_amdgcn_permlane32_swap(v, v, false, false);
    a = r[0];
    b = r[1];
  } else {
    a = v;
    b = lane_xor_u32(v, j);
  }
}

// Bitonic sort (ascending) of one u64 per lane within aligned groups of
// GROUP lanes (GROUP = 32 or 64).
template <int GROUP>
__device__ __forceinline__ uint64_t bitonic_group(uint64_t v) {
#pragma unroll
  for (int k = 2; k <= GROUP; k <<= 1) {
#pragma unroll
    for (int j = k >> 1; j > 0; j >>= 1)
      v = bitonic_ce(v, lane_xor_u64(v, j), __builtin_amdgcn_inverse_ballot_w64(bitonic_min_lanes(GROUP, k, j)));
  }
  return v;
}
// The u32 form takes the minimum and the maximum, which read the other lane
// by DPP themselves, and one select: three instructions for most steps.
template <int GROUP>
__device__ __forceinline__ uint32_t bitonic_group_u32(uint32_t v) {
#pragma unroll
  for (int k = 2; k <= GROUP; k <<= 1) {
#pragma unroll
    for (int j = k >> 1; j > 0; j >>= 1) {
      uint32_t a, b;
      lane_pair_u32(v, j, a, b);
      const uint32_t mn = a < b ? a : b, mx = a < b ? b : a;
      v = __builtin_amdgcn_inverse_ballot_w64(bitonic_min_lanes(GROUP, k, j)) ? mn : mx;
    }
  }
  return v;
}

// Bitonic sort (ascending) of 128 u64 keys held as 2 per lane: element
// index i = r * 64 + lane for register r.
__device__ __forceinline__ void bitonic128(uint64_t& r0, uint64_t& r1) {
  const unsigned lane = __lane_id();
#pragma unroll
  for (int k = 2; k <= 128; k <<= 1) {
#pragma unroll
    for (int j = k >> 1; j > 0; j >>= 1) {
      if (j == 64) {
        // partner is the other register of the same lane; i = lane (< 64)
        // and i ^ 64 = 64 + lane; k == 128 here, so ascending.
        const uint64_t mn = r0 < r1 ? r0 : r1, mx = r0 < r1 ? r1 : r0;
        r0 = mn;
        r1 = mx;
      } else {
        const uint64_t o0 = lane_xor_u64(r0, j), o1 = lane_xor_u64(r1, j);
        const bool low = (lane & j) == 0;
        // element indices lane (r0) and 64 + lane (r1)
        const bool up0 = (k == 128) ? true : ((lane & k) == 0);
        const bool up1 = (k == 128) ? true : (((64u + lane) & k) == 0);
        r0 = bitonic_ce(r0, o0, low == up0);
        r1 = bitonic_ce(r1, o1, low == up1);
      }
    }
  }
}

// ---- kernel families (launch wrappers) -----------------------------------
// prims.hip
int fill_i32(hdb_ctx* ctx, int32_t* p, int64_t n, int32_t v);
int fill_u64(hdb_ctx* ctx, uint64_t* p, int64_t n, uint64_t v);
// Exclusive scan of n int32 counts into n+1 int64 offsets (out[n] = total).
int scan_i32_to_i64(hdb_ctx* ctx, const int32_t* in, int64_t n, int64_t* out);
// Stable LSD radix sort.  Keys u32 (bits [bit0, bit1)) with u64 payload.
int radix_sort_u32_u64(hdb_ctx* ctx, uint32_t* keys, uint64_t* vals, int64_t n, int bit0, int bit1);
// seg_start/seg_end[k] = [first, last+1) position of segment k = key >> shift
// in keys sorted by that value (k < nseg); untouched segments keep 0.
// count: a device pointer to the number of keys where the host does not know
// it (at most m), or nullptr.
int segment_bounds(hdb_ctx* ctx, const uint32_t* sorted_keys, int64_t m, int64_t nseg, int32_t* seg_start,
                   int32_t* seg_end, int shift = 0, const int64_t* count = nullptr);
// The same with int64 positions (for streams that may pass 2^31 keys).
int segment_bounds(hdb_ctx* ctx, const uint32_t* sorted_keys, int64_t m, int64_t nseg, int64_t* seg_start,
                   int64_t* seg_end, int shift = 0);
int bits_for(int64_t max_key);
// Keys-only u64 radix sort over bits [bit0, bit1).
int radix_sort_u64(hdb_ctx* ctx, uint64_t* keys, int64_t n, int bit0, int bit1);
// u64 keys with u32 payload.
int radix_sort_u64_u32(hdb_ctx* ctx, uint64_t* keys, uint32_t* vals, int64_t n, int bit0, int bit1);
// Input in nseg (<= 64) segments: logical index i in segment g (seg_pre[g] <=
// i < seg_pre[g+1], device array) is at g * seg_cap + i - seg_pre[g].  The
// sorted result is left where *kout / *vout point (the input buffers or the
// sort's scratch), so these calls make no final copy.
int radix_sort_u32_u64_segs(hdb_ctx* ctx, uint32_t* keys, uint64_t* vals, int64_t n, const int64_t* seg_pre,
                            int nseg, int64_t seg_cap, int bit0, int bit1, uint32_t** kout, uint64_t** vout);
int radix_sort_u32_u32_out(hdb_ctx* ctx, uint32_t* keys, uint32_t* vals, int64_t n, int bit0, int bit1,
                           uint32_t** kout, uint32_t** vout);
// The same without the keys equal to `drop` (past every other key): *count
// receives a device pointer to the number of the others, in the sort's
// scratch (valid until the next sort), or nullptr where all were kept.
int radix_sort_u32_u32_drop(hdb_ctx* ctx, uint32_t* keys, uint32_t* vals, int64_t n, int bit0, int bit1, uint32_t drop,
                            uint32_t** kout, uint32_t** vout, const int64_t** count);
int read_i64(hdb_ctx* ctx, const int64_t* p, int64_t* out);
// Queue a copy of *p into pinned word `slot` (0 or 1) and mark it with
// event `slot`; wait_i64 waits for that event only, so kernels queued after
// the copy keep running.
constexpr int kPinnedWords = 8;
int read_i64_async(hdb_ctx* ctx, const int64_t* p, int slot);
int wait_i64(hdb_ctx* ctx, int slot, int64_t* out);
int read_i32(hdb_ctx* ctx, const int32_t* p, int32_t* out);

// nndescent.hip
// Initial lists: xorshift ids; the caller's ids (distances recomputed,
// sorted, duplicates dropped); the caller's lists taken as they are (sorted,
// distinct, exact distances, as hdb_learned_init writes them).
enum class NndInit { kRandom, kGiven, kExact };
int nnd_run(hdb_ctx* ctx, const float* X, int64_t n, int d, const hdb_params& prm,
            hdb_nnd_element* lists, NndInit init, int iterations);
int nnd_merge_pair(hdb_ctx* ctx, const float* X, int64_t n1, int64_t n2, int d,
                   const hdb_nnd_element* g1, const hdb_nnd_element* g2, const hdb_params& prm,
                   hdb_nnd_element* out);
int nnd_blocked(hdb_ctx* ctx, const float* X, int64_t n, int d, int blocks, const hdb_params& prm,
                hdb_nnd_element* out);
// Shard boundaries of KNNDataManager (tools/knndata_manager.hpp:29-52):
// n / shards points per shard, the last shard the rest.
std::vector<int64_t> shard_offsets(int64_t n, int shards);
// UpdateKNNGraphKernel + UniqueMergeSequential (gen_large_knngraph.cu:
// 136-228): rows of `running` (global ids) merged with pair-graph rows
// row0_pair.. (ids < n_first -> off_a + id, else off_b + id - n_first).
int unique_merge(hdb_ctx* ctx, hdb_nnd_element* running, const hdb_nnd_element* pair, int64_t n_first, int64_t rows,
                 int64_t row0_pair, int64_t off_a, int64_t off_b);
int bruteforce_knn(hdb_ctx* ctx, const float* X, int64_t n, int d, const int32_t* qids, int64_t m,
                   int kq, int32_t* out_ids, float* out_d2);
// refine.hip: exact 32-NN from lists whose entry 31 bounds each point's
// 32nd distance (BF16 MFMA survivor pass, FP32 re-rank).
int refine_knng(hdb_ctx* ctx, const float* X, int64_t n, int d, hdb_nnd_element* lists, int64_t* candidates_out,
                int64_t* overflow_out);
// The same pass for m query points only (their lists give the bounds and
// are left as they are): exact kq-NN ids (and FP32 distances) per query.
int exact_knn_bounded(hdb_ctx* ctx, const float* X, int64_t n, int d, const hdb_nnd_element* lists,
                      const int32_t* qids, int64_t m, int kq, int32_t* out_ids, float* out_d2);
// Sum over the m queries of |first kq ids of lists[qids[i]] n gt[i]|.
int recall_hits(hdb_ctx* ctx, const hdb_nnd_element* lists, int64_t n, const int32_t* qids, int64_t m,
                const int32_t* gt, int kq, int64_t* hits_out);

// graph.hip
int hub_counts(hdb_ctx* ctx, const hdb_nnd_element* lists, int64_t n, int k, int32_t* counts);
int antihubs(hdb_ctx* ctx, const hdb_nnd_element* lists, const int32_t* counts, int64_t n, int k,
             int32_t* ids, int64_t* h_out);
int core_distances(hdb_ctx* ctx, const float* X, const hdb_nnd_element* lists, int64_t n, int d,
                   int k, int mpts, float* core);
// Full (symmetric) MRD CSR, rows in neighbour-id order.  nlist == nullptr:
// size query (nindex and *edges_out only).  mrd_graph = mrd_prep (reverse
// pairs sorted by row, in-degrees into counts when non-null) + mrd_rows,
// which reads the state mrd_prep left in the context's scratch.
int mrd_prep(hdb_ctx* ctx, const hdb_nnd_element* lists, int64_t n, int k, int32_t* counts);
int mrd_rows(hdb_ctx* ctx, const float* X, const hdb_nnd_element* lists, const float* core,
             const int32_t* ah, int64_t h, int64_t n, int d, int k,
             int64_t* nindex, int32_t* nlist, float* w, int64_t* edges_out);
int mrd_graph(hdb_ctx* ctx, const float* X, const hdb_nnd_element* lists, const float* core,
              const int32_t* ah, int64_t h, int64_t n, int d, int k,
              int64_t* nindex, int32_t* nlist, float* w, int64_t* edges_out);

// tree.hip
// Labels of n points from the m = n - 1 MST edges sorted by weight, with
// the semantics of the host hdb_labels; *clusters_out = selected clusters.
int labels_gpu(hdb_ctx* ctx, const hdb_mst_edge* edges, int64_t m, int64_t n, int mpts, int32_t* labels,
               int32_t* clusters_out);

// coresg.hip
// Core-SG CSR: symmetric kNN graph u the m MST edges, rows sorted by
// neighbour id, each pair once per endpoint; dist = Euclidean distance per
// entry.  nlist == nullptr: size query (nindex and *edges_out only).
int core_sg(hdb_ctx* ctx, const float* X, const hdb_nnd_element* lists, int64_t n, int d, int k,
            const hdb_mst_edge* mst, int64_t m, int64_t* nindex, int32_t* nlist, float* dist, int64_t* edges_out);
// w[e] = max(core[row], core[col], dist[e]) over a Core-SG CSR.
int core_sg_weights(hdb_ctx* ctx, const int64_t* nindex, const int32_t* nlist, const float* dist, const float* core,
                    int64_t n, float* w);

// mst.hip
// Minimum spanning forest of a full (symmetric) CSR under the order
// (weight, min id, max id); out (capacity n-1) receives the edges in CSR
// order (from < to).  Weights must not be NaN.
int mst_csr(hdb_ctx* ctx, const int64_t* nindex, const int32_t* nlist, const float* w, int64_t n,
            hdb_mst_edge* out, int64_t* m_out, int64_t* components_out);
int sort_edges(hdb_ctx* ctx, hdb_mst_edge* edges, int64_t m);

}  // namespace hdb
