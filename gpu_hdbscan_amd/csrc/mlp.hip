// Learned initialiser for NN-Descent on gfx950 (no reference counterpart: it
// replaces the random index init of InitKNNGraphIndexKernel,
// gpuknn/nndescent.cu:1673-1692, with bucket co-members).
//
// Network: d_in -> 128 -> 128 -> 12, GELU after the two hidden layers.  Every
// product runs on v_mfma_f32_16x16x32_bf16: operands (inputs, activations,
// gradients and the FP32 master weights) are rounded to BF16 when the
// fragments are formed, accumulation is FP32.  Lane layout of the
// instruction: A/B lane l holds row (l % 16), k = 8*(l/16) .. +7; the result
// lane l holds rows 4*(l/16) + q (q = 0..3), column l % 16.
//
// Training pairs: anchor a, positive = a kNN neighbour of a (from a plain
// NN-Descent graph of a subsample), negative = a random point.  With
// t = tanh(z):  L = mean_batch[ |t_a - t_p|^2 / 12 + (t_a . t_n / 12)^2 ]
//                   + sum_bits mean_rows(t)^2
// (agreeing signs for neighbours, uncorrelated codes for random pairs,
// balanced bits).  The 12 sign bits of z are the bucket code.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "hdb_internal.hpp"

namespace hdb {

constexpr int kHid = 128;
constexpr int kCode = 12;
constexpr int kOutP = 16;  // padded output width

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

struct MlpLayout {
  int kin, kinp;  // input width and its multiple of 32
  int64_t w1, b1, w2, b2, w3, b3, total;
};

static MlpLayout mlp_layout(int kin) {
  MlpLayout L;
  L.kin = kin;
  L.kinp = (kin + 31) & ~31;
  L.w1 = 0;
  L.b1 = L.w1 + static_cast<int64_t>(L.kinp) * kHid;
  L.w2 = L.b1 + kHid;
  L.b2 = L.w2 + kHid * kHid;
  L.w3 = L.b2 + kHid;
  L.b3 = L.w3 + kHid * kOutP;
  L.total = L.b3 + kOutP;
  return L;
}

// GELU in its tanh form (Hendrycks & Gimpel, "Gaussian Error Linear Units",
// 2016): gelu(x) = x s(x), s(x) = sigmoid(z), z = 2 sqrt(2 / pi) (x +
// 0.044715 x^3), which stays within 4.8e-4 of x Phi(x).  s = 1 / (1 +
// exp2(x (c0 + c1 x^2))) with c0 = -2 sqrt(2 / pi) log2(e), c1 = 0.044715 c0:
// an exp2 and a reciprocal, where the erf form needs a longer polynomial as
// well.  Large |x| saturate to s = 0 or 1 without NaN.
__device__ __forceinline__ float gelu_sig(float x) {
  const float e = __builtin_amdgcn_exp2f(x * __builtin_fmaf(x * x, -0.10294324f, -2.3022082f));
  return __builtin_amdgcn_rcpf(1.0f + e);
}
__device__ __forceinline__ float gelu(float x) { return x * gelu_sig(x); }
// d/dx x s(x) = s + x s (1 - s) z'(x), z'(x) = 2 sqrt(2 / pi) (1 + 3 * 0.044715 x^2)
__device__ __forceinline__ float gelu_grad(float x) {
  const float s = gelu_sig(x);
  return __builtin_fmaf(x * s * (1.0f - s), __builtin_fmaf(x * x, 0.21406445f, 1.5957692f), s);
}

__device__ __forceinline__ f32x4 mfma(const bf16x8& a, const bf16x8& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// ------------------------------------------------------------ training --
// One Adam step of up to kMaxTables networks is six launches, each over
// every table (blockIdx.y, or .z for the products):
//   k_tr_fwd    triples (or the caller's rows) -> forward pass per 16-row
//               tile: Z, P1 and P2 (FP32, row-major) for the backward pass,
//               the BF16 operands of the weight-gradient products (X rows,
//               H1, H2) and per-tile sums of tanh(Z) for the balance term
//   k_tr_tmean  those sums -> the mean of tanh(Z) per bit (one block)
//   k_tr_bwd    loss and dZ per row (its partner rows' Z read back), then
//               dP2 = (dZ W3^T) * gelu'(P2) and dP1 = (dP2 W2^T) * gelu'(P1);
//               BF16 operands dZ, dP2, dP1 and per-tile bias and loss sums
//   k_tr_wgrad  dW1 = X^T dP1, dW2 = H1^T dP2, dW3 = H2^T dZ split over row
//               ranges; each wave one 32 x 32 output region, its fragments
//               loaded straight from HBM
//   k_tr_bred   per-tile bias sums -> bias gradients (a wave per column)
//   k_tr_apply  the partial sums in a fixed order -> gradient -> Adam
// Every reduction has a fixed order, so a step is deterministic.
// Every product takes the BF16 roundings of its FP32 operands and
// accumulates in FP32.  BF16 operands are stored blocked and transposed:
// element (r, c) of an Rp x C matrix sits at ((r >> 5) * C + c) * 32 +
// (r & 31) (Rp = rows rounded up to 32, padding rows zero), so the 8
// consecutive rows of one column that form a lane's MFMA fragment are one
// 16-byte load.
constexpr int kMaxTables = 8;
constexpr int kTrWaves = 2;     // waves per k_tr_fwd block
constexpr int kBiasCols = 272;  // per-tile bias sums: db1[128], db2[128], db3[16]

typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));

struct TrainNet {
  float* prm;
  float* grad;
  float* m;
  float* v;
  const uint8_t* mask;
  const uint32_t* codes;  // partition-code loss when set, else the triple loss
  uint64_t seed;          // triple stream of this step
  float c1, c2;           // Adam bias corrections of this step
};

struct TrainArgs {
  TrainNet net[kMaxTables];
  MlpLayout L;
  const float* X;
  int d;
  int64_t n;
  const hdb_nnd_element* lists;  // triples drawn from these lists, or
  const int32_t* given_rows;     // the caller's 3B rows (one table)
  int64_t B, R, Rp, tiles;       // triples, rows 3B, rows rounded up to 32, Rp / 16
  // per-table scratch, with the element stride between tables
  int32_t* rows;
  int64_t s_rows;  // R
  float* Z;
  int64_t s_z;  // Rp x 16
  float* P;
  int64_t s_p;  // P1 then P2, Rp x 128 each
  __bf16* opa;
  int64_t s_opa;  // X rows (Rp x kinp), H1, H2 (Rp x 128 each), blocked
  __bf16* opb;
  int64_t s_opb;  // dP1, dP2 (Rp x 128 each), dZ (Rp x 16), blocked
  float* tsum;
  int64_t s_tsum;  // tiles x 16
  float* bsum;
  int64_t s_bsum;  // kBiasCols x tiles (column-major: one bias column per row)
  float* tmean;
  int64_t s_tmean;  // 16: mean of tanh(z) per code bit over the R rows
  float* gbias;
  int64_t s_gbias;  // kBiasCols: the bias gradients
  float* lsum;
  int64_t s_lsum;  // tiles
  float* wpart;
  int64_t s_wpart;  // splits x L.total (weight entries)
  int splits, chunks_per_split;
  float lr;
  int adam;
};

__device__ __forceinline__ int64_t blk_at(int64_t r, int c, int C) {
  return ((r >> 5) * static_cast<int64_t>(C) + c) * 32 + (r & 31);
}

// Row r of the triples of one step (rows [0, B) anchors, [B, 2B) positives,
// [2B, 3B) the rest): anchor uniform, positive a uniform entry of the
// anchor's kNN list; the negative is, three times in four, the end of a
// kNegWalk-step random walk over the lists (a point of the anchor's own
// region beyond its neighbours, so that decorrelating it splits large
// clusters into several buckets), otherwise uniform.  One xorshift64*
// stream per triple.
constexpr int kNegWalk = 3;

__device__ __forceinline__ int64_t triple_row(const hdb_nnd_element* __restrict__ lists, int64_t n, int64_t B,
                                              uint64_t seed, int64_t r) {
  const int64_t b = r % B;
  const int64_t role = r / B;
  uint64_t h = xorshift64star(seed ^ (static_cast<uint64_t>(b) * 0x9E3779B97F4A7C15ull));
  const int64_t a = static_cast<int64_t>(h % static_cast<uint64_t>(n));
  if (role == 0) return a;
  h = xorshift64star(h);
  uint32_t pid = label_id(lists[a * kK + static_cast<int>(h % kK)].label);
  if (pid == kInvalidId || static_cast<int64_t>(pid) >= n) pid = static_cast<uint32_t>(a);
  if (role == 1) return pid;
  h = xorshift64star(h);
  int64_t neg;
  if ((h & 3u) != 0) {
    neg = a;
    for (int s = 0; s < kNegWalk; ++s) {
      h = xorshift64star(h);
      const uint32_t nx = label_id(lists[neg * kK + static_cast<int>(h % kK)].label);
      if (nx != kInvalidId && static_cast<int64_t>(nx) < n) neg = nx;
    }
  } else {
    h = xorshift64star(h);
    neg = static_cast<int64_t>(h % static_cast<uint64_t>(n));
  }
  return neg;
}

// One wave: out[16 x N] = act(in[16 x K] . W[K x N] + bias), `in` a
// row-major LDS tile (stride ldi), W row-major in global memory.  Results go
// to the LDS tile `out` (stride ldo); when gP is set, the FP32
// pre-activations of the valid rows go to gP (row-major, N columns) and the
// BF16 activations to gH (blocked, zero for rows past `valid`).
template <bool GELU>
__device__ __forceinline__ void tr_layer(const float* in, int ldi, int K, const float* __restrict__ W,
                                         const float* __restrict__ bias, int N, float* out, int ldo,
                                         float* __restrict__ gP, __bf16* __restrict__ gH, int64_t r0,
                                         int64_t valid) {
  const unsigned l = __lane_id();
  const int r16 = l & 15, kq = l >> 4;
  for (int n0 = 0; n0 < N; n0 += 16) {
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int k0 = 0; k0 < K; k0 += 32) {
      bf16x8 a, b;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int k = k0 + 8 * kq + e;
        a[e] = static_cast<__bf16>(in[r16 * ldi + k]);
        b[e] = static_cast<__bf16>(W[static_cast<int64_t>(k) * N + n0 + r16]);
      }
      acc = mfma(a, b, acc);
    }
    const int col = n0 + r16;
    bf16x4 hv;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int row = 4 * kq + q;
      const float pre = acc[q] + bias[col];
      const float v = GELU ? gelu(pre) : pre;
      out[row * ldo + col] = v;
      hv[q] = static_cast<__bf16>(row < valid ? v : 0.0f);
      if (gP && row < valid) gP[(r0 + row) * N + col] = pre;
    }
    if (gH) *reinterpret_cast<bf16x4*>(gH + blk_at(r0 + 4 * kq, col, N)) = hv;
  }
}

__global__ __launch_bounds__(kTrWaves * 64) void k_tr_fwd(TrainArgs A) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  const int t = blockIdx.y;
  const MlpLayout L = A.L;
  const float* prm = A.net[t].prm;
  const unsigned l = __lane_id();
  const unsigned w = threadIdx.x >> 6;
  const int ldi = L.kinp + 4, lda = kHid + 4;
  float* in = lds + w * (16 * ldi + 2 * 16 * lda);
  float* a1 = in + 16 * ldi;
  float* a2 = a1 + 16 * lda;
  const int64_t tile = static_cast<int64_t>(blockIdx.x) * kTrWaves + w;
  if (tile >= A.tiles) return;  // no block barriers in this kernel
  const int64_t r0 = tile * 16;
  const int64_t valid = A.R - r0 < 16 ? (A.R - r0 > 0 ? A.R - r0 : 0) : 16;
  int32_t* rows = A.rows + t * A.s_rows;
  int64_t src = -1;
  if (l < static_cast<unsigned>(valid)) {
    src = A.given_rows ? A.given_rows[r0 + l] : triple_row(A.lists, A.n, A.B, A.net[t].seed, r0 + l);
    rows[r0 + l] = static_cast<int32_t>(src);
  }
  for (int i = 0; i < 16; ++i) {
    const int64_t s = static_cast<int64_t>(__shfl(static_cast<int>(src), i));
    for (int k = l; k < L.kinp; k += 64) in[i * ldi + k] = (i < valid && k < A.d) ? A.X[s * A.d + k] : 0.0f;
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  __bf16* opa = A.opa + t * A.s_opa;
  // X rows as BF16 operands: lane c writes column c of the tile's 16 rows
  for (int c = l; c < L.kinp; c += 64) {
    bf16x8 lo, hi;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      lo[e] = static_cast<__bf16>(in[e * ldi + c]);
      hi[e] = static_cast<__bf16>(in[(e + 8) * ldi + c]);
    }
    bf16x8* dst = reinterpret_cast<bf16x8*>(opa + blk_at(r0, c, L.kinp));
    dst[0] = lo;
    dst[1] = hi;
  }
  float* P = A.P + t * A.s_p;
  tr_layer<true>(in, ldi, L.kinp, prm + L.w1, prm + L.b1, kHid, a1, lda, P, opa + A.Rp * L.kinp, r0, valid);
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  tr_layer<true>(a1, lda, kHid, prm + L.w2, prm + L.b2, kHid, a2, lda, P + A.Rp * kHid,
                 opa + A.Rp * L.kinp + A.Rp * kHid, r0, valid);
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  // layer 3: Z rows and the tile's sums of tanh(Z) per code bit
  {
    const int r16 = l & 15, kq = l >> 4;
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int k0 = 0; k0 < kHid; k0 += 32) {
      bf16x8 a, b;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int k = k0 + 8 * kq + e;
        a[e] = static_cast<__bf16>(a2[r16 * lda + k]);
        b[e] = static_cast<__bf16>(prm[L.w3 + static_cast<int64_t>(k) * kOutP + r16]);
      }
      acc = mfma(a, b, acc);
    }
    float* Z = A.Z + t * A.s_z;
    float ts = 0.0f;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int row = 4 * kq + q;
      const float z = acc[q] + prm[L.b3 + r16];
      Z[(r0 + row) * kOutP + r16] = row < valid ? z : 0.0f;
      if (row < valid && r16 < kCode) ts += tanhf(z);
    }
    ts += __shfl_xor(ts, 16);
    ts += __shfl_xor(ts, 32);
    if (kq == 0) A.tsum[t * A.s_tsum + tile * 16 + r16] = ts;
  }
}

// Loss rows and dZ of one 16-row tile: lane l holds row l % 16, columns
// 4 (l / 16) .. + 3; the sums over a row's 12 columns combine the four
// lanes of the row (xor 16, xor 32).
__global__ __launch_bounds__(256) void k_tr_bwd(TrainArgs A) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  const int t = blockIdx.y;
  const MlpLayout L = A.L;
  const float* prm = A.net[t].prm;
  const uint32_t* codes = A.net[t].codes;
  const unsigned l = __lane_id();
  const unsigned w = threadIdx.x >> 6;
  const int lda = kHid + 4;
  float* gz = lds + w * (16 * 36 + 16 * lda + 16);
  float* g2 = gz + 16 * 36;
  float* rl = g2 + 16 * lda;  // per-row loss
  const int64_t tile = static_cast<int64_t>(blockIdx.x) * 4 + w;
  if (tile >= A.tiles) return;  // no block barriers in this kernel
  const int64_t r0 = tile * 16;
  const int64_t B = A.B, R = A.R;
  const float* Z = A.Z + t * A.s_z;
  const int i = static_cast<int>(l & 15), kq = static_cast<int>(l >> 4);
  const int64_t r = r0 + i;
  const bool valid = r < R;
  float dz[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  float row_loss = 0.0f;
  if (!codes) {
    // mean of tanh(z) per bit over the R rows (k_tr_tmean)
    const float mean_c = A.tmean[t * A.s_tmean + i];  // lane l: bit l % 16
    const int role = valid ? static_cast<int>(r / B) : 3;
    const int64_t b = valid ? r % B : 0;
    float ta[4], tp[4], tn[4], mean[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int c = 4 * kq + j;
      mean[j] = __shfl(mean_c, c);
      const bool on = valid && c < kCode;
      ta[j] = on ? tanhf(Z[b * kOutP + c]) : 0.0f;
      tp[j] = (on && role <= 1) ? tanhf(Z[(B + b) * kOutP + c]) : 0.0f;
      tn[j] = (on && role != 1) ? tanhf(Z[(2 * B + b) * kOutP + c]) : 0.0f;
    }
    float s = 0.0f, lpos = 0.0f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      s += ta[j] * tn[j];
      const float df = ta[j] - tp[j];
      lpos += df * df;
    }
    s += __shfl_xor(s, 16);
    s += __shfl_xor(s, 32);
    lpos += __shfl_xor(lpos, 16);
    lpos += __shfl_xor(lpos, 32);
    s /= kCode;
    lpos /= kCode;
    const float inv_b = 1.0f / static_cast<float>(B);
    const float bal = 2.0f / static_cast<float>(3 * B);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (!valid || 4 * kq + j >= kCode) continue;
      float dt, tt;
      if (role == 0) {
        dt = (2.0f / kCode) * (ta[j] - tp[j]) * inv_b + (2.0f * s / kCode) * tn[j] * inv_b + bal * mean[j];
        tt = ta[j];
      } else if (role == 1) {
        dt = -(2.0f / kCode) * (ta[j] - tp[j]) * inv_b + bal * mean[j];
        tt = tp[j];
      } else {
        dt = (2.0f * s / kCode) * ta[j] * inv_b + bal * mean[j];
        tt = tn[j];
      }
      dz[j] = dt * (1.0f - tt * tt);
    }
    row_loss = (valid && role == 0) ? lpos + s * s : 0.0f;
  } else {
    // partition-code loss: (t - s_code)^2 on every row, the kNN pair term on
    // rows (b, B + b)
    const int32_t* rows = A.rows + t * A.s_rows;
    const uint32_t code = valid ? codes[rows[r]] : 0u;
    const bool paired = valid && r < 2 * B;
    const int64_t other = r < B ? r + B : r - B;
    const float inv_r = 1.0f / static_cast<float>(R);
    const float inv_b = 1.0f / static_cast<float>(B);
    float lt = 0.0f, lp = 0.0f;
    float tv[4], dfv[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int c = 4 * kq + j;
      const bool on = valid && c < kCode;
      tv[j] = on ? tanhf(Z[r * kOutP + c]) : 0.0f;
      dfv[j] = (on && paired) ? tv[j] - tanhf(Z[other * kOutP + c]) : 0.0f;
      const float e = on ? tv[j] - (((code >> c) & 1u) ? 1.0f : -1.0f) : 0.0f;
      lt += e * e;
      lp += dfv[j] * dfv[j];
      float dt = (2.0f / kCode) * e * inv_r;
      if (paired) dt += (2.0f / kCode) * dfv[j] * inv_b;
      dz[j] = on ? dt * (1.0f - tv[j] * tv[j]) : 0.0f;
    }
    lt += __shfl_xor(lt, 16);
    lt += __shfl_xor(lt, 32);
    lp += __shfl_xor(lp, 16);
    lp += __shfl_xor(lp, 32);
    row_loss = valid ? lt / kCode * inv_r + (r < B ? lp / kCode * inv_b : 0.0f) : 0.0f;
  }
  // dZ tile in LDS (columns 16..31 zero: the k padding of dH2 = dZ W3^T)
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    gz[i * 36 + 4 * kq + j] = dz[j];
    gz[i * 36 + 16 + 4 * kq + j] = 0.0f;
  }
  if (kq == 0) rl[i] = row_loss;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  float* bs = A.bsum + t * A.s_bsum + tile;  // column c at bs[c * tiles]
  __bf16* opb = A.opb + t * A.s_opb;
  if (l < 16) {  // db3 and the BF16 dZ operand: lane c takes column c
    float sum = 0.0f;
    bf16x8 lo, hi;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      sum += gz[e * 36 + l];
      lo[e] = static_cast<__bf16>(gz[e * 36 + l]);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      sum += gz[(e + 8) * 36 + l];
      hi[e] = static_cast<__bf16>(gz[(e + 8) * 36 + l]);
    }
    bs[(256 + l) * A.tiles] = sum;
    bf16x8* dst = reinterpret_cast<bf16x8*>(opb + 2 * A.Rp * kHid + blk_at(r0, static_cast<int>(l), kOutP));
    dst[0] = lo;
    dst[1] = hi;
  }
  if (l == 16) {
    float s = 0.0f;
    for (int q = 0; q < 16; ++q) s += rl[q];
    A.lsum[t * A.s_lsum + tile] = s;
  }
  const float* P1 = A.P + t * A.s_p;
  const float* P2 = P1 + A.Rp * kHid;
  const float* W3 = prm + L.w3;  // [128][16]
  const float* W2 = prm + L.w2;  // [128][128]
  const int r16 = i;
  // dP2 = (dZ W3^T) * gelu'(P2): BF16 operand, db2, and the LDS tile for dP1
  for (int n0 = 0; n0 < kHid; n0 += 16) {
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    bf16x8 a, b;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int k = 8 * kq + e;  // output unit of layer 3
      a[e] = static_cast<__bf16>(gz[r16 * 36 + k]);
      b[e] = static_cast<__bf16>(k < kOutP ? W3[(n0 + r16) * kOutP + k] : 0.0f);
    }
    acc = mfma(a, b, acc);
    const int col = n0 + r16;
    bf16x4 hv;
    float cs = 0.0f;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int row = 4 * kq + q;
      const bool ok = r0 + row < R;
      const float g = ok ? acc[q] * gelu_grad(P2[(r0 + row) * kHid + col]) : 0.0f;
      g2[row * lda + col] = g;
      hv[q] = static_cast<__bf16>(g);
      cs += g;
    }
    *reinterpret_cast<bf16x4*>(opb + A.Rp * kHid + blk_at(r0 + 4 * kq, col, kHid)) = hv;
    cs += __shfl_xor(cs, 16);
    cs += __shfl_xor(cs, 32);
    if (kq == 0) bs[(128 + col) * A.tiles] = cs;
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  // dP1 = (dP2 W2^T) * gelu'(P1): BF16 operand and db1
  for (int n0 = 0; n0 < kHid; n0 += 16) {
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int k0 = 0; k0 < kHid; k0 += 32) {
      bf16x8 a, b;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int k = k0 + 8 * kq + e;  // unit of hidden layer 2
        a[e] = static_cast<__bf16>(g2[r16 * lda + k]);
        b[e] = static_cast<__bf16>(W2[(n0 + r16) * kHid + k]);
      }
      acc = mfma(a, b, acc);
    }
    const int col = n0 + r16;
    bf16x4 hv;
    float cs = 0.0f;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int row = 4 * kq + q;
      const bool ok = r0 + row < R;
      const float g = ok ? acc[q] * gelu_grad(P1[(r0 + row) * kHid + col]) : 0.0f;
      hv[q] = static_cast<__bf16>(g);
      cs += g;
    }
    *reinterpret_cast<bf16x4*>(opb + blk_at(r0 + 4 * kq, col, kHid)) = hv;
    cs += __shfl_xor(cs, 16);
    cs += __shfl_xor(cs, 32);
    if (kq == 0) bs[col * A.tiles] = cs;
  }
}

// Weight-gradient products over the row chunks of one split: wave = one
// 32 x 32 region (2 x 2 MFMA tiles) of dW1 (kinp x 128), dW2 (128 x 128) or
// dW3 (128 x 16, one column tile).  Output (m, n) of the product is entry
// m * N + n of the weight; partials go to wpart[split][weight offset + ...].
__global__ __launch_bounds__(256) void k_tr_wgrad(TrainArgs A) {
  const int t = blockIdx.z, split = blockIdx.y;
  const MlpLayout L = A.L;
  const unsigned l = __lane_id();
  const int r16 = static_cast<int>(l & 15), kq = static_cast<int>(l >> 4);
  const int region = static_cast<int>(blockIdx.x) * 4 + static_cast<int>(threadIdx.x >> 6);
  const int g1 = (L.kinp / 32) * 4;
  const __bf16* opa = A.opa + t * A.s_opa;
  const __bf16* opb = A.opb + t * A.s_opb;
  const __bf16 *Ab, *Bb;
  int CA, CB, N, m0, n0, nt;
  int64_t woff;
  if (region < g1) {  // dW1 = X^T dP1
    Ab = opa, CA = L.kinp, Bb = opb, CB = kHid, N = kHid, woff = L.w1;
    m0 = (region / 4) * 32, n0 = (region % 4) * 32, nt = 2;
  } else if (region < g1 + 16) {  // dW2 = H1^T dP2
    const int q = region - g1;
    Ab = opa + A.Rp * L.kinp, CA = kHid, Bb = opb + A.Rp * kHid, CB = kHid, N = kHid, woff = L.w2;
    m0 = (q / 4) * 32, n0 = (q % 4) * 32, nt = 2;
  } else if (region < g1 + 20) {  // dW3 = H2^T dZ
    const int q = region - g1 - 16;
    Ab = opa + A.Rp * L.kinp + A.Rp * kHid, CA = kHid, Bb = opb + 2 * A.Rp * kHid, CB = kOutP, N = kOutP;
    woff = L.w3, m0 = q * 32, n0 = 0, nt = 1;
  } else {
    return;
  }
  const int64_t nchunks = A.Rp / 32;
  const int64_t kc0 = static_cast<int64_t>(split) * A.chunks_per_split;
  const int64_t kc1 = kc0 + A.chunks_per_split < nchunks ? kc0 + A.chunks_per_split : nchunks;
  f32x4 acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[a][b] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  for (int64_t kc = kc0; kc < kc1; ++kc) {
    bf16x8 fa[2], fb[2];
#pragma unroll
    for (int a = 0; a < 2; ++a)
      fa[a] = *reinterpret_cast<const bf16x8*>(Ab + ((kc * CA + m0 + 16 * a + r16) * 32 + 8 * kq));
#pragma unroll
    for (int b = 0; b < 2; ++b)
      if (b < nt) fb[b] = *reinterpret_cast<const bf16x8*>(Bb + ((kc * CB + n0 + 16 * b + r16) * 32 + 8 * kq));
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      acc[a][0] = mfma(fa[a], fb[0], acc[a][0]);
      if (nt > 1) acc[a][1] = mfma(fa[a], fb[1], acc[a][1]);
    }
  }
  float* out = A.wpart + t * A.s_wpart + static_cast<int64_t>(split) * L.total + woff;
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      if (b >= nt) continue;
#pragma unroll
      for (int q = 0; q < 4; ++q) out[(m0 + 16 * a + 4 * kq + q) * N + n0 + 16 * b + r16] = acc[a][b][q];
    }
}

// Mean of tanh(z) per code bit over the R rows, from the per-tile sums of
// k_tr_fwd in a fixed order (16 strided partial sums, then in order): one
// block per table.
__global__ __launch_bounds__(256) void k_tr_tmean(TrainArgs A) {
  __shared__ float part[16][16];
  const int t = blockIdx.x;
  const int bit = static_cast<int>(threadIdx.x & 15), q = static_cast<int>(threadIdx.x >> 4);
  const float* ts = A.tsum + t * A.s_tsum;
  float s = 0.0f;
  for (int64_t tt = q; tt < A.tiles; tt += 16) s += ts[tt * 16 + bit];
  part[q][bit] = s;
  __syncthreads();
  if (threadIdx.x < 16) {
    float m = 0.0f;
    for (int k = 0; k < 16; ++k) m += part[k][threadIdx.x];
    A.tmean[t * A.s_tmean + threadIdx.x] = m / static_cast<float>(A.R);
  }
}

// Bias gradients: one wave per bias column sums its per-tile partials
// (lane-strided, then a fixed xor tree).
__global__ __launch_bounds__(256) void k_tr_bred(TrainArgs A) {
  const int t = blockIdx.y;
  const int col = static_cast<int>(blockIdx.x) * 4 + static_cast<int>(threadIdx.x >> 6);
  if (col >= kBiasCols) return;
  const unsigned lane = __lane_id();
  const float* bs = A.bsum + t * A.s_bsum + static_cast<int64_t>(col) * A.tiles;
  float s = 0.0f;
  for (int64_t tt = lane; tt < A.tiles; tt += 64) s += bs[tt];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
  if (lane == 0) A.gbias[t * A.s_gbias + col] = s;
}

// Gradient entry i of table blockIdx.y = its partial sums in a fixed order
// (row splits for weights, row tiles for biases); then, when A.adam, one
// Adam step (beta 0.9 / 0.999, eps 1e-8) on the trainable entries.
__global__ __launch_bounds__(256) void k_tr_apply(TrainArgs A) {
  const int t = blockIdx.y;
  const MlpLayout L = A.L;
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= L.total) return;
  const TrainNet& net = A.net[t];
  int bias = -1;
  if (i >= L.b1 && i < L.b1 + kHid) bias = static_cast<int>(i - L.b1);
  else if (i >= L.b2 && i < L.b2 + kHid) bias = 128 + static_cast<int>(i - L.b2);
  else if (i >= L.b3 && i < L.b3 + kOutP) bias = 256 + static_cast<int>(i - L.b3);
  float g = 0.0f;
  if (bias >= 0) {
    g = A.gbias[t * A.s_gbias + bias];
  } else {
    const float* wp = A.wpart + t * A.s_wpart + i;
    for (int s = 0; s < A.splits; ++s) g += wp[static_cast<int64_t>(s) * L.total];
  }
  net.grad[i] = g;
  if (!A.adam || !net.mask[i]) return;
  const float mi = 0.9f * net.m[i] + 0.1f * g;
  const float vi = 0.999f * net.v[i] + 0.001f * g * g;
  net.m[i] = mi;
  net.v[i] = vi;
  net.prm[i] -= A.lr * (mi / net.c1) / (sqrtf(vi / net.c2) + 1e-8f);
}

// Balanced random-projection tree codes: at level l every cell (the l code
// bits so far) splits at the median of x . r(l, cell); r is a Gaussian
// direction drawn by Box-Muller from xorshift64*(seed, l, cell).  Keys are
// (cell << 52) | (orderable projection bits << 20) | point id (n <= 2^20).
__global__ void k_rp_keys(const float* __restrict__ X, int64_t n, int d, int level, uint64_t seed,
                          const uint32_t* __restrict__ code, uint64_t* __restrict__ keys) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t c = code[i];
  uint64_t h = xorshift64star(seed ^ (static_cast<uint64_t>(level + 1) << 44) ^
                              (static_cast<uint64_t>(c) * 0x9E3779B97F4A7C15ull));
  float proj = 0.0f;
  for (int k = 0; k < d; k += 2) {
    h = xorshift64star(h);
    const float u1 = (static_cast<float>(h >> 40) + 1.0f) * (1.0f / 16777217.0f);
    h = xorshift64star(h);
    const float u2 = static_cast<float>(h >> 40) * (1.0f / 16777216.0f);
    const float rad = sqrtf(-2.0f * logf(u1));
    proj = __builtin_fmaf(X[i * d + k], rad * cosf(6.2831853f * u2), proj);
    if (k + 1 < d) proj = __builtin_fmaf(X[i * d + k + 1], rad * sinf(6.2831853f * u2), proj);
  }
  uint32_t b = __float_as_uint(proj);
  b = (b & 0x80000000u) ? ~b : (b | 0x80000000u);
  keys[i] = (static_cast<uint64_t>(c) << 52) | (static_cast<uint64_t>(b) << 20) | static_cast<uint64_t>(i);
}

__global__ void k_rp_cells(const uint64_t* __restrict__ keys, int64_t n, uint32_t* __restrict__ cell) {
  const int64_t s = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (s < n) cell[s] = static_cast<uint32_t>(keys[s] >> 52);
}

// The lower half (floor) of each cell's sorted run gets bit 0, the rest 1.
__global__ void k_rp_split(const uint64_t* __restrict__ keys, int64_t n, const int32_t* __restrict__ cs,
                           const int32_t* __restrict__ ce, uint32_t* __restrict__ code) {
  const int64_t s = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (s >= n) return;
  const uint64_t k = keys[s];
  const uint32_t c = static_cast<uint32_t>(k >> 52);
  const int64_t id = static_cast<int64_t>(k & 0xFFFFFull);
  const int32_t half = (ce[c] - cs[c]) / 2;
  code[id] = (c << 1) | ((s - cs[c]) >= half ? 1u : 0u);
}

// ------------------------------------------------------- inference path --
// Weights packed into MFMA fragment order (BF16): fragment f holds, for lane
// l, the 8 weights W[k0 + kperm(l/16, e)][n0 + l%16] (e = 0..7) of column
// tile n0 and k step k0.  Layer 1 has (kinp/32) x 8 fragments (column tile
// major) with kperm(g, e) = 8 g + e; layer 2 has 4 x 8 and layer 3 4 (N = 16)
// with kperm(g, e) = 4 g + e for e < 4 and 16 + 4 g + (e - 4) above: the
// order in which the transposed product leaves the previous layer's units in
// a lane (units 4 g .. 4 g + 3 of two consecutive 16-unit tiles), so each
// layer's output feeds the next layer's MFMA from registers.
__host__ __device__ inline int infer_frags(int kinp) { return (kinp / 32) * 8 + 32 + 4; }

__global__ void k_mlp_pack(const float* __restrict__ prm, MlpLayout L, __bf16* __restrict__ packed) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const int ks1 = L.kinp / 32;
  const int nf1 = ks1 * 8, nf2 = 32;
  if (t >= static_cast<int64_t>(infer_frags(L.kinp)) * 64) return;
  int f = static_cast<int>(t >> 6);
  const int lane = static_cast<int>(t & 63);
  const float* W;
  int N, nt, ks;
  if (f < nf1) {
    W = prm + L.w1, N = kHid, nt = f / ks1, ks = f % ks1;
  } else if (f < nf1 + nf2) {
    f -= nf1;
    W = prm + L.w2, N = kHid, nt = f / 4, ks = f % 4;
  } else {
    f -= nf1 + nf2;
    W = prm + L.w3, N = kOutP, nt = 0, ks = f;
  }
  const int r16 = lane & 15, kq = lane >> 4;
  const bool l1 = static_cast<int>(t >> 6) < nf1;
  for (int e = 0; e < 8; ++e) {
    const int k = ks * 32 + (l1 ? 8 * kq + e : (e < 4 ? 4 * kq + e : 16 + 4 * kq + (e - 4)));
    packed[t * 8 + e] = static_cast<__bf16>(W[static_cast<int64_t>(k) * N + nt * 16 + r16]);
  }
}

// Bucket keys written by the inference kernel in place of Z: key =
// (sign code of outputs 0..11) << qbits | the projection x.u quantised to
// qbits bits over [-lim, lim].
struct InferKeys {
  const float* u;
  float lim;
  int qbits;
  uint32_t* keys;
  uint32_t* ids;
};

__device__ __forceinline__ uint32_t proj_q(const float* __restrict__ x, const float* __restrict__ u, int d,
                                           float lim, int qbits) {
  float s = 0.0f;
  for (int k = 0; k < d; ++k) s = __builtin_fmaf(x[k], u[k], s);
  float t = (s / lim) * 0.5f + 0.5f;
  t = t < 0.0f ? 0.0f : (t > 1.0f ? 1.0f : t);
  return static_cast<uint32_t>(t * static_cast<float>((1u << qbits) - 1u));
}

// Projection bits of the bucket keys: enough levels that a level holds about
// 2^8 points or fewer at n points, 12 at least and 20 at most, so a key of
// 12 + qbits bits sorts in three passes up to about a million points and in
// four beyond.  The order inside a projection level is arbitrary, so coarse
// levels at large n fill a window with unrelated points.
inline int proj_bits(int64_t n) {
  int lg = 0;
  while ((int64_t{1} << lg) < n) ++lg;
  const int q = lg - 8;
  return q < 12 ? 12 : (q > 20 ? 20 : q);
}

// Z = forward(X) for R rows as the transposed products Z^T = W3^T g(W2^T
// g(W1^T X^T)): the packed fragments are the A operands and each 16-row tile
// is the B operand, so a layer's output -- lane (g, r) holds units 4 g .. 4 g
// + 3 of each 16-unit tile for row r -- is the next layer's B operand as it
// stands (the fragments' K order matches), and activations never leave the
// registers.  The block keeps the packed weights and biases in LDS; each
// wave strides over 16-row tiles.  KEYS: the rows' bucket keys instead of Z
// (a row's 12 code bits from four ballots).
template <bool KEYS>
__global__ __launch_bounds__(512, 6) void k_mlp_infer(const float* __restrict__ X, int d, int64_t R,
                                                  const __bf16* __restrict__ packed, const float* __restrict__ prm,
                                                  MlpLayout L, float* __restrict__ Z, InferKeys ko) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_b[];
  const int ks1 = L.kinp / 32;
  const int nfrag = infer_frags(L.kinp);
  const int waves = static_cast<int>(blockDim.x >> 6);
  __bf16* sw = reinterpret_cast<__bf16*>(lds_b);
  float* sb = reinterpret_cast<float*>(sw + nfrag * 512);  // b1 | b2 | b3: 128 + 128 + 16
  for (int i = threadIdx.x; i < nfrag * 64; i += blockDim.x)
    reinterpret_cast<uint4*>(sw)[i] = reinterpret_cast<const uint4*>(packed)[i];
  for (int i = threadIdx.x; i < 272; i += blockDim.x)
    sb[i] = i < kHid ? prm[L.b1 + i] : (i < 2 * kHid ? prm[L.b2 + i - kHid] : prm[L.b3 + i - 2 * kHid]);
  __syncthreads();
  const unsigned l = __lane_id();
  const int w = static_cast<int>(threadIdx.x >> 6);
  const int r16 = static_cast<int>(l & 15), kq = static_cast<int>(l >> 4);
  auto frag = [&](int f) { return *reinterpret_cast<const bf16x8*>(sw + (f * 64 + static_cast<int>(l)) * 8); };
  // bias + GELU of two 16-unit tiles into one B operand (units 32 s + kperm)
  auto act = [&](const f32x4& lo, const f32x4& hi, const float* bias, int s) {
    const float4 blo = *reinterpret_cast<const float4*>(bias + 32 * s + 4 * kq);
    const float4 bhi = *reinterpret_cast<const float4*>(bias + 32 * s + 16 + 4 * kq);
    bf16x8 v;
    v[0] = static_cast<__bf16>(gelu(lo[0] + blo.x));
    v[1] = static_cast<__bf16>(gelu(lo[1] + blo.y));
    v[2] = static_cast<__bf16>(gelu(lo[2] + blo.z));
    v[3] = static_cast<__bf16>(gelu(lo[3] + blo.w));
    v[4] = static_cast<__bf16>(gelu(hi[0] + bhi.x));
    v[5] = static_cast<__bf16>(gelu(hi[1] + bhi.y));
    v[6] = static_cast<__bf16>(gelu(hi[2] + bhi.z));
    v[7] = static_cast<__bf16>(gelu(hi[3] + bhi.w));
    return v;
  };
  const int64_t ntiles = (R + 15) / 16;
  for (int64_t tile = static_cast<int64_t>(blockIdx.x) * waves + w; tile < ntiles;
       tile += static_cast<int64_t>(gridDim.x) * waves) {
    // the weight fragments are the same every tile: an acquire fence keeps
    // the compiler from hoisting all 44 of them out of the loop (176
    // registers) and makes each tile read them from LDS as it goes
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int64_t row = tile * 16 + r16;  // this lane's row (B operand column)
    const bool rv = row < R;
    f32x4 acc[8];
#pragma unroll
    for (int nt = 0; nt < 8; ++nt) acc[nt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    for (int ks = 0; ks < ks1; ++ks) {  // layer 1: inputs ks * 32 + 8 g + e of the lane's row
      bf16x8 xb;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int k = ks * 32 + 8 * kq + e;
        xb[e] = static_cast<__bf16>((rv && k < d) ? X[row * d + k] : 0.0f);
      }
#pragma unroll
      for (int nt = 0; nt < 8; ++nt) acc[nt] = mfma(frag(nt * ks1 + ks), xb, acc[nt]);
    }
    bf16x8 hb[4];
#pragma unroll
    for (int s2 = 0; s2 < 4; ++s2) hb[s2] = act(acc[2 * s2], acc[2 * s2 + 1], sb, s2);
#pragma unroll
    for (int nt = 0; nt < 8; ++nt) acc[nt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int s2 = 0; s2 < 4; ++s2)  // layer 2
#pragma unroll
      for (int nt = 0; nt < 8; ++nt) acc[nt] = mfma(frag(ks1 * 8 + nt * 4 + s2), hb[s2], acc[nt]);
#pragma unroll
    for (int s2 = 0; s2 < 4; ++s2) hb[s2] = act(acc[2 * s2], acc[2 * s2 + 1], sb + kHid, s2);
    f32x4 o = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int s2 = 0; s2 < 4; ++s2) o = mfma(frag(ks1 * 8 + 32 + s2), hb[s2], o);  // layer 3
    // lane (g, r) holds outputs 4 g .. 4 g + 3 of row r
    const float4 b3 = *reinterpret_cast<const float4*>(sb + 2 * kHid + 4 * kq);
    o[0] += b3.x;
    o[1] += b3.y;
    o[2] += b3.z;
    o[3] += b3.w;
    if (KEYS) {
      // bit 16 g + r of ballot q: output 4 g + q of row r is positive
      uint64_t m[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) m[q] = __ballot(4 * kq + q < kCode && o[q] > 0.0f);
      if (kq == 0 && rv) {
        uint32_t code = 0;
#pragma unroll
        for (int g = 0; g < kCode / 4; ++g)
#pragma unroll
          for (int q = 0; q < 4; ++q)
            code |= static_cast<uint32_t>((m[q] >> (16 * g + r16)) & 1ull) << (4 * g + q);
        ko.keys[row] = (code << ko.qbits) | proj_q(X + row * d, ko.u, d, ko.lim, ko.qbits);
        ko.ids[row] = static_cast<uint32_t>(row);
      }
    } else if (rv) {
#pragma unroll
      for (int q = 0; q < 4; ++q) Z[row * kOutP + 4 * kq + q] = o[q];
    }
  }
}

// Points permuted into the bucket order: row r of Xs is point order[r].
__global__ void k_mlp_permute(const float* __restrict__ X, const uint32_t* __restrict__ order, int64_t n, int d,
                              float* __restrict__ Xs) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= n * d) return;
  const int64_t r = t / d;
  const int k = static_cast<int>(t - r * d);
  Xs[t] = X[static_cast<int64_t>(order[r]) * d + k];
}

constexpr int kSeedTables = 8;  // bucket tables at most
constexpr int kSeedSlots = 64;  // candidate slots per point (one per lane in the merge)
constexpr int kSeedPts = 256;   // points per block, one per lane

template <int W>
__device__ __forceinline__ int64_t seed_lo(int64_t r, int64_t n) {
  int64_t lo = r - W / 2;
  if (lo > n - W - 1) lo = n - W - 1;
  return lo < 0 ? 0 : lo;
}

// Lane r (a position in the table's bucket order) keeps the K nearest of
// the W positions around it (itself skipped), ranked by 32-bit keys: the
// distance bits with the low log2(W) replaced by the window slot, kept in
// registers by a median-of-three insertion.  The winners' exact keys
// are recomputed.  Rows come from LDS when STAGED (stride d + 1, an odd
// stride across lanes); D > 0 fixes d and keeps the point's own row in
// registers.
template <int D, int W, int K, bool STAGED>
__global__ __launch_bounds__(kSeedPts) void k_mlp_seed(const float* __restrict__ Xs,
                                                        const uint32_t* __restrict__ order, int64_t n, int d,
                                                        int slot0, uint64_t* __restrict__ cand) {
  extern __shared__ __attribute__((aligned(16))) float lds_rows[];
  static_assert((W & (W - 1)) == 0 && W <= 512, "window is a power of two");
  const int64_t r0 = static_cast<int64_t>(blockIdx.x) * kSeedPts;
  const int64_t sb = seed_lo<W>(r0, n);
  const float* rows = Xs + sb * d;
  int dp = d;
  if (STAGED) {
    const int64_t last = r0 + kSeedPts - 1 < n ? r0 + kSeedPts - 1 : n - 1;
    int64_t se = seed_lo<W>(last, n) + W + 1;
    if (se > n) se = n;
    dp = d + 1;
    for (int64_t t = threadIdx.x; t < (se - sb) * d; t += kSeedPts) {
      const int64_t rr = t / d;
      lds_rows[rr * dp + (t - rr * d)] = Xs[sb * d + t];
    }
    __syncthreads();
    rows = lds_rows;
  }
  const int64_t r = r0 + threadIdx.x;
  if (r >= n) return;  // after the block's only barrier
  const int64_t lo = seed_lo<W>(r, n);
  const float* self_row = rows + (r - sb) * dp;
  float own[D > 0 ? D : 1];
  if (D > 0) {
#pragma unroll
    for (int k = 0; k < (D > 0 ? D : 1); ++k) own[k] = self_row[k];
  }
  uint32_t best[K];
#pragma unroll
  for (int j = 0; j < K; ++j) best[j] = 0xFFFFFFFFu;
  for (int slot = 0; slot < W; ++slot) {
    int64_t p = lo + slot;
    if (p >= r) p += 1;
    if (p >= n) break;  // only when n <= W: the remaining slots are past the end too
    const float* pr = rows + (p - sb) * dp;
    float acc = 0.0f;
    if (D > 0) {
#pragma unroll
      for (int k = 0; k < (D > 0 ? D : 1); ++k) {
        const float diff = pr[k] - own[k];
        acc = __builtin_fmaf(diff, diff, acc);
      }
    } else {
      acc = d2_any(pr, self_row, d);
    }
    uint32_t key = (__float_as_uint(acc) & ~static_cast<uint32_t>(W - 1)) | static_cast<uint32_t>(slot);
    top_insert_med3<K>(best, key);
  }
  uint64_t* out = cand + static_cast<int64_t>(order[r]) * kSeedSlots + slot0;
#pragma unroll
  for (int j = 0; j < K; ++j) {
    uint64_t key = kKeyMax;
    if (best[j] != 0xFFFFFFFFu) {
      int64_t p = lo + static_cast<int64_t>(best[j] & static_cast<uint32_t>(W - 1));
      if (p >= r) p += 1;
      key = make_key(d2_any(rows + (p - sb) * dp, self_row, d), order[p], 1u);
    }
    out[j] = key;
  }
}

// k_mlp_seed for d = D in {12, 32}: rows staged at a stride of D floats when
// D / 4 is odd, else D + 4 (16-byte rows whose starts fall in distinct
// 4-bank groups for 16 consecutive lanes), read as float4, and ranked by
// |x|^2 + |y|^2 - 2 x.y (clamped at 0) with the rows' norms staged beside
// them; the winners' exact keys are recomputed as in k_mlp_seed.
template <int D, int W, int K>
__global__ __launch_bounds__(kSeedPts) void k_mlp_seed4(const float* __restrict__ Xs,
                                                         const uint32_t* __restrict__ order, int64_t n,
                                                         int slot0, uint64_t* __restrict__ cand) {
  static_assert(D % 4 == 0 && D <= 32, "float4 rows");
  static_assert((W & (W - 1)) == 0 && W <= 512, "window is a power of two");
  constexpr int S = ((D / 4) & 1) ? D : D + 4;
  extern __shared__ __attribute__((aligned(16))) float lds_rows[];
  const int64_t r0 = static_cast<int64_t>(blockIdx.x) * kSeedPts;
  const int64_t sb = seed_lo<W>(r0, n);
  const int64_t last = r0 + kSeedPts - 1 < n ? r0 + kSeedPts - 1 : n - 1;
  int64_t se = seed_lo<W>(last, n) + W + 1;
  if (se > n) se = n;
  const int nrows = static_cast<int>(se - sb);
  float* s_norm = lds_rows + (kSeedPts + W + 1) * S;
  for (int rr = threadIdx.x; rr < nrows; rr += kSeedPts) {
    const float4* src = reinterpret_cast<const float4*>(Xs + (sb + rr) * D);
    float4* dst = reinterpret_cast<float4*>(lds_rows + rr * S);
    float nrm = 0.0f;
#pragma unroll
    for (int k = 0; k < D / 4; ++k) {
      const float4 x = src[k];
      dst[k] = x;
      nrm = __builtin_fmaf(x.x, x.x, nrm);
      nrm = __builtin_fmaf(x.y, x.y, nrm);
      nrm = __builtin_fmaf(x.z, x.z, nrm);
      nrm = __builtin_fmaf(x.w, x.w, nrm);
    }
    s_norm[rr] = nrm;
  }
  __syncthreads();
  const int64_t r = r0 + threadIdx.x;
  if (r >= n) return;  // after the block's only barrier
  const int64_t lo = seed_lo<W>(r, n);
  const float* self_row = lds_rows + (r - sb) * S;
  float4 own[D / 4];
#pragma unroll
  for (int k = 0; k < D / 4; ++k) own[k] = reinterpret_cast<const float4*>(self_row)[k];
  const float own_norm = s_norm[r - sb];
  uint32_t best[K];
#pragma unroll
  for (int j = 0; j < K; ++j) best[j] = 0xFFFFFFFFu;
  for (int slot = 0; slot < W; ++slot) {
    int64_t p = lo + slot;
    if (p >= r) p += 1;
    if (p >= n) break;  // only when n <= W: the remaining slots are past the end too
    const int pl = static_cast<int>(p - sb);
    const float4* pr = reinterpret_cast<const float4*>(lds_rows + pl * S);
    float dot = 0.0f;
#pragma unroll
    for (int k = 0; k < D / 4; ++k) {
      const float4 y = pr[k];
      dot = __builtin_fmaf(own[k].x, y.x, dot);
      dot = __builtin_fmaf(own[k].y, y.y, dot);
      dot = __builtin_fmaf(own[k].z, y.z, dot);
      dot = __builtin_fmaf(own[k].w, y.w, dot);
    }
    const float acc = fmaxf(__builtin_fmaf(-2.0f, dot, own_norm + s_norm[pl]), 0.0f);
    uint32_t key = (__float_as_uint(acc) & ~static_cast<uint32_t>(W - 1)) | static_cast<uint32_t>(slot);
    top_insert_med3<K>(best, key);
  }
  uint64_t* out = cand + static_cast<int64_t>(order[r]) * kSeedSlots + slot0;
#pragma unroll
  for (int j = 0; j < K; ++j) {
    uint64_t key = kKeyMax;
    if (best[j] != 0xFFFFFFFFu) {
      int64_t p = lo + static_cast<int64_t>(best[j] & static_cast<uint32_t>(W - 1));
      if (p >= r) p += 1;
      key = make_key(d2_any(lds_rows + (p - sb) * S, self_row, D), order[p], 1u);
    }
    out[j] = key;
  }
}

// The window search for d = 12 on the matrix cores.  A wave takes 16
// consecutive positions and the span of W + 32 rows that holds all their
// windows (u0 = min(seed_lo(first), n - span)); tile t of the span is 16 rows.
// Rows are staged with two extra features, so that one 16x16x4 FP32 MFMA
// chain over k = 16 gives every ranking distance of the tile directly:
//   A row w = (w_0..w_11, |w|^2, 1, 0, 0), B column p = (-2 p_0..-2 p_11, 1, |p|^2, 0, 0),
//   (A B)[w][p] = |w|^2 + |p|^2 - 2 w.p.
// Feature 4s + g of a row is stored at float 4g + s (row stride 20 floats),
// so lane group g (lanes 16g..16g+15) reads its four k-slices as one
// float4; 20 floats is an odd number of float4s, so 8 consecutive rows fall
// in distinct 4-bank groups.  Lane (g, c) receives rows 4g..4g+3 of each
// tile for position c and keeps the K/2 nearest of them in registers
// (median-of-three insertion); the four lanes of a position then merge
// their lists (xor 16, xor 32) into the K + 1 nearest of the union.  A
// lane's quarter holds more than K/2 of the span's K + 1 nearest rarely
// (then a slightly farther row takes the place): these are initial
// candidates, and every key written is exact.  The position itself
// (distance 0) is dropped when the exact keys are written; each of the four
// lanes writes every fourth winner.  The span rows beyond a window are
// further candidates.
__device__ __forceinline__ float f4_at(const float4& v, int i) {
  return i == 0 ? v.x : (i == 1 ? v.y : (i == 2 ? v.z : v.w));
}

constexpr int kSmWaves = 16;            // waves per block of k_mlp_seed_mfma
constexpr int kSmPts = 16 * kSmWaves;   // positions per block
constexpr int kSmStride = 20;           // staged row stride, floats

constexpr int seed_mfma_span(int W) { return 16 * (W / 16 + 2); }
constexpr size_t seed_mfma_lds(int W) {
  return static_cast<size_t>(kSmPts - 16 + seed_mfma_span(W)) * kSmStride * sizeof(float);
}

template <int W, int K>
__global__ __launch_bounds__(64 * kSmWaves) void k_mlp_seed_mfma(const float* __restrict__ X,
                                                                  const uint32_t* __restrict__ order, int64_t n,
                                                                  int slot0, uint64_t* __restrict__ cand) {
  constexpr int D = 12;
  constexpr int kTiles = W / 16 + 2;
  constexpr int kSpan = 16 * kTiles;
  constexpr int kRow4 = kSmStride / 4;  // float4s per staged row
  constexpr uint32_t kMask = 2u * W - 1u;
  constexpr int kLane = K / 2;  // nearest kept per lane (a quarter of the span)
  static_assert((W & (W - 1)) == 0 && W >= 64 && W <= 512, "window is a power of two");
  static_assert(kSpan <= 2 * W, "span slots fit the key's low bits");
  static_assert(4 * kLane >= K + 1 && 2 * kLane <= K + 1, "lane lists cover the K + 1 nearest");
  extern __shared__ __attribute__((aligned(16))) float4 lds_span4[];
  auto span_lo = [n](int64_t r) {
    const int64_t lo = seed_lo<W>(r, n);
    return lo < n - kSpan ? lo : n - kSpan;
  };
  const int64_t r0 = static_cast<int64_t>(blockIdx.x) * kSmPts;
  const int64_t sb = span_lo(r0);
  const int64_t last_wave = r0 + ((n - r0 < kSmPts ? n - r0 : kSmPts) - 1) / 16 * 16;
  const int nrows = static_cast<int>(span_lo(last_wave) + kSpan - sb);
  for (int j = threadIdx.x; j < nrows; j += 64 * kSmWaves) {
    // row j of the span is point order[sb + j], gathered from X directly
    const float4* src = reinterpret_cast<const float4*>(X + static_cast<int64_t>(order[sb + j]) * D);
    const float4 x0 = src[0], x1 = src[1], x2 = src[2];
    float nrm = 0.0f;
    nrm = __builtin_fmaf(x0.x, x0.x, nrm);
    nrm = __builtin_fmaf(x0.y, x0.y, nrm);
    nrm = __builtin_fmaf(x0.z, x0.z, nrm);
    nrm = __builtin_fmaf(x0.w, x0.w, nrm);
    nrm = __builtin_fmaf(x1.x, x1.x, nrm);
    nrm = __builtin_fmaf(x1.y, x1.y, nrm);
    nrm = __builtin_fmaf(x1.z, x1.z, nrm);
    nrm = __builtin_fmaf(x1.w, x1.w, nrm);
    nrm = __builtin_fmaf(x2.x, x2.x, nrm);
    nrm = __builtin_fmaf(x2.y, x2.y, nrm);
    nrm = __builtin_fmaf(x2.z, x2.z, nrm);
    nrm = __builtin_fmaf(x2.w, x2.w, nrm);
    float4* dst = lds_span4 + j * kRow4;
    dst[0] = make_float4(x0.x, x1.x, x2.x, nrm);   // features 0, 4, 8, 12
    dst[1] = make_float4(x0.y, x1.y, x2.y, 1.0f);  // features 1, 5, 9, 13
    dst[2] = make_float4(x0.z, x1.z, x2.z, 0.0f);  // features 2, 6, 10, 14
    dst[3] = make_float4(x0.w, x1.w, x2.w, 0.0f);  // features 3, 7, 11, 15
  }
  __syncthreads();
  const int wv = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  const int g = lane >> 4;
  const int c = lane & 15;
  const int64_t rw = r0 + 16 * wv;
  if (rw >= n) return;  // wave-uniform, after the block's only barrier
  const int j0 = static_cast<int>(span_lo(rw) - sb);
  const int64_t r = rw + c;
  const bool valid = r < n;
  const int jr = valid ? static_cast<int>(r - sb) : j0;
  // B column: this lane's position, k-slices 4s + g scaled by -2, and
  // features 12..15 = (1, |p|^2, 0, 0)
  float4 bq = lds_span4[jr * kRow4 + g];
  const float nr = lds_span4[jr * kRow4].w;
  bq.x *= -2.0f;
  bq.y *= -2.0f;
  bq.z *= -2.0f;
  bq.w = g == 0 ? 1.0f : (g == 1 ? nr : 0.0f);
  if (!valid) bq = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  uint32_t part[kLane];
#pragma unroll
  for (int j = 0; j < kLane; ++j) part[j] = 0xFFFFFFFFu;
  const float4* arow = lds_span4 + (j0 + c) * kRow4 + g;
#pragma unroll 2
  for (int t = 0; t < kTiles; ++t) {
    const float4 av = arow[t * 16 * kRow4];
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(av.x, bq.x, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(av.y, bq.y, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(av.z, bq.z, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(av.w, bq.w, acc, 0, 0, 0);
    const uint32_t s0 = static_cast<uint32_t>(16 * t + 4 * g);
#pragma unroll
    for (int q = 0; q < 4; ++q) top_insert_med3<kLane>(part, (nonneg_bits(acc[q]) & ~kMask) | (s0 + q));
  }
  // lanes g and g ^ 1: the nearest 2 kLane of half the span, sorted
  uint32_t top[K + 1];
#pragma unroll
  for (int j = 0; j <= K; ++j) top[j] = j < kLane ? part[j] : 0xFFFFFFFFu;
#pragma unroll
  for (int j = 0; j < kLane; ++j)
    top_insert_med3<K + 1>(top, static_cast<uint32_t>(__shfl_xor(static_cast<int>(part[j]), 16)));
  // with lanes g ^ 2: over ascending lists A (g < 2) and B (g >= 2),
  // min(A[j], B[K - j]) is the K + 1 smallest of both (in no particular
  // order); all four lanes form the same array, so the every-fourth split
  // below writes each winner once
  const bool hi = (g & 2) != 0;
  uint32_t mrg[K + 1];
#pragma unroll
  for (int j = 0; j <= K; ++j) {
    const uint32_t mine = hi ? top[K - j] : top[j];
    const uint32_t o = static_cast<uint32_t>(__shfl_xor(static_cast<int>(mine), 32));
    mrg[j] = mine < o ? mine : o;
  }
#pragma unroll
  for (int j = 0; j <= K; ++j) top[j] = mrg[j];
  if (!valid) return;
  int selfpos = K + 1;
#pragma unroll
  for (int j = 0; j <= K; ++j)
    if (top[j] != 0xFFFFFFFFu && j0 + static_cast<int>(top[j] & kMask) == jr) selfpos = j;
  uint64_t* out = cand + static_cast<int64_t>(order[r]) * kSeedSlots + slot0;
  // feature k of a staged row is float k / 4 of its float4 k % 4
  float4 self4[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) self4[e] = lds_span4[jr * kRow4 + e];
#pragma unroll
  for (int jj = 0; jj < (K + 4) / 4; ++jj) {
    const int j = 4 * jj + g;
    if (j > K) break;
    uint32_t key = top[4 * jj];
#pragma unroll
    for (int e = 1; e < 4; ++e)
      if (4 * jj + e <= K && g == e) key = top[4 * jj + e];
    const int o = j - (selfpos < j ? 1 : 0);
    if (j == selfpos || o >= K) continue;
    uint64_t v = kKeyMax;
    if (key != 0xFFFFFFFFu) {
      const int js = j0 + static_cast<int>(key & kMask);
      float4 row4[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) row4[e] = lds_span4[js * kRow4 + e];
      // the oracle's operation order: diff = row - self, fmaf over k = 0..11
      float acc = 0.0f;
#pragma unroll
      for (int k = 0; k < D; ++k) {
        const float diff = f4_at(row4[k % 4], k / 4) - f4_at(self4[k % 4], k / 4);
        acc = __builtin_fmaf(diff, diff, acc);
      }
      v = make_key(acc, order[sb + js], 1u);
    }
    out[o] = v;
  }
}

// Per point: the 32 nearest distinct ids among its table candidates, sorted
// with exact keys.  Slots no candidate fills take xorshift ids, stepped +1
// past the point itself and past ids already in the list (n > 33 ids leave
// room), with their exact distances.
__global__ __launch_bounds__(256) void k_mlp_merge(const uint64_t* __restrict__ cand, const float* __restrict__ X,
                                                   int64_t n, int d, uint64_t seed,
                                                   hdb_nnd_element* __restrict__ lists) {
  __shared__ uint64_t s_key[4][64];
  const unsigned w = threadIdx.x >> 6;
  const int64_t p = static_cast<int64_t>(blockIdx.x) * 4 + w;
  if (p >= n) return;  // uniform across the wave; no block barriers below
  const unsigned lane = __lane_id();
  uint64_t key = cand[p * kSeedSlots + lane];
  key = bitonic_group<64>(key);
  const uint64_t prev = shfl_u64(key, (lane + 63) & 63);
  const bool keep = key != kKeyMax && (lane == 0 || (prev >> 1) != (key >> 1));
  const uint64_t bal = __ballot(keep);
  const int pos = __popcll(bal & lanemask_lt());
  const int total = __popcll(bal);
  s_key[w][lane] = kKeyMax;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  if (keep && pos < kK) s_key[w][pos] = key;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  key = s_key[w][lane];
  if (total < kK) {  // uniform
    const float* xp = X + p * d;
    for (int j = total; j < kK; ++j) {
      uint32_t id = static_cast<uint32_t>(xorshift64star(seed + static_cast<uint64_t>(p) * kK + j + 1) %
                                          static_cast<uint64_t>(n));
      for (;;) {  // at most 33 ids are excluded, so this ends
        const bool hit = static_cast<int>(lane) < j && key_id(key) == id;
        if (id != static_cast<uint32_t>(p) && __ballot(hit) == 0) break;
        id = static_cast<uint32_t>((id + 1) % static_cast<uint64_t>(n));
      }
      if (static_cast<int>(lane) == j) key = make_key(d2_any(xp, X + static_cast<int64_t>(id) * d, d), id, 1u);
    }
    key = bitonic_group<32>(key);
  }
  if (lane < static_cast<unsigned>(kK))
    lists[p * kK + lane] = hdb_nnd_element{key_d2(key), static_cast<int32_t>(key_id(key))};
}

}  // namespace hdb

// ------------------------------------------------------------- C ABI --
using namespace hdb;

struct hdb_mlp {
  MlpLayout L;
  float* prm = nullptr;   // device: parameters (FP32 master)
  float* grad = nullptr;  // device: gradient
  float* m = nullptr;
  float* v = nullptr;
  uint8_t* mask = nullptr;  // trainable entries (zero padding excluded)
  int64_t step = 0;
};

namespace {

// Work on the context's second stream inside one call: begin() makes
// stream2 wait for everything queued on `stream`; join() (also run at scope
// exit, so an early error return leaves no work outstanding on stream2)
// makes `stream` wait for stream2.
struct StreamFork {
  hdb_ctx* ctx;
  bool forked = false;
  explicit StreamFork(hdb_ctx* c) : ctx(c) {}
  int begin() {
    HDB_HIP(hipEventRecord(ctx->fork_ev, ctx->stream));
    HDB_HIP(hipStreamWaitEvent(ctx->stream2, ctx->fork_ev, 0));
    forked = true;
    return HDB_OK;
  }
  int join() {
    if (!forked) return HDB_OK;
    forked = false;
    HDB_HIP(hipEventRecord(ctx->join_ev, ctx->stream2));
    HDB_HIP(hipStreamWaitEvent(ctx->stream, ctx->join_ev, 0));
    return HDB_OK;
  }
  ~StreamFork() { (void)join(); }
};

// While alive (and enabled): launches go to stream2 and the per-table slots
// (keys, order, sort and scan scratch, packed weights, permuted points) are
// the second set, so they never alias the buffers of work on `stream`.
struct AltSlots {
  hdb_ctx* ctx;
  hipStream_t saved;
  bool on;
  static void swap_all(hdb_ctx* c) {
    static const Slot a[] = {kSlotMisc1,    kSlotMisc2,   kSlotSortKeys, kSlotSortVals, kSlotSortHist,
                             kSlotSortAux, kSlotScanTmp, kSlotMlpPack,  kSlotSeedX};
    static const Slot b[] = {kSlotAlt0, kSlotAlt1, kSlotAlt2, kSlotAlt3, kSlotAlt4,
                             kSlotAlt5, kSlotAlt6, kSlotAlt7, kSlotAlt8};
    static_assert(sizeof(a) == sizeof(b), "slot pairs");
    for (size_t i = 0; i < sizeof(a) / sizeof(a[0]); ++i) scratch_swap(c, a[i], b[i]);
  }
  AltSlots(hdb_ctx* c, bool enable) : ctx(c), saved(c->stream), on(enable) {
    if (on) {
      ctx->stream = ctx->stream2;
      swap_all(ctx);
    }
  }
  ~AltSlots() {
    if (on) {
      swap_all(ctx);
      ctx->stream = saved;
    }
  }
};

int mlp_alloc(hdb_ctx* ctx, void** p, size_t bytes) {
  if (hipMalloc(p, bytes) != hipSuccess) {
    (void)hipGetLastError();
    return ctx->fail(HDB_ENOMEM, "MLP allocation failed");
  }
  return HDB_OK;
}

// Inference forward Z = f(X) over R rows (packed-weight kernel).
int mlp_infer(hdb_ctx* ctx, hdb_mlp* net, const float* X, int d, int64_t R, float* Z, const InferKeys* ko) {
  const MlpLayout& L = net->L;
  const int nfrag = infer_frags(L.kinp);
  __bf16* packed;
  HDB_CALL(scratch_t(ctx, kSlotMlpPack, static_cast<int64_t>(nfrag) * 512, &packed));
  hipLaunchKernelGGL(k_mlp_pack, dim3(grid_for(static_cast<int64_t>(nfrag) * 64, 256)), dim3(256), 0, ctx->stream,
                     net->prm, L, packed);
  HDB_LAUNCHED();
  const int waves = 8;
  const size_t lds = static_cast<size_t>(nfrag) * 1024 + 272 * sizeof(float);
  const int64_t tiles = (R + 15) / 16;
  const unsigned grid = static_cast<unsigned>(std::max<int64_t>(1, std::min<int64_t>((tiles + waves - 1) / waves, 1024)));
  if (ko)
    hipLaunchKernelGGL(k_mlp_infer<true>, dim3(grid), dim3(waves * 64), lds, ctx->stream, X, d, R, packed, net->prm, L,
                       Z, *ko);
  else
    hipLaunchKernelGGL(k_mlp_infer<false>, dim3(grid), dim3(waves * 64), lds, ctx->stream, X, d, R, packed, net->prm,
                       L, Z, InferKeys{nullptr, 1.0f, 12, nullptr, nullptr});
  HDB_LAUNCHED();
  return HDB_OK;
}

// One Adam step (adam) or one loss-and-gradient evaluation (!adam) of
// `tables` networks of one layout.  Triples come from `lists` with table t's
// stream seeds[t], or are the caller's 3B `rows` (one table).  codes: null,
// or per table the partition codes (null entries: the triple loss).  loss
// (optional, per table) receives each table's loss.
int train_step(hdb_ctx* ctx, hdb_mlp* const* nets, int tables, const float* X, int64_t n, int d,
               const hdb_nnd_element* lists, const int32_t* rows, const uint32_t* const* codes, int64_t B,
               const uint64_t* seeds, float lr, bool adam, double* loss) {
  if (tables < 1 || tables > kMaxTables) return ctx->fail(HDB_EINVAL, "tables must be in 1..8");
  if (rows && tables != 1) return ctx->fail(HDB_EINVAL, "given rows train one table");
  const MlpLayout L = nets[0]->L;
  for (int t = 1; t < tables; ++t)
    if (nets[t]->L.kin != L.kin) return ctx->fail(HDB_EINVAL, "tables of one step share their input width");
  TrainArgs A;
  std::memset(&A, 0, sizeof(A));
  A.L = L;
  A.X = X;
  A.d = d;
  A.n = n;
  A.lists = lists;
  A.given_rows = rows;
  A.B = B;
  A.R = 3 * B;
  A.Rp = (A.R + 31) & ~static_cast<int64_t>(31);
  A.tiles = A.Rp / 16;
  const int regions = (L.kinp / 32) * 4 + 20;
  const int rblocks = (regions + 3) / 4;
  const int64_t nchunks = A.Rp / 32;
  int64_t splits = std::max<int64_t>(1, std::min<int64_t>((1024 + tables * rblocks - 1) / (tables * rblocks), nchunks));
  const int64_t cps = (nchunks + splits - 1) / splits;
  splits = (nchunks + cps - 1) / cps;
  A.splits = static_cast<int>(splits);
  A.chunks_per_split = static_cast<int>(cps);
  A.lr = lr;
  A.adam = adam ? 1 : 0;
  auto up64 = [](int64_t x) { return (x + 63) & ~static_cast<int64_t>(63); };
  const int64_t fz = up64(A.Rp * kOutP), fp = up64(2 * A.Rp * kHid), ft = up64(A.tiles * 16),
                fb = up64(A.tiles * kBiasCols), fl = up64(A.tiles), fw = up64(splits * L.total),
                fm = up64(16), fg = up64(kBiasCols);
  const int64_t fstride = fz + fp + ft + fb + fl + fw + fm + fg;
  const int64_t ba = up64(A.Rp * (L.kinp + 2 * kHid)), bb = up64(A.Rp * (2 * kHid + kOutP));
  const int64_t bstride = ba + bb;
  const int64_t rstride = up64(A.R);
  float* fbase;
  __bf16* bbase;
  int32_t* rbase;
  HDB_CALL(scratch_t(ctx, kSlotMisc0, tables * fstride, &fbase));
  HDB_CALL(scratch_t(ctx, kSlotMisc1, tables * bstride, &bbase));
  HDB_CALL(scratch_t(ctx, kSlotAhKeys2, tables * rstride, &rbase));
  A.Z = fbase, A.s_z = fstride;
  A.P = fbase + fz, A.s_p = fstride;
  A.tsum = fbase + fz + fp, A.s_tsum = fstride;
  A.bsum = fbase + fz + fp + ft, A.s_bsum = fstride;
  A.lsum = fbase + fz + fp + ft + fb, A.s_lsum = fstride;
  A.wpart = fbase + fz + fp + ft + fb + fl, A.s_wpart = fstride;
  A.tmean = A.wpart + fw, A.s_tmean = fstride;
  A.gbias = A.tmean + fm, A.s_gbias = fstride;
  A.opa = bbase, A.s_opa = bstride;
  A.opb = bbase + ba, A.s_opb = bstride;
  A.rows = rbase, A.s_rows = rstride;
  for (int t = 0; t < tables; ++t) {
    hdb_mlp* net = nets[t];
    const int64_t step = net->step + 1;
    A.net[t] = TrainNet{net->prm, net->grad, net->m, net->v, net->mask, codes ? codes[t] : nullptr,
                        seeds ? seeds[t] : 0ull, 1.0f - std::pow(0.9f, static_cast<float>(step)),
                        1.0f - std::pow(0.999f, static_cast<float>(step))};
  }
  const size_t flds = static_cast<size_t>(kTrWaves) * (16 * (L.kinp + 4) + 2 * 16 * (kHid + 4)) * sizeof(float);
  hipLaunchKernelGGL(k_tr_fwd, dim3(grid_for(A.tiles, kTrWaves), tables), dim3(kTrWaves * 64), flds, ctx->stream, A);
  HDB_LAUNCHED();
  hipLaunchKernelGGL(k_tr_tmean, dim3(tables), dim3(256), 0, ctx->stream, A);
  HDB_LAUNCHED();
  const size_t blds = static_cast<size_t>(4) * (16 * 36 + 16 * (kHid + 4) + 16) * sizeof(float);
  hipLaunchKernelGGL(k_tr_bwd, dim3(grid_for(A.tiles, 4), tables), dim3(256), blds, ctx->stream, A);
  HDB_LAUNCHED();
  hipLaunchKernelGGL(k_tr_wgrad, dim3(rblocks, static_cast<unsigned>(splits), tables), dim3(256), 0, ctx->stream, A);
  HDB_LAUNCHED();
  hipLaunchKernelGGL(k_tr_bred, dim3((kBiasCols + 3) / 4, tables), dim3(256), 0, ctx->stream, A);
  HDB_LAUNCHED();
  hipLaunchKernelGGL(k_tr_apply, dim3(grid_for(L.total, 256), tables), dim3(256), 0, ctx->stream, A);
  HDB_LAUNCHED();
  if (adam)
    for (int t = 0; t < tables; ++t) nets[t]->step += 1;
  if (loss) {
    std::vector<float> ls(A.tiles), ts(A.tiles * 16);
    for (int t = 0; t < tables; ++t) {
      HDB_HIP(hipMemcpyAsync(ls.data(), A.lsum + t * fstride, A.tiles * sizeof(float), hipMemcpyDeviceToHost,
                             ctx->stream));
      HDB_HIP(hipMemcpyAsync(ts.data(), A.tsum + t * fstride, A.tiles * 16 * sizeof(float), hipMemcpyDeviceToHost,
                             ctx->stream));
      HDB_HIP(hipStreamSynchronize(ctx->stream));
      double s = 0.0;
      for (float x : ls) s += x;
      if (codes && codes[t]) {
        loss[t] = s;
      } else {
        s /= static_cast<double>(B);
        for (int c = 0; c < kCode; ++c) {
          double m = 0.0;
          for (int64_t tt = 0; tt < A.tiles; ++tt) m += ts[tt * 16 + c];
          m /= static_cast<double>(A.R);
          s += m * m;
        }
        loss[t] = s;
      }
    }
  }
  return HDB_OK;
}

// `steps` Adam steps of `tables` networks; table t draws its triples from
// the stream seed + 97 t (+ 0x100000001 per step of that network).
int train_tables(hdb_ctx* ctx, hdb_mlp* const* nets, int tables, const float* X, int64_t n, int d,
                 const hdb_nnd_element* lists, const uint32_t* const* codes, int steps, int64_t batch, float lr,
                 uint64_t seed, double* final_loss) {
  uint64_t seeds[kMaxTables];
  for (int s = 0; s < steps; ++s) {
    for (int t = 0; t < tables; ++t)
      seeds[t] = seed + 97ull * static_cast<uint64_t>(t) + 0x100000001ull * static_cast<uint64_t>(nets[t]->step);
    HDB_CALL(train_step(ctx, nets, tables, X, n, d, lists, nullptr, codes, batch, seeds, lr, true,
                        s == steps - 1 ? final_loss : nullptr));
  }
  return HDB_OK;
}

}  // namespace

extern "C" {

int hdb_mlp_create(hdb_ctx* ctx, int32_t d_in, uint64_t seed, hdb_mlp** out) {
  if (!ctx || !out || d_in < 1 || d_in > 128) return ctx ? ctx->fail(HDB_EINVAL, "MLP input width must be 1..128") : HDB_EINVAL;
  HDB_HIP(hipSetDevice(ctx->device));
  hdb_mlp* net = new hdb_mlp();
  net->L = mlp_layout(d_in);
  const MlpLayout& L = net->L;
  std::vector<float> h(L.total, 0.0f);
  std::vector<uint8_t> mask(L.total, 0);
  // He-style uniform init from xorshift64*, zero biases; padding stays zero
  uint64_t s = seed * 0x9E3779B97F4A7C15ull + 1;
  auto uni = [&s]() {
    s = xorshift64star(s);
    return static_cast<float>((s >> 11) * (1.0 / 9007199254740992.0)) * 2.0f - 1.0f;
  };
  const float a1 = std::sqrt(6.0f / d_in), a2 = std::sqrt(6.0f / kHid);
  for (int k = 0; k < L.kinp; ++k)
    for (int j = 0; j < kHid; ++j)
      if (k < d_in) {
        h[L.w1 + k * kHid + j] = a1 * uni();
        mask[L.w1 + k * kHid + j] = 1;
      }
  for (int j = 0; j < kHid; ++j) mask[L.b1 + j] = mask[L.b2 + j] = 1;
  for (int k = 0; k < kHid * kHid; ++k) {
    h[L.w2 + k] = a2 * uni();
    mask[L.w2 + k] = 1;
  }
  for (int k = 0; k < kHid; ++k)
    for (int j = 0; j < kCode; ++j) {
      h[L.w3 + k * kOutP + j] = a2 * uni();
      mask[L.w3 + k * kOutP + j] = 1;
    }
  for (int j = 0; j < kCode; ++j) mask[L.b3 + j] = 1;
  int st = HDB_OK;
  if ((st = mlp_alloc(ctx, reinterpret_cast<void**>(&net->prm), L.total * 4)) != HDB_OK ||
      (st = mlp_alloc(ctx, reinterpret_cast<void**>(&net->grad), L.total * 4)) != HDB_OK ||
      (st = mlp_alloc(ctx, reinterpret_cast<void**>(&net->m), L.total * 4)) != HDB_OK ||
      (st = mlp_alloc(ctx, reinterpret_cast<void**>(&net->v), L.total * 4)) != HDB_OK ||
      (st = mlp_alloc(ctx, reinterpret_cast<void**>(&net->mask), L.total)) != HDB_OK) {
    hdb_mlp_destroy(net);
    return st;
  }
  HDB_HIP(hipMemcpy(net->prm, h.data(), L.total * 4, hipMemcpyHostToDevice));
  HDB_HIP(hipMemcpy(net->mask, mask.data(), L.total, hipMemcpyHostToDevice));
  HDB_HIP(hipMemset(net->grad, 0, L.total * 4));
  HDB_HIP(hipMemset(net->m, 0, L.total * 4));
  HDB_HIP(hipMemset(net->v, 0, L.total * 4));
  *out = net;
  return HDB_OK;
}

int hdb_mlp_destroy(hdb_mlp* net) {
  if (!net) return HDB_EINVAL;
  (void)hipFree(net->prm);
  (void)hipFree(net->grad);
  (void)hipFree(net->m);
  (void)hipFree(net->v);
  (void)hipFree(net->mask);
  delete net;
  return HDB_OK;
}

int64_t hdb_mlp_param_count(const hdb_mlp* net) { return net ? net->L.total : -1; }

int hdb_mlp_params(hdb_ctx* ctx, hdb_mlp* net, float* host_in, float* host_out) {
  if (!ctx || !net) return HDB_EINVAL;
  HDB_HIP(hipStreamSynchronize(ctx->stream));
  if (host_in) HDB_HIP(hipMemcpy(net->prm, host_in, net->L.total * 4, hipMemcpyHostToDevice));
  if (host_out) HDB_HIP(hipMemcpy(host_out, net->prm, net->L.total * 4, hipMemcpyDeviceToHost));
  return HDB_OK;
}

int hdb_mlp_forward(hdb_ctx* ctx, hdb_mlp* net, const float* X, int64_t m, int32_t d, float* Z) {
  if (!ctx || !net || !X || !Z || m < 0 || d != net->L.kin) return ctx ? ctx->fail(HDB_EINVAL, "bad forward args") : 1;
  HDB_HIP(hipSetDevice(ctx->device));
  if (m == 0) return HDB_OK;
  return mlp_infer(ctx, net, X, d, m, Z, nullptr);
}

int hdb_mlp_loss_grad(hdb_ctx* ctx, hdb_mlp* net, const float* X, int64_t n, int32_t d, const int32_t* rows,
                      const uint32_t* codes, int64_t batch, double* loss, float* grad_host) {
  if (!ctx || !net || !X || !rows || batch < 1 || d != net->L.kin || n < 1)
    return ctx ? ctx->fail(HDB_EINVAL, "bad loss_grad args") : 1;
  HDB_HIP(hipSetDevice(ctx->device));
  const uint32_t* cp[1] = {codes};
  HDB_CALL(train_step(ctx, &net, 1, X, n, d, nullptr, rows, cp, batch, nullptr, 0.0f, false, loss));
  if (grad_host) {
    HDB_HIP(hipMemcpyAsync(grad_host, net->grad, net->L.total * 4, hipMemcpyDeviceToHost, ctx->stream));
    HDB_HIP(hipStreamSynchronize(ctx->stream));
  }
  return HDB_OK;
}

int hdb_mlp_train(hdb_ctx* ctx, hdb_mlp* net, const float* X, int64_t n, int32_t d, const hdb_nnd_element* lists,
                  const uint32_t* codes, int32_t steps, int32_t batch, float lr, uint64_t seed, double* final_loss) {
  if (!ctx || !net || !X || !lists || n < 2 || steps < 0 || batch < 1 || d != net->L.kin)
    return ctx ? ctx->fail(HDB_EINVAL, "bad train args") : 1;
  HDB_HIP(hipSetDevice(ctx->device));
  Stage st(ctx, "mlp_train");
  const uint32_t* cp[1] = {codes};
  return train_tables(ctx, &net, 1, X, n, d, lists, cp, steps, batch, lr, seed, final_loss);
}

int hdb_mlp_train_tables(hdb_ctx* ctx, hdb_mlp* const* nets, int32_t tables, const float* X, int64_t n, int32_t d,
                         const hdb_nnd_element* lists, const uint32_t* const* codes, int32_t steps, int32_t batch,
                         float lr, uint64_t seed, double* final_loss) {
  if (!ctx || !nets || tables < 1 || tables > kMaxTables || !X || !lists || n < 2 || steps < 0 || batch < 1)
    return ctx ? ctx->fail(HDB_EINVAL, "bad train args") : 1;
  for (int t = 0; t < tables; ++t)
    if (!nets[t] || nets[t]->L.kin != d) return ctx->fail(HDB_EINVAL, "every network must take d inputs");
  HDB_HIP(hipSetDevice(ctx->device));
  Stage st(ctx, "mlp_train");
  return train_tables(ctx, nets, tables, X, n, d, lists, codes, steps, batch, lr, seed, final_loss);
}

int hdb_rp_codes(hdb_ctx* ctx, const float* X, int64_t n, int32_t d, uint64_t seed, uint32_t* codes) {
  if (!ctx || !X || !codes || n < 2 || d < 1) return ctx ? ctx->fail(HDB_EINVAL, "bad rp_codes args") : 1;
  if (n > (1ll << 20)) return ctx->fail(HDB_EUNSUPPORTED, "rp_codes takes at most 2^20 points");
  HDB_HIP(hipSetDevice(ctx->device));
  Stage st(ctx, "rp_codes");
  uint64_t* keys;
  uint32_t* cell;
  int32_t* bounds;
  HDB_CALL(scratch_t(ctx, kSlotSeedCand, n, &keys));
  HDB_CALL(scratch_t(ctx, kSlotMisc1, n, &cell));
  HDB_CALL(scratch_t(ctx, kSlotMisc2, 2 << kCode, &bounds));
  HDB_CALL(fill_i32(ctx, reinterpret_cast<int32_t*>(codes), n, 0));
  const unsigned g = grid_for(n, 256);
  for (int l = 0; l < kCode; ++l) {
    hipLaunchKernelGGL(k_rp_keys, dim3(g), dim3(256), 0, ctx->stream, X, n, d, l, seed, codes, keys);
    HDB_LAUNCHED();
    HDB_CALL(radix_sort_u64(ctx, keys, n, 20, 52 + l + 1));
    hipLaunchKernelGGL(k_rp_cells, dim3(g), dim3(256), 0, ctx->stream, keys, n, cell);
    HDB_LAUNCHED();
    const int64_t ncell = 1ll << l;
    HDB_CALL(segment_bounds(ctx, cell, n, ncell, bounds, bounds + ncell));
    hipLaunchKernelGGL(k_rp_split, dim3(g), dim3(256), 0, ctx->stream, keys, n, bounds, bounds + ncell, codes);
    HDB_LAUNCHED();
  }
  return HDB_OK;
}

// out[i][c] = X[rows[i]][c]; a row outside [0, n) gives zeros and sets *bad.
__global__ __launch_bounds__(256) void k_gather_rows(const float* __restrict__ X, int64_t n, int d,
                                                     const int64_t* __restrict__ rows, int64_t m,
                                                     float* __restrict__ out, int32_t* __restrict__ bad) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= m * d) return;
  const int64_t i = t / d;
  const int c = static_cast<int>(t - i * d);
  const int64_t r = rows[i];
  const bool ok = r >= 0 && r < n;
  out[t] = ok ? X[r * d + c] : 0.0f;
  if (!ok && c == 0) *bad = 1;  // a plain store: only zero / nonzero is read
}

int hdb_gather_rows(hdb_ctx* ctx, const float* X, int64_t n, int32_t d, const int64_t* rows, int64_t m, float* out) {
  if (!ctx) return 1;
  if (!X || !rows || !out || n < 1 || d < 1 || m < 0) return ctx->fail(HDB_EINVAL, "bad gather_rows arguments");
  if (m == 0) return HDB_OK;
  HDB_HIP(hipSetDevice(ctx->device));
  int32_t* bad;
  HDB_CALL(scratch_t(ctx, kSlotGatherFlag, 1, &bad));
  HDB_CALL(fill_i32(ctx, bad, 1, 0));
  hipLaunchKernelGGL(k_gather_rows, dim3(grid_for(m * d, 256)), dim3(256), 0, ctx->stream, X, n, d, rows, m, out, bad);
  HDB_LAUNCHED();
  int32_t flag = 0;
  HDB_CALL(read_i32(ctx, bad, &flag));
  if (flag) return ctx->fail(HDB_EINVAL, "gather_rows: a row id outside [0, n)");
  return HDB_OK;
}

int hdb_learned_init(hdb_ctx* ctx, hdb_mlp* const* nets, int32_t tables, const float* X, int64_t n, int32_t d,
                     int32_t window, uint64_t seed, hdb_nnd_element* lists) {
  if (!ctx || !nets || tables < 1 || tables > kSeedTables || !X || !lists || n < 34)
    return ctx ? ctx->fail(HDB_EINVAL, "bad learned_init args (1..8 networks, n must exceed 33)") : 1;
  if (window != 128 && window != 256 && window != 512) return ctx->fail(HDB_EINVAL, "window must be 128, 256 or 512");
  for (int t = 0; t < tables; ++t)
    if (!nets[t] || nets[t]->L.kin != d) return ctx->fail(HDB_EINVAL, "network input width differs from d");
  if (n >= (1ll << 31)) return ctx->fail(HDB_EUNSUPPORTED, "more than 2^31 points");
  HDB_HIP(hipSetDevice(ctx->device));
  Stage st(ctx, "learned_init");
  const int keep = tables <= 4 ? 16 : 8;  // nearest window entries kept per table
  const int qbits = proj_bits(n);
  float* dirs;
  uint64_t* cand;
  HDB_CALL(scratch_t(ctx, kSlotBfTmp, static_cast<int64_t>(tables) * d, &dirs));
  HDB_CALL(scratch_t(ctx, kSlotSeedCand, n * kSeedSlots, &cand));
  // per table: a unit direction for the order inside a bucket, Box-Muller
  // from xorshift64*
  std::vector<float> hd(static_cast<size_t>(tables) * d);
  uint64_t s = seed * 0x2545F4914F6CDD1Dull + 7;
  for (int t = 0; t < tables; ++t) {
    double nrm = 0.0;
    for (int k = 0; k < d; ++k) {
      s = xorshift64star(s);
      const double u1 = ((s >> 11) + 1.0) / 9007199254740993.0;
      s = xorshift64star(s);
      const double u2 = (s >> 11) / 9007199254740992.0;
      hd[t * d + k] = static_cast<float>(std::sqrt(-2.0 * std::log(u1)) * std::cos(6.283185307179586 * u2));
      nrm += static_cast<double>(hd[t * d + k]) * hd[t * d + k];
    }
    for (int k = 0; k < d; ++k) hd[t * d + k] = static_cast<float>(hd[t * d + k] / std::sqrt(nrm));
  }
  HDB_HIP(hipMemcpyAsync(dirs, hd.data(), hd.size() * sizeof(float), hipMemcpyHostToDevice, ctx->stream));
  if (tables * keep < kSeedSlots) HDB_CALL(fill_u64(ctx, cand, n * kSeedSlots, kKeyMax));
  const size_t lds = static_cast<size_t>(kSeedPts + window + 1) * (d + 1) * sizeof(float);
  const bool staged = lds <= 80 * 1024;
  const dim3 grid(static_cast<unsigned>(grid_for(n, kSeedPts)));
  const dim3 gridm(static_cast<unsigned>(grid_for(n, kSmPts)));
  const bool mfma_search = d == 12 && n >= window + 32 && (reinterpret_cast<uintptr_t>(X) & 15) == 0;
  // Tables alternate between the context's two streams, each with its own
  // keys, sort scratch and packed weights, so one table's sort (a few
  // hundred blocks) overlaps the other's network and window search; the
  // window searches write disjoint candidate slots.
  StreamFork fork(ctx);
  HDB_CALL(fork.begin());
  for (int t = 0; t < tables; ++t) {
    AltSlots alt(ctx, (t & 1) != 0);
    uint32_t *keys, *order;
    float* Xs = nullptr;
    HDB_CALL(scratch_t(ctx, kSlotMisc1, n, &keys));
    HDB_CALL(scratch_t(ctx, kSlotMisc2, n, &order));
    // x.u range: 64 covers the spread of a unit direction over typical data
    const InferKeys ko{dirs + t * d, 64.0f, qbits, keys, order};
    HDB_CALL(mlp_infer(ctx, nets[t], X, d, n, nullptr, &ko));
    // the sorted order stays wherever the last pass left it (no copy back)
    uint32_t *skeys, *ids;
    HDB_CALL(radix_sort_u32_u32_out(ctx, keys, order, n, 0, kCode + qbits, &skeys, &ids));
    if (!mfma_search) {  // the other searches read the points in bucket order
      HDB_CALL(scratch_t(ctx, kSlotSeedX, n * d, &Xs));
      hipLaunchKernelGGL(k_mlp_permute, dim3(grid_for(n * d, 256)), dim3(256), 0, ctx->stream, X, ids, n, d, Xs);
      HDB_LAUNCHED();
    }
    const int slot0 = t * keep;
#define HDB_SEED(D_, W_, K_, ST_)                                                                                   \
  hipLaunchKernelGGL((k_mlp_seed<D_, W_, K_, ST_>), grid, dim3(kSeedPts), ST_ ? lds : 0, ctx->stream, Xs, ids, n, d, \
                     slot0, cand)
#define HDB_SEED_K(D_, W_, ST_)                 \
  do {                                          \
    if (keep == 16) HDB_SEED(D_, W_, 16, ST_);  \
    else HDB_SEED(D_, W_, 8, ST_);              \
  } while (0)
#define HDB_SEED_W(D_, ST_)                                \
  do {                                                     \
    if (window == 128) HDB_SEED_K(D_, 128, ST_);           \
    else if (window == 256) HDB_SEED_K(D_, 256, ST_);      \
    else HDB_SEED_K(D_, 512, ST_);                         \
  } while (0)
#define HDB_SEED4(D_, W_)                                                                                         \
  do {                                                                                                            \
    const size_t l4 = static_cast<size_t>(kSeedPts + W_ + 1) * ((((D_) / 4) & 1) ? (D_) : (D_) + 4) * 4 +       \
                      static_cast<size_t>(kSeedPts + W_ + 1) * 4;                                                 \
    if (keep == 16)                                                                                               \
      hipLaunchKernelGGL((k_mlp_seed4<D_, W_, 16>), grid, dim3(kSeedPts), l4, ctx->stream, Xs, ids, n, slot0, cand); \
    else                                                                                                          \
      hipLaunchKernelGGL((k_mlp_seed4<D_, W_, 8>), grid, dim3(kSeedPts), l4, ctx->stream, Xs, ids, n, slot0, cand);  \
  } while (0)
#define HDB_SEED4_W(D_)                 \
  do {                                  \
    if (window == 128) HDB_SEED4(D_, 128); \
    else if (window == 256) HDB_SEED4(D_, 256); \
    else HDB_SEED4(D_, 512);            \
  } while (0)
#define HDB_SEEDM(W_)                                                                                         \
  do {                                                                                                        \
    if (keep == 16)                                                                                           \
      hipLaunchKernelGGL((k_mlp_seed_mfma<W_, 16>), gridm, dim3(64 * kSmWaves), seed_mfma_lds(W_), ctx->stream, \
                         X, ids, n, slot0, cand);                                                             \
    else                                                                                                      \
      hipLaunchKernelGGL((k_mlp_seed_mfma<W_, 8>), gridm, dim3(64 * kSmWaves), seed_mfma_lds(W_), ctx->stream,  \
                         X, ids, n, slot0, cand);                                                             \
  } while (0)
    if (mfma_search) {
      if (window == 128) HDB_SEEDM(128);
      else if (window == 256) HDB_SEEDM(256);
      else HDB_SEEDM(512);
    } else if (d == 12) HDB_SEED4_W(12);
    else if (d == 32) HDB_SEED4_W(32);
    else if (staged) HDB_SEED_W(0, true);
    else HDB_SEED_W(0, false);
#undef HDB_SEEDM
#undef HDB_SEED4_W
#undef HDB_SEED4
#undef HDB_SEED_W
#undef HDB_SEED_K
#undef HDB_SEED
    HDB_LAUNCHED();
  }
  HDB_CALL(fork.join());
  hipLaunchKernelGGL(k_mlp_merge, dim3(grid_for(n, 4)), dim3(256), 0, ctx->stream, cand, X, n, d, seed, lists);
  HDB_LAUNCHED();
  return HDB_OK;
}

}  // extern "C"
