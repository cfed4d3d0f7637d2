// Candidate-model scoring on the matrix cores, with every decision and every
// summed residual taken in FP64.
//
// MSAC scoring (scoring_function.h:137-233) of a model over a pair's points is
// a dense contraction: for the Sampson distance (fundamental_estimator.h:
// 195-222) the numerator is C = x2^T F x1 = vec(F) . z with
// z = x2 (x) x1 = (x2x1, x2y1, x2, y2x1, y2y1, y2, x1, y1, 1), and the
// denominator is linear in 11 squared terms.  For
// the homography transfer error (homography_estimator.h:181-199) the
// quantities P = x2 w - u, Q = y2 w - v and W = w (u, v, w = H x1) are linear
// in z, with r^2 = (P^2 + Q^2) / W^2.  So one wave scores 32 models x 32
// points per step as two (Sampson) or three (transfer) 32x32 MFMA tiles
// whose reduction dimension holds the terms.
//
// Precision.  Points are scaled by a per-pair power of two 1/s (exact) so
// that |x'| <= 1, models to F'' = S F S / m (S = diag(s, s, 1), m = max |.|,
// so |F''| <= 1; the inlier test C^2 < tau^2 den becomes C''^2 <
// (tau / s)^2 den'' for the Sampson distance, and likewise for the transfer
// error).  Each operand is split into FP16 hi + lo parts and the MFMA sums
// hi*hi + hi*lo + lo*hi in FP32 (27 terms, padded to 32: two 32x32x16 MFMAs
// per quantity).  The error of a quantity q = c . z against its exact value is
// below 2^-18.5 sum_t |c_t||z_t| + 2^-25 (9 + sum_t |z_t|) (operand splits
// 2^-22 relative each, the dropped lo*lo term 2^-22, FP32 rounding of z
// 2^-24, FP32 accumulation of 27 exact products 27 * 2^-24, FP16 subnormal
// spacing 2^-24); with |c_t| <= 1 the kernel uses delta = 2^-17 S + 2^-20,
// S the sum of |z_t| over the terms the quantity reads (at most (1 + |x1| +
// |y1|) (1 + |x2| + |y2|)).  The denominators |(F x1)_01|^2 + |(F^T x2)_01|^2
// and W^2 are linear forms too, in the 11 squared terms (x1^2, x1 y1, y1^2, x1,
// y1, the same of the second image, 1); a quarter, D, has |coefficients| <= 1,
// and 11 + 10 + 11 products fill the 32 (the lo of the 1 is 0), so its bound is
// the same with 32 terms: dD = 2^-17 S + 2^-20.
//
// A point is dropped for a model only when the bounds prove it an outlier.  With
// X = tau''^2 times the denominator (= 4 tau''^2 D), sqrt(C^2) > sqrt(X) follows
// from c^2 > (1 + h) X + (1 + 1/h) dC^2 for the computed c, |c - C| <= dC, and
// any h > 0 (h = 2^-4 here; the transfer error's (P, Q) likewise, where sqrt(2)
// times the error of each stays below the same dC).  So the test is, with the
// pair's scales sigma and kappa = 4 tau''^2 (1 + 2^-14) (1 + h) sigma^2 inside
// the model's operands,
//   c^2 > d + slack,  slack = (1 + 2^-14) [max(kappa, 1) dD + (1 + 1/h) (sigma dC)^2],
// c from sigma C, d from kappa D, one slack per point, which is the product's
// initial accumulator (the factors 1 + 2^-14 cover the FP32 rounding of the
// slack, of its way through the accumulator, 33 * 2^-23, and of the FP64
// decision).  The test is one multiply-add whose sign is the answer; no operand
// is a NaN (models and points that are not finite have zero operands, and a
// positive slack drops nothing).  Every other point -- all inliers and every
// point near the threshold -- is evaluated by the FP64 routines of the FP64 kernel
// (f_sampson_parts with its guard band, f_sq_sampson, f_sq_symmetric,
// h_sq_residual) and the MSAC value is accumulated in ascending point order
// on the model's lane.  Counts, values and symmetric counts are therefore the
// FP64 kernel's bits.
//
// What bounds the two passes: the rejection its vector instructions (a
// multiply-add and a shift per 64 models x points, beside the matrix units'
// 128 cycles per 32 x 32) and, near that, the points' operands from the caches
// (hence 64 models per wave); the exact pass the latency of the queued points'
// loads and the in-order sums.  Measured on MI355X, 32 essential pairs of
// 10,000 points, ms per call.  Rejection: 248 with ten products, ballots and
// selects per tile, 158 with four products and lane writes of ballots (four
// streams at once); the latter 156 and this form 96 with one stream.  Exact
// pass: 184 with a walk over single mask bits, 74 with a word per lane (four
// streams) and 38 with one, 30 with the queue in 16 bits.
#include "dev_common.hpp"
#include "kernels.hpp"
#include "mx_rules.hpp"

namespace gcr {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

namespace {

constexpr int kCompactPerBlock = 2048;  // slots per block of the ordered compaction
// The exact pass's grid: the workgroups that are resident at 70 VGPRs, seven
// waves per SIMD (2,048 workgroups, an eighth of them alone in a second round,
// took 74.6 ms where these take 60.4).
constexpr int kMxExactBlocks = 1792;
// list entries per rejection + exact pass: as many as keep the segment's
// candidate masks within kMxMaskBudget bytes, between kMxSegMin and
// kMxSegMax (each segment costs three launches; the masks bound the memory)
constexpr int64_t kMxSegMin = 65536, kMxSegMax = 1048576;
constexpr int64_t kMxMaskBudget = 512ll << 20;
// The rejection's grid: four waves per SIMD are resident (126 VGPRs).  A work item starts
// with four dependent loads (entry, pair, sizes, operands: about 3,000 cycles
// against about 500 per 32 points), so the points are cut into only as many
// slices as one round of the grid's waves takes, by the list's length, which
// only the device knows; from half as many tiles as waves on, four rounds (their
// last one is then a small part).  A slice is a multiple of kMxSliceMin points,
// the four mask words of one store.
constexpr int kMxRejectBlocks = 1024;
constexpr int kMxSliceMin = 128;
constexpr int kMxTile = 64;             // list entries per work item
constexpr int64_t kMxPlaneHalves = 16;  // 16-bit words of a point in one operand plane
constexpr int kNumXcd = 8;

__device__ __forceinline__ f32x16 mfma16(const h8& a, const h8& b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ f32x16 zero16() {
  f32x16 z;
#pragma unroll
  for (int j = 0; j < 16; ++j) z[j] = 0.0f;
  return z;
}

}  // namespace

// ---- per-pair scale and per-point operands ------------------------------------

// 1 / s per pair: s = the smallest power of two >= max |coordinate| of the
// pair's points (1 when that is 0 or not finite).
__global__ void __launch_bounds__(256) k_mx_pair_scale(const double* __restrict__ pts,
                                                       const int64_t* __restrict__ pair_pt_off,
                                                       const int32_t* __restrict__ pair_n, int num_pairs,
                                                       double* __restrict__ inv_scale) {
  __shared__ double red[4];
  const int p = blockIdx.x;
  if (p >= num_pairs) return;
  const double* P = pts + 4 * pair_pt_off[p];
  const int64_t n4 = 4 * (int64_t)pair_n[p];
  double m = 0.0;
  for (int64_t i = threadIdx.x; i < n4; i += blockDim.x) {
    const double v = fabs(P[i]);
    m = (v > m || v != v) ? v : m;
  }
  for (int s = 32; s >= 1; s >>= 1) {
    const double o = __shfl_down(m, s, 64);
    m = (o > m || o != o) ? o : m;
  }
  if (lane_id() == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    double mm = 0.0;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) mm = (red[w] > mm || red[w] != red[w]) ? red[w] : mm;
    double inv = 1.0;
    if (mm > 0.0 && mm <= 1e300) {
      int e = 0;
      const double f = frexp(mm, &e);  // mm = f 2^e, f in [0.5, 1)
      (void)f;
      inv = ldexp(1.0, -e);             // 2^e >= mm
    }
    inv_scale[p] = inv;
  }
}

// k of the reduction dimension of a quantity of T terms -> (hi, lo) element:
// k < T hi*hi of term k, then hi(coef)*lo(z) of the terms but the last when L is
// T - 1 (its z is 1, whose lo is 0), then lo(coef)*hi(z), zero beyond.
template <int T, int L>
__device__ __forceinline__ _Float16 k_elem(const _Float16* first, const _Float16* second, const _Float16* third,
                                           int k) {
  return k < T ? first[k] : (k < T + L ? second[k - T] : (k < 2 * T + L ? third[k - T - L] : (_Float16)0.0f));
}

// Per point: the operand slices of both lane halves (k order, FP16) of z and of
// the squared terms d; a plane per MFMA, so that a wave's load of 32 points is
// one contiguous kilobyte.  A point outside |x'| <= 1 (only where the pair's
// coordinates are not all finite) gets zeros: nothing is dropped for it.
__global__ void __launch_bounds__(256) k_mx_points(const double* __restrict__ pts,
                                                   const int32_t* __restrict__ pt_pair,
                                                   const double* __restrict__ inv_scale, int64_t total,
                                                   uint16_t* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= total) return;
  const double is = inv_scale[pt_pair[i]];
  const double x1 = pts[4 * i] * is, y1 = pts[4 * i + 1] * is, x2 = pts[4 * i + 2] * is, y2 = pts[4 * i + 3] * is;
  const bool ok = fabs(x1) <= 1.0 && fabs(y1) <= 1.0 && fabs(x2) <= 1.0 && fabs(y2) <= 1.0;
  double zd[9], dd[11];
  mx_terms(x1, y1, x2, y2, zd, dd);
  h8* const o = reinterpret_cast<h8*>(out);
  _Float16 hi[11], lo[11];
#pragma unroll
  for (int t = 0; t < 9; ++t) {
    const float z = ok ? (float)zd[t] : 0.0f;
    hi[t] = (_Float16)z;
    lo[t] = (_Float16)(z - (float)hi[t]);
  }
#pragma unroll
  for (int kh = 0; kh < 2; ++kh)
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
      h8 v;
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = k_elem<9, 9>(hi, lo, hi, 16 * kh + 8 * hf + e);
      o[(kh * total + i) * 2 + hf] = v;
    }
#pragma unroll
  for (int t = 0; t < 11; ++t) {
    const float z = ok ? (float)dd[t] : 0.0f;
    hi[t] = (_Float16)z;
    lo[t] = (_Float16)(z - (float)hi[t]);
  }
#pragma unroll
  for (int kh = 0; kh < 2; ++kh)
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
      h8 v;
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = k_elem<11, 10>(hi, lo, hi, 16 * kh + 8 * hf + e);
      o[((2 + kh) * total + i) * 2 + hf] = v;
    }
}

// Per point of [first, first + count): the slack of its test under its pair's
// threshold (the plane behind the operands).
__global__ void __launch_bounds__(256) k_mx_slack(const double* __restrict__ pts, const int32_t* __restrict__ pt_pair,
                                                  const double* __restrict__ pair_sq_thr,
                                                  const double* __restrict__ inv_scale, int64_t first, int64_t count,
                                                  float* __restrict__ slack) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= count) return;
  const int64_t i = first + t;
  const int p = pt_pair[i];
  const double is = inv_scale[p];
  const MxScale sc = mx_scale(pair_sq_thr[p], is);
  slack[i] = mx_slack(sc, pts[4 * i] * is, pts[4 * i + 1] * is, pts[4 * i + 2] * is, pts[4 * i + 3] * is);
}

// ---- ordered compaction of the active model slots ------------------------------

// Pass 1: inactive slots get their empty result; per block, the number of
// active slots.
__global__ void __launch_bounds__(256) k_mx_count(const int8_t* __restrict__ active, int64_t num_models,
                                                  int32_t* __restrict__ counts, double* __restrict__ values,
                                                  int32_t* __restrict__ sym_counts, int32_t* __restrict__ blk) {
  __shared__ int32_t part[4];
  const int64_t s0 = (int64_t)blockIdx.x * kCompactPerBlock;
  int c = 0;
  for (int e = 0; e < kCompactPerBlock / 256; ++e) {
    const int64_t s = s0 + (int64_t)e * 256 + threadIdx.x;
    if (s < num_models) {
      if (active[s] == 2) {
        ++c;
      } else {
        counts[s] = -1;
        values[s] = 0.0;
        if (sym_counts) sym_counts[s] = 0;
      }
    }
  }
  for (int s = 32; s >= 1; s >>= 1) c += __shfl_down(c, s, 64);
  if (lane_id() == 0) part[threadIdx.x >> 6] = c;
  __syncthreads();
  if (threadIdx.x == 0) blk[blockIdx.x] = part[0] + part[1] + part[2] + part[3];
}

// Pass 2 (one block): exclusive scan of the block counts; the total goes to
// *list_count.
__global__ void __launch_bounds__(1024) k_mx_scan(int32_t* __restrict__ blk, int nblk,
                                                  uint32_t* __restrict__ list_count) {
  __shared__ int32_t buf[1024];
  __shared__ int32_t carry;
  if (threadIdx.x == 0) carry = 0;
  __syncthreads();
  for (int base = 0; base < nblk; base += 1024) {
    const int i = base + (int)threadIdx.x;
    const int v = i < nblk ? blk[i] : 0;
    buf[threadIdx.x] = v;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {
      const int t = threadIdx.x >= (unsigned)off ? buf[threadIdx.x - off] : 0;
      __syncthreads();
      buf[threadIdx.x] += t;
      __syncthreads();
    }
    if (i < nblk) blk[i] = carry + buf[threadIdx.x] - v;
    __syncthreads();
    if (threadIdx.x == 1023) carry += buf[1023];
    __syncthreads();
  }
  if (threadIdx.x == 0) *list_count = (uint32_t)carry;
}

// Pass 3: each block writes its active slots, in slot order, from its offset.
__global__ void __launch_bounds__(256) k_mx_write(const int8_t* __restrict__ active, int64_t num_models,
                                                  const int32_t* __restrict__ blk, int32_t* __restrict__ list) {
  __shared__ int32_t wbase[4];
  __shared__ int32_t run;
  if (threadIdx.x == 0) run = blk[blockIdx.x];
  __syncthreads();
  const int64_t s0 = (int64_t)blockIdx.x * kCompactPerBlock;
  const int w = threadIdx.x >> 6;
  for (int e = 0; e < kCompactPerBlock / 256; ++e) {
    const int64_t s = s0 + (int64_t)e * 256 + threadIdx.x;
    const bool act = s < num_models && active[s] == 2;
    const uint64_t b = ballot64(act);
    if (lane_id() == 0) wbase[w] = __popcll(b);
    __syncthreads();
    int before = run;
    for (int k = 0; k < w; ++k) before += wbase[k];
    if (act)
      list[before + __builtin_amdgcn_mbcnt_hi((uint32_t)(b >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)b, 0u))] =
          (int32_t)s;
    __syncthreads();
    if (threadIdx.x == 0) run += wbase[0] + wbase[1] + wbase[2] + wbase[3];
    __syncthreads();
  }
}

// ---- per-model operands -----------------------------------------------------------

// One thread per (list entry of the segment, lane half): the entry's scaled,
// normalised coefficient vectors split into FP16 hi / lo and laid out as the
// MFMA operand slices of that lane half (NQ quantities x 2 MFMAs x 8).  A
// zero, inf or NaN model gets zero operands (mx_normalise; nothing is rejected
// for it: the sign of a NaN would decide otherwise).
template <int KIND>
__global__ void __launch_bounds__(256) k_mx_coefs(const double* __restrict__ pair_sq_thr,
                                                  const double* __restrict__ pair_inv_scale,
                                                  const double* __restrict__ models,
                                                  const int32_t* __restrict__ model_pair,
                                                  const int32_t* __restrict__ list,
                                                  const uint32_t* __restrict__ list_count, int64_t seg_begin,
                                                  int64_t seg_len, h8* __restrict__ coefs, int slots_per) {
  constexpr int NQ = KIND == 1 ? 2 : 3;
  const int64_t total = (int64_t)*list_count;
  if (seg_begin >= total) return;
  const int64_t seg_n = total - seg_begin < seg_len ? total - seg_begin : seg_len;
  const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= 2 * seg_n) return;
  const int64_t e = g >> 1;
  const int hf = (int)(g & 1);
  const int64_t slot = list[seg_begin + e];
  const int p = model_pair[slots_per == 1 ? slot : slot / slots_per];
  double M[9];
#pragma unroll
  for (int k = 0; k < 9; ++k) M[k] = models[9 * slot + k];
  const double is = pair_inv_scale[p];
  const double s = 1.0 / is;  // a power of two: exact
  const MxScale ts = mx_scale(pair_sq_thr[p], is);
  double Fs[9];
  mx_normalise<KIND>(M, s, ts.on, Fs);
  double cq[2][9], dq[11];
  mx_quantities<KIND>(Fs, cq);
  mx_denominator<KIND>(Fs, dq);
  h8* out = coefs + (e * 2 + hf) * (2 * NQ);
  _Float16 hi[11], lo[11];
#pragma unroll
  for (int q = 0; q + 1 < NQ; ++q) {
#pragma unroll
    for (int k = 0; k < 9; ++k) {
      const double v = cq[q][k] * ts.sigma;
      hi[k] = (_Float16)v;
      lo[k] = (_Float16)(v - (double)hi[k]);
    }
#pragma unroll
    for (int kh = 0; kh < 2; ++kh) {
      h8 v;
#pragma unroll
      for (int x = 0; x < 8; ++x)
        v[x] = hf ? k_elem<9, 9>(hi, hi, lo, 16 * kh + 8 + x) : k_elem<9, 9>(hi, hi, lo, 16 * kh + x);
      out[2 * q + kh] = v;
    }
  }
#pragma unroll
  for (int k = 0; k < 11; ++k) {
    const double v = dq[k] * ts.kappa;
    hi[k] = (_Float16)v;
    lo[k] = (_Float16)(v - (double)hi[k]);
  }
#pragma unroll
  for (int kh = 0; kh < 2; ++kh) {
    h8 v;
#pragma unroll
    for (int x = 0; x < 8; ++x)
      v[x] = hf ? k_elem<11, 10>(hi, hi, lo, 16 * kh + 8 + x) : k_elem<11, 10>(hi, hi, lo, 16 * kh + x);
    out[2 * NQ - 2 + kh] = v;
  }
}

// ---- phase 1: rejection on the matrix cores ---------------------------------------

// Work item (tile t, slice j): the 64 list entries 64 t .. 64 t + 63 of the
// segment (slot order, so the entries of one pair are adjacent; a tile that
// spans pairs is handled pair by pair) against points slice j .. slice j + slice
// - 1 of their pair.  The points are the products' rows and the models their
// columns, and row 8 (j / 4) + 4 hf + (j % 4), accumulator slot j of lane half
// hf, holds point 16 hf + j of the 32: a lane's slots are consecutive points of
// its own model, the sign of each slot's test is shifted into the lane's mask
// word, and one exchange of lane halves completes the words of entries e0 + lane
// (bit b of a word: point base + b must be evaluated in FP64).  The points'
// slack is the initial accumulator of the denominator.  Words of points at or
// beyond the pair's n are zero up to the next multiple of four words.
template <int KIND>
__global__ void __launch_bounds__(256, KIND == 1 ? 4 : 3) k_mx_reject(
    const int64_t* __restrict__ pair_pt_off, const int32_t* __restrict__ pair_n, const uint16_t* __restrict__ mxp,
    int64_t mx_total, const h8* __restrict__ coefs, const int32_t* __restrict__ model_pair,
    const int32_t* __restrict__ list, const uint32_t* __restrict__ list_count, int64_t seg_begin, int64_t seg_len,
    int max_n, int words, uint32_t* __restrict__ mask, int slots_per) {
  constexpr int NQ = KIND == 1 ? 2 : 3;
  struct __attribute__((packed, aligned(4))) F4 {
    float v[4];
  };
  const int lane = lane_id();
  const int hf = lane >> 5, r = lane & 31;
  const int row_pt = 16 * ((r >> 2) & 1) + 4 * (r >> 3) + (r & 3);
  const int64_t total = (int64_t)*list_count;
  if (seg_begin >= total) return;
  const int64_t seg_n = total - seg_begin < seg_len ? total - seg_begin : seg_len;
  const int tiles = (int)((seg_n + kMxTile - 1) / kMxTile), waves = (int)gridDim.x * 4;
  int slices = 2 * tiles <= waves ? waves / tiles : (4 * waves + tiles - 1) / tiles;
  const int slice = ((max_n + slices - 1) / slices + kMxSliceMin - 1) / kMxSliceMin * kMxSliceMin;
  slices = (max_n + slice - 1) / slice;
  const int64_t items = (int64_t)tiles * slices;
  // gridDim.x is a multiple of kNumXcd: workgroup b runs on XCD b % kNumXcd,
  // which takes a contiguous range of items (adjacent items share a pair)
  const int xcd = (int)(blockIdx.x % kNumXcd);
  const int64_t waves_per_xcd = (int64_t)(gridDim.x / kNumXcd) * 4;
  const int64_t w = (int64_t)(blockIdx.x / kNumXcd) * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t lo_u = items * xcd / kNumXcd, hi_u = items * (xcd + 1) / kNumXcd;
  for (int64_t u = lo_u + w; u < hi_u; u += waves_per_xcd) {
    const int64_t t = u / slices;
    const int first = slice * (int)(u - t * slices);
    const int64_t e0 = kMxTile * t;  // within the segment
    const int cnt_all = (int)(seg_n - e0 < kMxTile ? seg_n - e0 : kMxTile);
    const int64_t slot = lane < cnt_all ? (int64_t)list[seg_begin + e0 + lane] : -1;
    const int my_pair = slot >= 0 ? model_pair[slots_per == 1 ? slot : slot / slots_per] : -1;
    uint32_t* __restrict__ my_mask = mask + (e0 + lane) * (int64_t)words;
    int done = 0;
    while (done < cnt_all) {
      const int p = __builtin_amdgcn_readlane(my_pair, done);
      const bool mine = lane >= done && my_pair == p;
      const int sub_end = done + __popcll(ballot64(mine));
      const int n = pair_n[p];
      if (first < n) {
        // the models' operands (columns 32 s + r, half hf); columns of other
        // pairs compute what nothing reads
        h8 B[2][NQ][2];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          const int e = 32 * s + r < cnt_all ? 32 * s + r : cnt_all - 1;
          const h8* __restrict__ my_coefs = coefs + ((e0 + e) * 2 + hf) * (2 * NQ);
#pragma unroll
          for (int q = 0; q < NQ; ++q)
#pragma unroll
            for (int kh = 0; kh < 2; ++kh) B[s][q][kh] = my_coefs[2 * q + kh];
        }
        const int64_t off = pair_pt_off[p];
        const h8* __restrict__ Z = reinterpret_cast<const h8*>(mxp) + 2 * off + hf;
        const float* __restrict__ K = reinterpret_cast<const float*>(mxp + kMxPlaneHalves * 4 * mx_total) + off;
        const int last = first + slice < n ? first + slice : n;
#pragma unroll 1
        for (int base = first; base < last; base += 128) {
          uint32_t wd[4];
#pragma unroll 1
          for (int k = 0; k < 4; ++k) {
            const int b = base + 32 * k;
            uint32_t word = 0;
            if (b < last) {
              // rows beyond the pair read its last point; their bits are cut below
              const int i = b + row_pt < n ? b + row_pt : n - 1;
              const h8 z0 = Z[2 * i], z1 = Z[2 * (mx_total + i)], d0 = Z[2 * (2 * mx_total + i)],
                       d1 = Z[2 * (3 * mx_total + i)];
              f32x16 slack;
#pragma unroll
              for (int j = 0; j < 16; j += 4) {
                const F4 v = *reinterpret_cast<const F4*>(K + b + 16 * hf + j);
#pragma unroll
                for (int x = 0; x < 4; ++x) slack[j + x] = v.v[x];
              }
              uint32_t half[2];
#pragma unroll
              for (int s = 0; s < 2; ++s) {
                f32x16 den = mfma16(d0, B[s][NQ - 1][0], slack);
                f32x16 c = mfma16(z0, B[s][0][0], zero16());
                den = mfma16(d1, B[s][NQ - 1][1], den);
                c = mfma16(z1, B[s][0][1], c);
                uint32_t bits = 0;
                if constexpr (KIND == 1) {
#pragma unroll
                  for (int j = 15; j >= 0; --j)
                    bits = __builtin_amdgcn_alignbit(
                        bits, __builtin_bit_cast(uint32_t, __builtin_fmaf(-c[j], c[j], den[j])), 31);
                } else {
                  f32x16 c2 = mfma16(z0, B[s][1][0], zero16());
                  c2 = mfma16(z1, B[s][1][1], c2);
#pragma unroll
                  for (int j = 15; j >= 0; --j)
                    bits = __builtin_amdgcn_alignbit(
                        bits,
                        __builtin_bit_cast(uint32_t,
                                           __builtin_fmaf(-c2[j], c2[j], __builtin_fmaf(-c[j], c[j], den[j]))),
                        31);
                }
                half[s] = bits;
              }
              // lanes < 32: entry r's two halves of points; lanes >= 32: entry 32 + r's
              const auto x = __builtin_amdgcn_permlane32_swap(half[0], half[1], false, false);
              const uint32_t live = n - b < 32 ? (1u << (n - b)) - 1u : ~0u;
              word = ~(x[0] | (x[1] << 16)) & live;
            }
            wd[0] = wd[1];
            wd[1] = wd[2];
            wd[2] = wd[3];
            wd[3] = word;
          }
          if (mine) *reinterpret_cast<uint4*>(my_mask + (base >> 5)) = make_uint4(wd[0], wd[1], wd[2], wd[3]);
        }
      }
      done = sub_end;
    }
  }
}

// ---- phase 2: the FP64 decisions and the in-order MSAC sums -----------------------

// One wave per list entry of the segment.  The mask row is taken 64 words
// (2,048 points) at a time, a word per lane: a prefix sum of the bit counts
// gives every lane its places in the window's queue of candidate points (point
// order), which the whole wave evaluates 64 at a time with the FP64 kernel's
// operations; fewer than 64 wait in registers for the next window's.  Inliers
// are accumulated in point order (value -= r2), as the FP64 kernel does.  The
// queue holds 16-bit offsets into the window, 16 KB per workgroup, so that
// registers (seven waves per SIMD) and not LDS bound the waves in flight: with
// 33 KB, four waves per SIMD, 48.7 us a launch in an essential batch of 32 pairs
// of 10,000 points and 58.0 in a fundamental one of 1,024 on MI355X, now 38.8 and
// 50.6.
template <int KIND>
__global__ void __launch_bounds__(256) k_mx_exact(const double* __restrict__ pts,
                                                  const int64_t* __restrict__ pair_pt_off,
                                                  const int32_t* __restrict__ pair_n,
                                                  const double* __restrict__ pair_sq_thr,
                                                  const double* __restrict__ models,
                                                  const int32_t* __restrict__ model_pair,
                                                  const int32_t* __restrict__ list,
                                                  const uint32_t* __restrict__ list_count, int64_t seg_begin,
                                                  int64_t seg_len, int words, const uint32_t* __restrict__ mask,
                                                  int32_t* __restrict__ counts, double* __restrict__ values,
                                                  int32_t* __restrict__ sym_counts, int slots_per) {
  __shared__ uint16_t queue[4][64 * 32];
  const int lane = lane_id();
  uint16_t* q = queue[threadIdx.x >> 6];
  const int64_t total = (int64_t)*list_count;
  if (seg_begin >= total) return;
  const int64_t seg_n = total - seg_begin < seg_len ? total - seg_begin : seg_len;
  const int xcd = (int)(blockIdx.x % kNumXcd);
  const int64_t waves_per_xcd = (int64_t)(gridDim.x / kNumXcd) * 4;
  const int64_t w = (int64_t)(blockIdx.x / kNumXcd) * 4 + (threadIdx.x >> 6);
  const int64_t lo_e = seg_n * xcd / kNumXcd, hi_e = seg_n * (xcd + 1) / kNumXcd;
  for (int64_t e = lo_e + w; e < hi_e; e += waves_per_xcd) {
    const int64_t slot = list[seg_begin + e];
    const int pair = model_pair[slots_per == 1 ? slot : slot / slots_per];
    const double* __restrict__ P = pts + 4 * pair_pt_off[pair];
    const int n = pair_n[pair];
    const double thr = pair_sq_thr[pair];
    double M[9];
#pragma unroll
    for (int k = 0; k < 9; ++k) M[k] = models[9 * slot + k];
    const uint32_t* __restrict__ mk = mask + e * (int64_t)words;
    double acc = 0.0;
    int64_t cnt = 0, scnt = 0;
    int kept = 0;     // candidates kept for the next 64, in order, on lanes 0 .. kept - 1
    int32_t mine = 0;
    // evaluates the candidates of lanes 0 .. cnt_flush - 1 and accumulates the
    // inliers among them in lane (= point) order
    auto flush = [&](int32_t point, int cnt_flush) {
      bool in = false, sym_in = false;
      double r2 = 0.0;
      if (lane < cnt_flush) {
        const double* s = P + 4 * (int64_t)point;
        if constexpr (KIND == 1) {
          double num, den;
          f_sampson_parts(s, M, num, den);
          const double t = thr * den;
          if (num < t * (1.0 - 1e-12)) in = true;
          else if (!(num > t * (1.0 + 1e-12))) in = (num / den) < thr;
          if (in) {
            r2 = f_sq_sampson(s, M);
            if (sym_counts) sym_in = f_sq_symmetric(s, M) < thr;
          }
        } else {
          r2 = h_sq_residual(s, M);
          in = r2 < thr;
        }
      }
      uint64_t b = ballot64(in);
      cnt += __popcll(b);
      if (KIND == 1 && sym_counts) scnt += __popcll(ballot64(sym_in));
      // many inliers: all 64 lanes in order (an outlier's r2 is no term); few:
      // one by one through the scalar unit (three instructions each)
      if (__popcll(b) > 20) {
        acc = wave_chain(acc, in ? r2 : 0.0, -1.0, cnt_flush);
      } else {
        while (b) {
          const int l = __ffsll((unsigned long long)b) - 1;
          acc = acc - readlane_f64(r2, l);
          b &= b - 1;
        }
      }
    };
    const int nw = (n + 31) >> 5;
    uint32_t next = lane < nw ? mk[lane] : 0u;
    for (int w0 = 0; w0 < nw; w0 += 64) {
      uint32_t bits = next;
      next = w0 + 64 + lane < nw ? mk[w0 + 64 + lane] : 0u;
      int before = __popc(bits);
      const int have = before;
      // inclusive prefix over the wave: inside the rows of 16 lanes, then the
      // rows before
      before += __builtin_amdgcn_update_dpp(0, before, 0x111, 0xF, 0xF, true);  // row_shr:1
      before += __builtin_amdgcn_update_dpp(0, before, 0x112, 0xF, 0xF, true);  // row_shr:2
      before += __builtin_amdgcn_update_dpp(0, before, 0x114, 0xF, 0xF, true);  // row_shr:4
      before += __builtin_amdgcn_update_dpp(0, before, 0x118, 0xF, 0xF, true);  // row_shr:8
      const int t0 = __builtin_amdgcn_readlane(before, 15), t1 = t0 + __builtin_amdgcn_readlane(before, 31),
                t2 = t1 + __builtin_amdgcn_readlane(before, 47), t3 = t2 + __builtin_amdgcn_readlane(before, 63);
      before += lane >= 48 ? t2 : (lane >= 32 ? t1 : (lane >= 16 ? t0 : 0));
      int at = before - have;
      while (bits) {
        q[at++] = (uint16_t)(32 * lane + __ffs(bits) - 1);
        bits &= bits - 1u;
      }
      wave_lds_handover();
      // the kept ones, then the window's
      const int all = kept + t3;
      auto point = [&](int k) { return k < kept ? mine : 32 * w0 + (int)q[k - kept]; };
      int h = 0;
      for (; h + 64 <= all; h += 64) flush(point(h + lane), 64);
      const int32_t rest = h + lane < all ? point(h + lane) : 0;
      mine = rest;
      kept = all - h;
      wave_lds_handover();  // the next window's queue
    }
    flush(mine, kept);
    if (lane == 0) {
      counts[slot] = (int32_t)cnt;
      values[slot] = cnt == 0 ? 0.0 : (acc + (double)cnt * thr) / thr;
      if (sym_counts) sym_counts[slot] = (int32_t)scnt;
    }
  }
}

// ---- launchers --------------------------------------------------------------------

void launch_mx_slack(hipStream_t st, const double* pts, const int32_t* pt_pair, const double* pair_sq_thr,
                     const double* inv_scale, int64_t first, int64_t count, int64_t total, uint16_t* out) {
  if (count <= 0) return;
  hipLaunchKernelGGL(k_mx_slack, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, st, pts, pt_pair, pair_sq_thr,
                     inv_scale, first, count, reinterpret_cast<float*>(out + kMxPlaneHalves * 4 * total));
}

void launch_mx_prepare(hipStream_t st, const double* pts, const int64_t* pair_pt_off, const int32_t* pair_n,
                       const int32_t* pt_pair, const double* pair_sq_thr, int num_pairs, int64_t total,
                       double* inv_scale, uint16_t* out) {
  if (num_pairs <= 0 || total <= 0) return;
  hipLaunchKernelGGL(k_mx_pair_scale, dim3((unsigned)num_pairs), dim3(256), 0, st, pts, pair_pt_off, pair_n,
                     num_pairs, inv_scale);
  hipLaunchKernelGGL(k_mx_points, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, pts, pt_pair, inv_scale,
                     total, out);
  launch_mx_slack(st, pts, pt_pair, pair_sq_thr, inv_scale, 0, total, total, out);
}

size_t mx_point_halves(int64_t total) {
  // four operand planes, the slack, and the slack that the last 32 points' loads run over
  return (size_t)(4 * kMxPlaneHalves * total + 2 * total + 64);
}

// 32-bit words of one entry's candidate mask (stored four at a time)
static int64_t mx_row_words(int max_n) { return (((int64_t)max_n + 31) / 32 + 3) & ~(int64_t)3; }

size_t mx_list_scratch_ints(int64_t num_models) {
  return (size_t)((num_models + kCompactPerBlock - 1) / kCompactPerBlock);
}

static int64_t mx_segment(int max_n) {
  const int64_t words = mx_row_words(max_n);
  const int64_t fit = kMxMaskBudget / (4 * words);
  // (whole tiles)
  return fit < kMxSegMin ? kMxSegMin : (fit > kMxSegMax ? kMxSegMax : fit & ~(int64_t)(kMxTile - 1));
}

size_t mx_mask_words(int max_n) {
  // the candidate masks, then the segment's operands (at most 3 x 2 x 2 x 16 B per entry)
  const int64_t seg = mx_segment(max_n);
  return (size_t)seg * (size_t)mx_row_words(max_n) + (size_t)seg * 48;
}

void launch_score_mx(hipStream_t st, int kind, const double* pts, const int64_t* pair_pt_off, const int32_t* pair_n,
                     const double* pair_sq_thr, const double* pair_inv_scale, const uint16_t* mxp, int64_t mx_total,
                     const double* models, const int32_t* model_pair, const int8_t* active, int64_t num_models,
                     int32_t* counts, double* values, int32_t* sym_counts, int slots_per, int32_t* work_list,
                     uint32_t* work_count, int32_t* blk_scratch, int max_n, uint32_t* mask) {
  if (num_models <= 0) return;
  const int nblk = (int)((num_models + kCompactPerBlock - 1) / kCompactPerBlock);
  hipLaunchKernelGGL(k_mx_count, dim3((unsigned)nblk), dim3(256), 0, st, active, num_models, counts, values,
                     sym_counts, blk_scratch);
  hipLaunchKernelGGL(k_mx_scan, dim3(1), dim3(1024), 0, st, blk_scratch, nblk, work_count);
  hipLaunchKernelGGL(k_mx_write, dim3((unsigned)nblk), dim3(256), 0, st, active, num_models, blk_scratch, work_list);
  const int slices = (max_n + kMxSliceMin - 1) / kMxSliceMin;  // at most
  const int words = (int)mx_row_words(max_n);
  const int64_t segment = mx_segment(max_n);
  h8* const coefs = reinterpret_cast<h8*>(mask + (size_t)segment * (size_t)words);
  // the active count is on the device; segments up to the slot count, and
  // each kernel returns at once past the end of the list
  for (int64_t seg = 0; seg < num_models; seg += segment) {
    const int64_t seg_len = num_models - seg < segment ? num_models - seg : segment;
    int64_t b1 = ((seg_len + kMxTile - 1) / kMxTile * slices + 3) / 4;
    if (b1 > kMxRejectBlocks) b1 = kMxRejectBlocks;
    b1 = (b1 + kNumXcd - 1) / kNumXcd * kNumXcd;
    int64_t b2 = (seg_len + 3) / 4;
    if (b2 > kMxExactBlocks) b2 = kMxExactBlocks;
    b2 = (b2 + kNumXcd - 1) / kNumXcd * kNumXcd;
    const unsigned bc = (unsigned)((2 * seg_len + 255) / 256);
    if (kind == 0) {
      hipLaunchKernelGGL(k_mx_coefs<0>, dim3(bc), dim3(256), 0, st, pair_sq_thr, pair_inv_scale, models,
                         model_pair, work_list, work_count, seg, seg_len, coefs, slots_per);
      hipLaunchKernelGGL(k_mx_reject<0>, dim3((unsigned)b1), dim3(256), 0, st, pair_pt_off, pair_n, mxp, mx_total,
                         coefs, model_pair, work_list, work_count, seg, seg_len, max_n, words, mask, slots_per);
      hipLaunchKernelGGL(k_mx_exact<0>, dim3((unsigned)b2), dim3(256), 0, st, pts, pair_pt_off, pair_n, pair_sq_thr,
                         models, model_pair, work_list, work_count, seg, seg_len, words, mask, counts, values,
                         sym_counts, slots_per);
    } else {
      hipLaunchKernelGGL(k_mx_coefs<1>, dim3(bc), dim3(256), 0, st, pair_sq_thr, pair_inv_scale, models,
                         model_pair, work_list, work_count, seg, seg_len, coefs, slots_per);
      hipLaunchKernelGGL(k_mx_reject<1>, dim3((unsigned)b1), dim3(256), 0, st, pair_pt_off, pair_n, mxp, mx_total,
                         coefs, model_pair, work_list, work_count, seg, seg_len, max_n, words, mask, slots_per);
      hipLaunchKernelGGL(k_mx_exact<1>, dim3((unsigned)b2), dim3(256), 0, st, pts, pair_pt_off, pair_n, pair_sq_thr,
                         models, model_pair, work_list, work_count, seg, seg_len, words, mask, counts, values,
                         sym_counts, slots_per);
    }
  }
}

}  // namespace gcr
