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
// S the sum of |z_t| over the terms the quantity reads (C, P, Q: (1 + |x1| +
// |y1|) (1 + |x2| + |y2|); W: 1 + |x1| + |y1|).  The Sampson denominator
// |(F x1)_01|^2 + |(F^T x2)_01|^2 is a linear form too, in the 11 squared terms
// (x1^2, x1 y1, y1^2, x1, y1, the same of the second image, 1); a quarter of it,
// D, has |coefficients| <= 1, and 11 + 10 + 11 products fill the 32 (the lo of
// the 1 is 0), so its bound is the same with 32 terms: dD = 2^-17 S + 2^-20.
//
// A point is dropped for a model only when the bounds prove it an outlier:
// Sampson (|C| - dC)+^2 > 4 tau''^2 (1 + 2^-16) (D + dD), transfer
// (|P| - dP)+^2 + (|Q| - dQ)+^2 > tau''^2 (1 + 2^-16) (|W| + dW)^2 (the
// factor 1 + 2^-16 covers the FP32 rounding of the test itself, about
// 10 * 2^-24).  Every other point -- all inliers and every point near the
// threshold -- is evaluated by the FP64 routines of the FP64 kernel
// (f_sampson_parts with its guard band, f_sq_sampson, f_sq_symmetric,
// h_sq_residual) and the MSAC value is accumulated in ascending point order
// on the model's lane.  Counts, values and symmetric counts are therefore the
// FP64 kernel's bits.  NaN / inf models or points never pass the rejection
// test, so they reach the FP64 path as before.
#include "dev_common.hpp"
#include "kernels.hpp"

namespace gcr {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

namespace {

constexpr float kDeltaRel = 0x1p-17f;
constexpr float kDeltaAbs = 0x1p-20f;
constexpr double kTauMargin = 1.0 + 0x1p-16;
constexpr int kCompactPerBlock = 2048;  // slots per block of the ordered compaction
constexpr int kMxBlocks = 2048;         // persistent grids: at most 8,192 waves
// list entries per rejection + exact pass: as many as keep the segment's
// candidate masks within kMxMaskBudget bytes, between kMxSegMin and
// kMxSegMax (each segment costs three launches; the masks bound the memory)
constexpr int64_t kMxSegMin = 65536, kMxSegMax = 1048576;
constexpr int64_t kMxMaskBudget = 512ll << 20;
// points per rejection work item: as many as leave kMxItems items (a tenth of
// the model slots hold a model to score at worst), between kMxSliceMin and
// kMxSliceMax (every item reads its 32 models' operands once)
constexpr int kMxSliceMin = 128, kMxSliceMax = 1024;
constexpr int64_t kMxItems = 16384;
constexpr int64_t kMxPlaneHalves = 16;  // 16-bit words of a point in one operand plane
constexpr int kNumXcd = 8;

__device__ __forceinline__ f32x16 mfma16(const h8& a, const h8& b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// v with lane `lane` replaced by the scalar x (clang 20 has no builtin for it)
extern "C" __device__ __attribute__((const)) uint32_t gcr_writelane(uint32_t x, uint32_t lane,
                                                                    uint32_t v) __asm("llvm.amdgcn.writelane.i32");

__device__ __forceinline__ f32x16 zero16() {
  f32x16 z;
#pragma unroll
  for (int j = 0; j < 16; ++j) z[j] = 0.0f;
  return z;
}

// One model's coefficient vectors over z (row-major 3x3 M): Sampson C;
// transfer P, Q, W.
template <int KIND>
__device__ __forceinline__ void quantity_coefs(const double* F, double c[][9]) {
  constexpr int NQ = KIND == 1 ? 1 : 3;
#pragma unroll
  for (int q = 0; q < NQ; ++q)
#pragma unroll
    for (int t = 0; t < 9; ++t) c[q][t] = 0.0;
  if constexpr (KIND == 1) {
#pragma unroll
    for (int t = 0; t < 9; ++t) c[0][t] = F[t];
  } else {
    c[0][0] = F[6]; c[0][1] = F[7]; c[0][2] = F[8]; c[0][6] = -F[0]; c[0][7] = -F[1]; c[0][8] = -F[2];
    c[1][3] = F[6]; c[1][4] = F[7]; c[1][5] = F[8]; c[1][6] = -F[3]; c[1][7] = -F[4]; c[1][8] = -F[5];
    c[2][6] = F[6]; c[2][7] = F[7]; c[2][8] = F[8];
  }
}

// A quarter of the Sampson denominator (F x1)_0^2 + (F x1)_1^2 + (F^T x2)_0^2 +
// (F^T x2)_1^2 as a linear form in d = (x1^2, x1 y1, y1^2, x1, y1, the same of
// the second image, 1): every coefficient is at most 1 when |F| <= 1.
__device__ __forceinline__ void denominator_coefs(const double* F, double g[11]) {
  const double a[2][3] = {{F[0], F[1], F[2]}, {F[3], F[4], F[5]}};
  const double b[2][3] = {{F[0], F[3], F[6]}, {F[1], F[4], F[7]}};
  g[10] = 0.0;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const double(*r)[3] = h ? b : a;
    g[5 * h] = 0.25 * (r[0][0] * r[0][0] + r[1][0] * r[1][0]);
    g[5 * h + 1] = 0.5 * (r[0][0] * r[0][1] + r[1][0] * r[1][1]);
    g[5 * h + 2] = 0.25 * (r[0][1] * r[0][1] + r[1][1] * r[1][1]);
    g[5 * h + 3] = 0.5 * (r[0][0] * r[0][2] + r[1][0] * r[1][2]);
    g[5 * h + 4] = 0.5 * (r[0][1] * r[0][2] + r[1][1] * r[1][2]);
    g[10] += 0.25 * (r[0][2] * r[0][2] + r[1][2] * r[1][2]);
  }
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

// Per point: the B-operand slices of both lane halves (k order, FP16) of z and
// of the squared terms d, and the error bounds; a plane per MFMA, so that a
// wave's load of 32 points is one contiguous kilobyte.
__global__ void __launch_bounds__(256) k_mx_points(const double* __restrict__ pts,
                                                   const int32_t* __restrict__ pt_pair,
                                                   const double* __restrict__ inv_scale, int64_t total,
                                                   uint16_t* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= total) return;
  const double is = inv_scale[pt_pair[i]];
  const double x1 = pts[4 * i] * is, y1 = pts[4 * i + 1] * is, x2 = pts[4 * i + 2] * is, y2 = pts[4 * i + 3] * is;
  const double zd[9] = {x2 * x1, x2 * y1, x2, y2 * x1, y2 * y1, y2, x1, y1, 1.0};
  const double dd[11] = {x1 * x1, x1 * y1, y1 * y1, x1, y1, x2 * x2, x2 * y2, y2 * y2, x2, y2, 1.0};
  h8* const o = reinterpret_cast<h8*>(out);
  _Float16 hi[11], lo[11];
#pragma unroll
  for (int t = 0; t < 9; ++t) {
    const float z = (float)zd[t];
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
    const float z = (float)dd[t];
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
  const float ax = fabsf((float)x1), ay = fabsf((float)y1), bx = fabsf((float)x2), by = fabsf((float)y2);
  const float sa = 1.0f + ax + ay, sb = 1.0f + bx + by;
  const float sd = 1.0f + ax * sa + ay * (1.0f + ay) + bx * sb + by * (1.0f + by);
  float4 d;
  d.x = kDeltaRel * (sa * sb) + kDeltaAbs;
  d.y = kDeltaRel * sa + kDeltaAbs;
  d.z = kDeltaRel * sd + kDeltaAbs;
  d.w = 0.0f;
  reinterpret_cast<float4*>(out + kMxPlaneHalves * 4 * total)[i] = d;
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

// ---- per-model A operands -----------------------------------------------------------

// One thread per (list entry of the segment, lane half): the entry's scaled,
// normalised coefficient vectors split into FP16 hi / lo and laid out as the
// MFMA A-operand slices of that lane half (NQ quantities x 2 MFMAs x 8).  A
// zero, inf or NaN model gets zero operands (nothing is rejected for it).
template <int KIND>
__global__ void __launch_bounds__(256) k_mx_coefs(const double* __restrict__ pair_inv_scale,
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
  const double sc[3] = {s, s, 1.0};
  double Fs[9], mx = 0.0;
  if constexpr (KIND == 1) {
    // F' = S F S: C, (F x1) and (F^T x2) in the scaled coordinates
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int k = 0; k < 3; ++k) Fs[3 * i + k] = M[3 * i + k] * sc[i] * sc[k];
  } else {
    // H' = S^-1 H S maps scaled x1 to scaled x2
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int k = 0; k < 3; ++k) Fs[3 * i + k] = M[3 * i + k] / sc[i] * sc[k];
  }
#pragma unroll
  for (int k = 0; k < 9; ++k) mx = fabs(Fs[k]) > mx ? fabs(Fs[k]) : mx;
  const bool lp_ok = mx > 0.0 && mx <= 1e300;
  const double inv_mx = lp_ok ? 1.0 / mx : 0.0;
#pragma unroll
  for (int k = 0; k < 9; ++k) Fs[k] = Fs[k] * inv_mx;
  double cq[3][9];
  quantity_coefs<KIND>(Fs, cq);
  h8* out = coefs + (e * 2 + hf) * (2 * NQ);
  _Float16 hi[11], lo[11];
#pragma unroll
  for (int q = 0; q < (KIND == 1 ? 1 : 3); ++q) {
#pragma unroll
    for (int k = 0; k < 9; ++k) {
      hi[k] = (_Float16)cq[q][k];
      lo[k] = (_Float16)(cq[q][k] - (double)hi[k]);
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
  if constexpr (KIND == 1) {
    double g[11];
    denominator_coefs(Fs, g);
#pragma unroll
    for (int k = 0; k < 11; ++k) {
      hi[k] = (_Float16)g[k];
      lo[k] = (_Float16)(g[k] - (double)hi[k]);
    }
#pragma unroll
    for (int kh = 0; kh < 2; ++kh) {
      h8 v;
#pragma unroll
      for (int x = 0; x < 8; ++x)
        v[x] = hf ? k_elem<11, 10>(hi, hi, lo, 16 * kh + 8 + x) : k_elem<11, 10>(hi, hi, lo, 16 * kh + x);
      out[2 + kh] = v;
    }
  }
}

// ---- phase 1: rejection on the matrix cores ---------------------------------------

// Work item (tile t, slice j): the 32 list entries 32 t .. 32 t + 31 of the
// segment (slot order, so the entries of one pair are adjacent; a tile that
// spans pairs is handled pair by pair) against points slice j .. slice j + slice
// - 1 of their pair.  Lane r < 32 owns entry r and writes, per 32-point chunk, the
// 32-bit word of its candidate mask (bit b: point base + b must be evaluated
// in FP64).  Words of points at or beyond the pair's n are not written.
template <int KIND>
__global__ void __launch_bounds__(256, 4) k_mx_reject(const int64_t* __restrict__ pair_pt_off,
                                                   const int32_t* __restrict__ pair_n,
                                                   const double* __restrict__ pair_sq_thr,
                                                   const double* __restrict__ pair_inv_scale,
                                                   const uint16_t* __restrict__ mxp, int64_t mx_total,
                                                   const h8* __restrict__ coefs,
                                                   const int32_t* __restrict__ model_pair,
                                                   const int32_t* __restrict__ list,
                                                   const uint32_t* __restrict__ list_count, int64_t seg_begin,
                                                   int64_t seg_len, int slice, int slices, int words, uint32_t* __restrict__ mask,
                                                   int slots_per) {
  constexpr int NQ = KIND == 1 ? 2 : 3;
  const int lane = lane_id();
  const int hf = lane >> 5, r = lane & 31;
  const int64_t total = (int64_t)*list_count;
  if (seg_begin >= total) return;
  const int64_t seg_n = total - seg_begin < seg_len ? total - seg_begin : seg_len;
  const int64_t items = (seg_n + 31) / 32 * slices;
  // gridDim.x is a multiple of kNumXcd: workgroup b runs on XCD b % kNumXcd,
  // which takes a contiguous range of items (adjacent items share a pair)
  const int xcd = (int)(blockIdx.x % kNumXcd);
  const int64_t waves_per_xcd = (int64_t)(gridDim.x / kNumXcd) * 4;
  const int64_t w = (int64_t)(blockIdx.x / kNumXcd) * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t lo_u = items * xcd / kNumXcd, hi_u = items * (xcd + 1) / kNumXcd;
  for (int64_t u = lo_u + w; u < hi_u; u += waves_per_xcd) {
    const int64_t t = u / slices;
    const int j = (int)(u - t * slices);
    const int64_t e0 = 32 * t;  // within the segment
    const int cnt_all = (int)(seg_n - e0 < 32 ? seg_n - e0 : 32);
    const int64_t slot = r < cnt_all ? (int64_t)list[seg_begin + e0 + r] : -1;
    const int my_pair = slot >= 0 ? model_pair[slots_per == 1 ? slot : slot / slots_per] : -1;
    uint32_t* __restrict__ my_mask = mask + (e0 + r) * (int64_t)words;
    int done = 0;
    while (done < cnt_all) {
      const int p = __builtin_amdgcn_readlane(my_pair, done);
      const bool mine = r >= done && r < cnt_all && my_pair == p;
      const int sub_end = done + __popcll(ballot64(mine) & 0xffffffffull);
      const int n = pair_n[p];
      const int first = slice * j;
      if (first < n) {
        // the sub-tile's A operands (lane: row r, half hf); other rows zero
        h8 A[NQ][2];
        const h8* __restrict__ my_coefs = coefs + ((e0 + r) * 2 + hf) * (2 * NQ);
#pragma unroll
        for (int q = 0; q < NQ; ++q)
#pragma unroll
          for (int kh = 0; kh < 2; ++kh) {
            if (mine) {
              A[q][kh] = my_coefs[2 * q + kh];
            } else {
#pragma unroll
              for (int e = 0; e < 8; ++e) A[q][kh][e] = (_Float16)0.0f;
            }
          }
        const double is = pair_inv_scale[p];
        const float tau2m = (float)(pair_sq_thr[p] * is * is * kTauMargin);
        const int64_t off = pair_pt_off[p];
        const h8* __restrict__ Z = reinterpret_cast<const h8*>(mxp) + 2 * off + hf;
        const float4* __restrict__ D = reinterpret_cast<const float4*>(mxp + kMxPlaneHalves * 4 * mx_total) + off;
        const int last = first + slice < n ? first + slice : n;
        for (int base = first; base < last; base += 32) {
          // points beyond the pair read its last one; their bits are cut below
          const int i = base + r < n ? base + r : n - 1;
          const h8 b0 = Z[2 * i], b1 = Z[2 * (mx_total + i)];
          const float4 dq = D[i];
          // accumulator slot j holds row 8 (j / 4) + 4 hf + (j % 4) of column
          // r; the ballot's halves are the words of its two rows, which go to
          // the lanes of those rows
          const uint32_t live = last - base < 32 ? (1u << (last - base)) - 1u : ~0u;  // uniform
          uint32_t word = 0;
          auto put = [&](int jj, bool rej) {
            const uint64_t k = ballot64(!rej);
            const int row = 8 * (jj >> 2) + (jj & 3);
            word = gcr_writelane((uint32_t)k, row, word);
            word = gcr_writelane((uint32_t)(k >> 32), row + 4, word);
          };
          if constexpr (KIND == 1) {
            const h8 b2 = Z[2 * (2 * mx_total + i)], b3 = Z[2 * (3 * mx_total + i)];
            f32x16 c = mfma16(A[0][0], b0, zero16());
            f32x16 den = mfma16(A[1][0], b2, zero16());
            c = mfma16(A[0][1], b1, c);
            den = mfma16(A[1][1], b3, den);
            const float k1 = 4.0f * tau2m;
            const float k2 = k1 * dq.z;
#pragma unroll
            for (int jj = 0; jj < 16; ++jj) {
              const float cl = fabsf(c[jj]) - dq.x;
              put(jj, cl * fabsf(cl) > __builtin_fmaf(den[jj], k1, k2));
            }
          } else {
            f32x16 pp = mfma16(A[0][0], b0, zero16());
            pp = mfma16(A[0][1], b1, pp);
            f32x16 qq = mfma16(A[1][0], b0, zero16());
            qq = mfma16(A[1][1], b1, qq);
            f32x16 ww = mfma16(A[2][0], b0, zero16());
            ww = mfma16(A[2][1], b1, ww);
#pragma unroll
            for (int jj = 0; jj < 16; ++jj) {
              const float pl = fmaxf(fabsf(pp[jj]) - dq.x, 0.0f);
              const float ql = fmaxf(fabsf(qq[jj]) - dq.x, 0.0f);
              const float wu = fabsf(ww[jj]) + dq.y;
              put(jj, __builtin_fmaf(pl, pl, ql * ql) > wu * wu * tau2m);
            }
          }
          if (mine && hf == 0) my_mask[base >> 5] = word & live;
        }
      }
      done = sub_end;
    }
  }
}

// ---- phase 2: the FP64 decisions and the in-order MSAC sums -----------------------

// One wave per list entry of the segment.  The mask row is taken 64 words
// (2,048 points) at a time, a word per lane: a prefix sum of the bit counts
// gives every lane its place in the queue of candidate points (point order),
// which the whole wave evaluates 64 at a time with the FP64 kernel's operations; inliers are accumulated in point order
// through the scalar unit (value -= r2), as the FP64 kernel does.
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
  __shared__ int32_t queue[4][64 + 64 * 32];
  const int lane = lane_id();
  int32_t* q = queue[threadIdx.x >> 6];
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
    int qn = 0;
    // evaluates the cnt_flush queued candidates from `at` on and accumulates the
    // inliers among them in queue (= point) order
    auto flush = [&](int at, int cnt_flush) {
      bool in = false, sym_in = false;
      double r2 = 0.0;
      if (lane < cnt_flush) {
        const double* s = P + 4 * (int64_t)q[at + lane];
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
      while (b) {
        const int l = __ffsll((unsigned long long)b) - 1;
        acc = acc - readlane_f64(r2, l);
        b &= b - 1;
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
      int at = qn + before - have;
      while (bits) {
        q[at++] = 32 * (w0 + lane) + __ffs(bits) - 1;
        bits &= bits - 1u;
      }
      qn += t3;
      int h = 0;
      for (; h + 64 <= qn; h += 64) flush(h, 64);
      if (h > 0) {
        const int rest = qn - h;
        const int32_t moved = lane < rest ? q[h + lane] : 0;
        if (lane < rest) q[lane] = moved;
        qn = rest;
      }
    }
    flush(0, qn);
    if (lane == 0) {
      counts[slot] = (int32_t)cnt;
      values[slot] = cnt == 0 ? 0.0 : (acc + (double)cnt * thr) / thr;
      if (sym_counts) sym_counts[slot] = (int32_t)scnt;
    }
  }
}

// ---- launchers --------------------------------------------------------------------

void launch_mx_prepare(hipStream_t st, const double* pts, const int64_t* pair_pt_off, const int32_t* pair_n,
                       const int32_t* pt_pair, int num_pairs, int64_t total, double* inv_scale, uint16_t* out) {
  if (num_pairs <= 0 || total <= 0) return;
  hipLaunchKernelGGL(k_mx_pair_scale, dim3((unsigned)num_pairs), dim3(256), 0, st, pts, pair_pt_off, pair_n,
                     num_pairs, inv_scale);
  hipLaunchKernelGGL(k_mx_points, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, pts, pt_pair, inv_scale,
                     total, out);
}

size_t mx_list_scratch_ints(int64_t num_models) {
  return (size_t)((num_models + kCompactPerBlock - 1) / kCompactPerBlock);
}

static int64_t mx_segment(int max_n) {
  const int64_t words = (max_n + 31) / 32 + 1;
  const int64_t fit = kMxMaskBudget / (4 * words);
  // (a multiple of 32: whole tiles, and the operands behind the masks stay aligned)
  return fit < kMxSegMin ? kMxSegMin : (fit > kMxSegMax ? kMxSegMax : fit & ~(int64_t)31);
}

size_t mx_mask_words(int max_n) {
  // the candidate masks, then the segment's A operands (at most 3 x 2 x 2 x 16 B per entry)
  const int64_t seg = mx_segment(max_n);
  return (size_t)seg * (size_t)((max_n + 31) / 32 + 1) + (size_t)seg * 48;
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
  int slice = kMxSliceMin;
  while (slice < kMxSliceMax && (num_models / 320 + 1) * ((max_n + 2 * slice - 1) / (2 * slice)) >= kMxItems) slice *= 2;
  const int slices = (max_n + slice - 1) / slice;
  const int words = (max_n + 31) / 32 + 1;
  const int64_t segment = mx_segment(max_n);
  h8* const coefs = reinterpret_cast<h8*>(mask + (size_t)segment * (size_t)words);
  // the active count is on the device; segments up to the slot count, and
  // each kernel returns at once past the end of the list
  for (int64_t seg = 0; seg < num_models; seg += segment) {
    const int64_t seg_len = num_models - seg < segment ? num_models - seg : segment;
    int64_t b1 = ((seg_len + 31) / 32 * slices + 3) / 4;
    if (b1 > kMxBlocks) b1 = kMxBlocks;
    b1 = (b1 + kNumXcd - 1) / kNumXcd * kNumXcd;
    int64_t b2 = (seg_len + 3) / 4;
    if (b2 > kMxBlocks) b2 = kMxBlocks;
    b2 = (b2 + kNumXcd - 1) / kNumXcd * kNumXcd;
    const unsigned bc = (unsigned)((2 * seg_len + 255) / 256);
    if (kind == 0) {
      hipLaunchKernelGGL(k_mx_coefs<0>, dim3(bc), dim3(256), 0, st, pair_inv_scale, models, model_pair, work_list,
                         work_count, seg, seg_len, coefs, slots_per);
      hipLaunchKernelGGL(k_mx_reject<0>, dim3((unsigned)b1), dim3(256), 0, st, pair_pt_off, pair_n, pair_sq_thr,
                         pair_inv_scale, mxp, mx_total, coefs, model_pair, work_list, work_count, seg, seg_len, slice, slices, words,
                         mask, slots_per);
      hipLaunchKernelGGL(k_mx_exact<0>, dim3((unsigned)b2), dim3(256), 0, st, pts, pair_pt_off, pair_n, pair_sq_thr,
                         models, model_pair, work_list, work_count, seg, seg_len, words, mask, counts, values,
                         sym_counts, slots_per);
    } else {
      hipLaunchKernelGGL(k_mx_coefs<1>, dim3(bc), dim3(256), 0, st, pair_inv_scale, models, model_pair, work_list,
                         work_count, seg, seg_len, coefs, slots_per);
      hipLaunchKernelGGL(k_mx_reject<1>, dim3((unsigned)b1), dim3(256), 0, st, pair_pt_off, pair_n, pair_sq_thr,
                         pair_inv_scale, mxp, mx_total, coefs, model_pair, work_list, work_count, seg, seg_len, slice, slices, words,
                         mask, slots_per);
      hipLaunchKernelGGL(k_mx_exact<1>, dim3((unsigned)b2), dim3(256), 0, st, pts, pair_pt_off, pair_n, pair_sq_thr,
                         models, model_pair, work_list, work_count, seg, seg_len, words, mask, counts, values,
                         sym_counts, slots_per);
    }
  }
}

}  // namespace gcr
