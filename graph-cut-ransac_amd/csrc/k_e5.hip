// Five-point essential-matrix minimal solver (Nister) over many samples.
//
// EssentialMatrixEstimator::estimateModel (essential_estimator.h:152-175) ->
// EssentialMatrixFivePointNisterSolver
// (solver_essential_matrix_five_point_nister.h:204-615) on K-normalised
// coordinates, then the oriented epipolar filter (essential_estimator.h:338-398).
// Every element of every matrix keeps the operations and the order of the
// sequential solver, so results are its bits.
//
// Four kernels, each with the mapping its step fits in registers:
//   k_e5_null_space   one thread per sample: null space of the 5 x 9 system
//                     (Gauss-Jordan with full pivoting, pivots applied by
//                     selects);
//   k_e5_constraints  one thread per sample: the ten cubic constraints;
//   k_e5_eliminate    four lanes per sample: LU with partial pivoting of the
//                     10 x 20 constraint matrix, lane q of a quad holding the
//                     columns c = q mod 4 (50 values), the pivot column
//                     broadcast inside the quad by DPP; only the solution's
//                     rows 4 .. 9, which the polynomial needs, are formed;
//   k_e5_roots        one thread per sample: the degree-10 polynomial, its
//                     real roots by Sturm sequences, the models and the
//                     orientation filter.
// Between them the values of a slab of samples go through HBM in tiles of 64
// samples, value by value (a wave's loads and stores are coalesced and its
// tile contiguous; rows of the whole slab, a power of two apart, took 245 us
// per 131,072 samples in the first two kernels each).
//
// What bounds it: in the first two kernels straight-line code (29 and 11 KB;
// their instruction fetches) and FP64 VALU, in the elimination the selects of
// the row exchanges, in the root search lanes that wait for the sample with
// the most bisections.  One thread per sample for the whole solver kept 5,360
// bytes of matrices per thread in scratch memory; here the matrices are in
// registers, and scratch holds the root search's rarely used deep intervals (560
// bytes, kE5StackMore) and 28 bytes of spills in the elimination.  Measured on MI355X, 32
// pairs of 10,000 points at 10 % inliers: 1,079 ms of the call's kernels then,
// 166 ms with these kernels (per 131,072 samples 139 + 86 + 118 + 224 us, four
// streams at once; alone 24 + 37 + 69 + 148); the call 1,173 -> 614 ms.
#include "dev_essential.hpp"
#include "kernels.hpp"

#include <algorithm>

namespace gcr {

namespace {

constexpr MulTable kMul = make_mul_table(kNisterOrder);

// out += s * (p * q), products added in (i, j) order.
__device__ __forceinline__ void mul11(const double* p, const double* q, double s, double* out) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) out[kMul.m11[4 * i + j]] = out[kMul.m11[4 * i + j]] + s * (p[i] * q[j]);
}
__device__ __forceinline__ void mul21(const double* p, const double* q, double s, double* out) {
#pragma unroll
  for (int i = 0; i < 10; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) out[kMul.m21[4 * i + j]] = out[kMul.m21[4 * i + j]] + s * (p[i] * q[j]);
}

}  // namespace

// Slab layout (doubles): value v of the slab's sample t is at
// (t / 64) kE5SlabValues 64 + 64 v + t % 64: N 0 .. 35, C 36 .. 235 (row-major
// 10 x 20), X 236 .. 295 (the solution's rows 4 .. 9, 10 columns each).
constexpr int kE5N = 0, kE5C = 36, kE5X = 236;
constexpr int kTile = 64;
__device__ __forceinline__ int64_t e5_tile(int t) {
  return (int64_t)(t / kTile) * (kE5SlabValues * kTile) + t % kTile;
}
static_assert(kE5X + 60 == kE5SlabValues, "slab layout");

__global__ void __launch_bounds__(64) k_e5_null_space(const double* __restrict__ pts,
                                                      const int64_t* __restrict__ pair_pt_off,
                                                      const int32_t* __restrict__ cand_pair,
                                                      const int32_t* __restrict__ samples, int64_t first, int count,
                                                      double* __restrict__ slab, int8_t* __restrict__ nmodels) {
  const int t = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  if (t >= count) return;
  const int64_t c = first + t;
  const int32_t* s = samples + 5 * c;
  double* o = slab + e5_tile(t);
  double a[5][9], N[36];
  bool ok = s[0] >= 0;
  if (ok) {
    const double* P = pts + 4 * pair_pt_off[cand_pair[c]];
#pragma unroll
    for (int i = 0; i < 5; ++i) e_row(P + 4 * (int64_t)s[i], 1.0, a[i]);
    ok = null_space_5x9(a, N);
  }
  nmodels[c] = ok ? 1 : 0;  // 1: the sample has a null space (the root kernel writes the count)
  if (!ok) return;
#pragma unroll
  for (int v = 0; v < 36; ++v) o[(kE5N + v) * kTile] = N[v];
}

// The nine trace constraints in a loop (entry (i, j)'s operands from LDS): 11 KB
// of code instead of 35, and the kernel stays in the instruction cache.  Fully
// unrolled together with the null space (66 KB) every wave fetched its code
// from the L2 line by line: 242 us per 131,072 samples.
__global__ void __launch_bounds__(64) k_e5_constraints(int64_t first, int count, double* __restrict__ slab,
                                                       const int8_t* __restrict__ nmodels) {
  __shared__ double l_ee[36][64];
  const int lane = threadIdx.x;
  const int t = (int)(blockIdx.x * 64 + threadIdx.x);
  if (t >= count || !nmodels[first + t]) return;
  double* o = slab + e5_tile(t);
  // ee(i, j): the four coefficients of E(i, j) = x N0 + y N1 + z N2 + N3
  double ee[3][3][4];
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        ee[i][j][k] = o[(kE5N + 9 * k + 3 * j + i) * kTile];
        l_ee[12 * i + 4 * j + k][lane] = ee[i][j][k];  // read by this lane only
      }
  double* oc = o + kE5C * kTile;
  {
    // det E along the third row
    constexpr int cof[3][4] = {{0, 1, 1, 2}, {0, 2, 1, 0}, {0, 0, 1, 1}};
    constexpr int cofn[3][4] = {{0, 2, 1, 1}, {0, 0, 1, 2}, {0, 1, 1, 0}};
    double row[20];
#pragma unroll
    for (int v = 0; v < 20; ++v) row[v] = 0.0;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      double d[10];
#pragma unroll
      for (int v = 0; v < 10; ++v) d[v] = 0.0;
      mul11(ee[cof[k][0]][cof[k][1]], ee[cof[k][2]][cof[k][3]], 1.0, d);
      mul11(ee[cofn[k][0]][cofn[k][1]], ee[cofn[k][2]][cofn[k][3]], -1.0, d);
      mul21(d, ee[2][k], 1.0, row);
    }
#pragma unroll
    for (int v = 0; v < 20; ++v) oc[(180 + v) * kTile] = row[v];
  }
  double tr[10];
#pragma unroll 1
  for (int i = 0; i < 3; ++i) {
    // the trace's diagonal entry (i, i) of E E^T
    double ei[3][4], d[10];
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
      for (int v = 0; v < 4; ++v) ei[k][v] = l_ee[12 * i + 4 * k + v][lane];
#pragma unroll
    for (int v = 0; v < 10; ++v) d[v] = 0.0;
#pragma unroll
    for (int k = 0; k < 3; ++k) mul11(ei[k], ei[k], 1.0, d);
#pragma unroll
    for (int v = 0; v < 10; ++v) tr[v] = i == 0 ? d[v] : tr[v] + d[v];
  }
#pragma unroll 1
  for (int i = 0; i < 3; ++i) {
    // row i of E E^T
    double ei[3][4], d[3][10];
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
      for (int v = 0; v < 4; ++v) ei[k][v] = l_ee[12 * i + 4 * k + v][lane];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
#pragma unroll
      for (int v = 0; v < 10; ++v) d[j][v] = 0.0;
#pragma unroll
      for (int k = 0; k < 3; ++k) mul11(ei[k], ee[j][k], 1.0, d[j]);
    }
#pragma unroll 1
    for (int j = 0; j < 3; ++j) {
      double row[20], q[4];
#pragma unroll
      for (int v = 0; v < 20; ++v) row[v] = 0.0;
#pragma unroll
      for (int k = 0; k < 3; ++k) {
#pragma unroll
        for (int v = 0; v < 4; ++v) q[v] = l_ee[12 * k + 4 * j + v][lane];
        mul21(d[k], q, 1.0, row);
      }
#pragma unroll
      for (int v = 0; v < 4; ++v) q[v] = l_ee[12 * i + 4 * j + v][lane];
      mul21(tr, q, -0.5, row);
      double* orow = oc + (int64_t)(20 * (3 * i + j)) * kTile;
#pragma unroll
      for (int v = 0; v < 20; ++v) orow[v * kTile] = row[v];
    }
  }
}

namespace {

// Lane Q of every quad to the whole quad.
template <int Q>
__device__ __forceinline__ double quad_bcast(double v) {
  return dpp_mov_f64<Q * 0x55>(v);
}
// value of column COL (lane COL % 4, register COL / 4), row i
#define COLUMN(COL, i) quad_bcast<(COL) % 4>(a[(COL) / 4][i])

template <int K>
__device__ __forceinline__ void eliminate_step(double (&a)[5][10], int q) {
  // the pivot column on every lane of the quad
  double col[10];
#pragma unroll
  for (int i = K; i < 10; ++i) col[i] = COLUMN(K, i);
  int p = K;
  double best = fabs(col[K]);
#pragma unroll
  for (int i = K + 1; i < 10; ++i) {
    const bool take = fabs(col[i]) > best;
    best = take ? fabs(col[i]) : best;
    p = take ? i : p;
  }
  // rows K and p change places in the columns still in use (c >= K)
#pragma unroll
  for (int i = K + 1; i < 10; ++i) {
    const bool sw = i == p;
#pragma unroll
    for (int r = K / 4; r < 5; ++r) {
      const double x = a[r][K];
      a[r][K] = sw ? a[r][i] : x;
      a[r][i] = sw ? x : a[r][i];
    }
    const double x = col[K];
    col[K] = sw ? col[i] : x;
    col[i] = sw ? x : col[i];
  }
  // the multipliers: lane q forms those of rows K + 1 + q, K + 5 + q, ..
  const double piv = col[K];
  double f[12];
#pragma unroll
  for (int g = K + 1; g < 10; g += 4) {
    double num = col[g];
#pragma unroll
    for (int d = 1; d < 4; ++d)
      if (g + d < 10) num = q == d ? col[g + d] : num;
    const double v = num / piv;
    f[g - K - 1] = quad_bcast<0>(v);
    if (g + 1 < 10) f[g - K] = quad_bcast<1>(v);
    if (g + 2 < 10) f[g - K + 1] = quad_bcast<2>(v);
    if (g + 3 < 10) f[g - K + 2] = quad_bcast<3>(v);
  }
#pragma unroll
  for (int i = K + 1; i < 10; ++i)
#pragma unroll
    for (int r = K / 4; r < 5; ++r) a[r][i] = a[r][i] - f[i - K - 1] * a[r][K];
}

}  // namespace

// Four lanes per sample; lane q of the quad holds columns q, q + 4, .., q + 16
// of the 10 x 20 matrix.  Columns left of the pivot are updated along with
// the others: their entries below the diagonal are read by nothing.
__global__ void __launch_bounds__(256, 3) k_e5_eliminate(double* __restrict__ slab, int count) {
  const int g = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  const int q = g & 3;
  // lanes past the end work on the last sample (the quad moves need every
  // lane) and store nothing
  const int t = (g >> 2) < count ? (g >> 2) : count - 1;
  const bool live = (g >> 2) < count;
  double* o = slab + e5_tile(t);
  double a[5][10];
#pragma unroll
  for (int r = 0; r < 5; ++r)
#pragma unroll
    for (int i = 0; i < 10; ++i) a[r][i] = o[(kE5C + 20 * i + 4 * r + q) * kTile];
  eliminate_step<0>(a, q);
  eliminate_step<1>(a, q);
  eliminate_step<2>(a, q);
  eliminate_step<3>(a, q);
  eliminate_step<4>(a, q);
  eliminate_step<5>(a, q);
  eliminate_step<6>(a, q);
  eliminate_step<7>(a, q);
  eliminate_step<8>(a, q);
  // the solution's rows 9 .. 4 in the right-hand columns 10 .. 19 (registers
  // 2, lanes 2 and 3, and registers 3 and 4)
#define BACK(I)                                                                      \
  {                                                                                  \
    double v2 = a[2][I], v3 = a[3][I], v4 = a[4][I];                                 \
    BACK_FROM(I, 5) BACK_FROM(I, 6) BACK_FROM(I, 7) BACK_FROM(I, 8) BACK_FROM(I, 9)  \
    const double d = COLUMN(I, I);                                                   \
    x[0][I - 4] = v2 / d;                                                            \
    x[1][I - 4] = v3 / d;                                                            \
    x[2][I - 4] = v4 / d;                                                            \
  }
#define BACK_FROM(I, J)                  \
  if (J > I) {                           \
    const double u = COLUMN(J, I);       \
    v2 = v2 - u * x[0][J - 4];           \
    v3 = v3 - u * x[1][J - 4];           \
    v4 = v4 - u * x[2][J - 4];           \
  }
  double x[3][6];
  BACK(9)
  BACK(8)
  BACK(7)
  BACK(6)
  BACK(5)
  BACK(4)
#undef BACK
#undef BACK_FROM
#undef COLUMN
  if (!live) return;
#pragma unroll
  for (int i = 0; i < 6; ++i) {
    if (q >= 2) o[(kE5X + 10 * i + q - 2) * kTile] = x[0][i];
    o[(kE5X + 10 * i + q + 2) * kTile] = x[1][i];
    o[(kE5X + 10 * i + q + 6) * kTile] = x[2][i];
  }
}

namespace {

// out (du + dv + 1 coefficients) = u v, products added in (i, j) order
template <int DU, int DV>
__device__ __forceinline__ void poly_mul(const double* u, const double* v, double* out) {
#pragma unroll
  for (int k = 0; k <= DU + DV; ++k) out[k] = 0.0;
#pragma unroll
  for (int i = 0; i <= DU; ++i)
#pragma unroll
    for (int j = 0; j <= DV; ++j) out[i + j] = out[i + j] + u[i] * v[j];
}

// The three rows of the polynomial system from the solution's rows
// (nister.h:360-470): A[i][0..12].
__device__ __forceinline__ void poly_rows(const double* x, double (&A)[3][13]) {
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    double r1[10], r2[10];
#pragma unroll
    for (int c = 0; c < 10; ++c) {
      r1[c] = x[(20 * i + c) * kTile];
      r2[c] = x[(20 * i + 10 + c) * kTile];
    }
    A[i][0] = 0.0;
#pragma unroll
    for (int c = 0; c < 3; ++c) A[i][1 + c] = r1[c];
#pragma unroll
    for (int c = 0; c < 3; ++c) A[i][c] = A[i][c] - r2[c];
    A[i][4] = 0.0;
#pragma unroll
    for (int c = 0; c < 3; ++c) A[i][5 + c] = r1[3 + c];
#pragma unroll
    for (int c = 0; c < 3; ++c) A[i][4 + c] = A[i][4 + c] - r2[3 + c];
    A[i][8] = 0.0;
#pragma unroll
    for (int c = 0; c < 4; ++c) A[i][9 + c] = r1[6 + c];
#pragma unroll
    for (int c = 0; c < 4; ++c) A[i][8 + c] = A[i][8 + c] - r2[6 + c];
  }
}

// det of the 3 x 3 polynomial matrix: the degree-10 polynomial, ascending.
__device__ __forceinline__ void poly_det(const double (&A)[3][13], double* c) {
  double P[3][4], Q[3][4], R[3][5];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      P[i][d] = A[i][3 - d];
      Q[i][d] = A[i][7 - d];
    }
#pragma unroll
    for (int d = 0; d < 5; ++d) R[i][d] = A[i][12 - d];
  }
#pragma unroll
  for (int k = 0; k < 11; ++k) c[k] = 0.0;
  double t1[8], t2[8], m7[8], full[11];
  poly_mul<3, 4>(Q[1], R[2], t1);
  poly_mul<3, 4>(Q[2], R[1], t2);
#pragma unroll
  for (int k = 0; k < 8; ++k) m7[k] = t1[k] - t2[k];
  poly_mul<3, 7>(P[0], m7, full);
#pragma unroll
  for (int k = 0; k < 11; ++k) c[k] = c[k] + full[k];
  poly_mul<3, 4>(P[1], R[2], t1);
  poly_mul<3, 4>(P[2], R[1], t2);
#pragma unroll
  for (int k = 0; k < 8; ++k) m7[k] = t1[k] - t2[k];
  poly_mul<3, 7>(Q[0], m7, full);
#pragma unroll
  for (int k = 0; k < 11; ++k) c[k] = c[k] - full[k];
  poly_mul<3, 3>(P[1], Q[2], t1);
  poly_mul<3, 3>(P[2], Q[1], t2);
  double m6[7];
#pragma unroll
  for (int k = 0; k < 7; ++k) m6[k] = t1[k] - t2[k];
  poly_mul<4, 6>(R[0], m6, full);
#pragma unroll
  for (int k = 0; k < 11; ++k) c[k] = c[k] + full[k];
}

}  // namespace

// Pending intervals of a thread's root search held in LDS, and beyond them in
// private memory.  An interval is pushed only when it holds a root (others
// are never looked at), so there are at most as many as roots (ten) unless
// rounding makes the sign counts inconsistent; one right sibling per level
// of a depth of 30 is the limit then.  Seven in LDS (19.2 KB with the intervals
// found) let eight waves be resident on a compute unit, a whole slab at once;
// with ten (23 KB) six were: 206 us per 131,072 samples on MI355X, 148 now.
constexpr int kE5Stack = 7, kE5StackMore = 27;

__global__ void __launch_bounds__(64) k_e5_roots(const double* __restrict__ pts,
                                                 const int64_t* __restrict__ pair_pt_off,
                                                 const int32_t* __restrict__ cand_pair,
                                                 const int32_t* __restrict__ samples, int64_t first, int count,
                                                 const double* __restrict__ slab,
                                                 double* __restrict__ models, int8_t* __restrict__ mstatus,
                                                 int8_t* __restrict__ nmodels) {
  __shared__ double l_a[kE5Stack][64], l_b[kE5Stack][64], l_lo[10][64], l_hi[10][64];
  __shared__ int l_s[kE5Stack][64];
  const int lane = threadIdx.x;
  const int t = (int)(blockIdx.x * 64 + threadIdx.x);
  if (t >= count) return;
  const int64_t cand = first + t;
  const double* tile = slab + e5_tile(t);
  int nr = 0;
  if (nmodels[cand]) {
    SturmSeq10 st;
    bool ok;
    {
      double A[3][13], c[11];
      poly_rows(tile + kE5X * kTile, A);
      poly_det(A, c);
      ok = st.init(c);
    }
    if (ok) {
      const double r0 = st.root_bound();
      double a = -r0, b = r0;
      int sa = st.sign_changes(a), sb = st.sign_changes(b), depth = 0, top = 0;
      double more_a[kE5StackMore], more_b[kE5StackMore];
      int more_s[kE5StackMore];
      bool have = sa - sb != 0;
      int ni = 0;  // isolating intervals, in ascending order
      // depth first, left half first: (a, b] is the current interval
      while (have) {
        const int n = sa - sb;
        bool next = true;  // take the next pending interval
        if (depth <= 30) {
          if (n > 1) {
            const double m = (a + b) * 0.5;
            const int sm = st.sign_changes(m);
            if (sa - sm >= 1) {
              if (sm - sb >= 1) {
                const int packed = sm | (sb << 4) | ((depth + 1) << 8);
                if (top < kE5Stack) {
                  l_a[top][lane] = m;
                  l_b[top][lane] = b;
                  l_s[top][lane] = packed;
                } else {
                  more_a[top - kE5Stack] = m;
                  more_b[top - kE5Stack] = b;
                  more_s[top - kE5Stack] = packed;
                }
                ++top;
              }
              b = m;
              sb = sm;
              ++depth;
              next = false;
            } else if (sm - sb >= 1) {
              a = m;
              sa = sm;
              ++depth;
              next = false;
            }
          } else if (n == 1 && ni < 10) {
            l_lo[ni][lane] = a;
            l_hi[ni][lane] = b;
            ++ni;
          }
        }
        if (next) {
          have = top > 0;
          if (have) {
            --top;
            int packed;
            if (top < kE5Stack) {
              a = l_a[top][lane];
              b = l_b[top][lane];
              packed = l_s[top][lane];
            } else {
              a = more_a[top - kE5Stack];
              b = more_b[top - kE5Stack];
              packed = more_s[top - kE5Stack];
            }
            sa = packed & 15;
            sb = (packed >> 4) & 15;
            depth = packed >> 8;
          }
        }
      }
      // the roots, every lane its q-th interval at a time (in the isolation
      // loop each lane meets its intervals at other steps, and the wave ran
      // the refinement at nearly every step: 527 us per 131,072 samples)
      for (int q = 0; q < ni; ++q) {
        double x;
        if (st.refine(l_lo[q][lane], l_hi[q][lane], 1e-10, x)) l_lo[nr++][lane] = x;
      }
    }
  }
  int kept = 0;
  double* out = models + 90 * cand;
  if (nr > 0) {
    double A[3][13], N[36];
    poly_rows(tile + kE5X * kTile, A);
#pragma unroll
    for (int v = 0; v < 36; ++v) N[v] = tile[(kE5N + v) * kTile];
    const double* P = pts + 4 * pair_pt_off[cand_pair[cand]];
    const int32_t* s = samples + 5 * cand;
    for (int q = 0; q < nr; ++q) {
      const double z = l_lo[q][lane];
      const double z2 = z * z, z3 = z2 * z, z4 = z2 * z2;
      double b0[3], b1[3], bb[3];
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        b0[i] = A[i][0] * z3 + A[i][1] * z2 + A[i][2] * z + A[i][3];
        b1[i] = A[i][4] * z3 + A[i][5] * z2 + A[i][6] * z + A[i][7];
        bb[i] = A[i][8] * z4 + A[i][9] * z3 + A[i][10] * z2 + A[i][11] * z + A[i][12];
      }
      const double det = b0[0] * b1[1] - b1[0] * b0[1];
      const double id = 1.0 / det;
      double xz[2];
      xz[0] = (b1[1] * id) * bb[0] + (-b1[0] * id) * bb[1];
      xz[1] = (-b0[1] * id) * bb[0] + (b0[0] * id) * bb[1];
      if (fabs(b0[2] * xz[0] + b1[2] * xz[1] - bb[2]) > 1e-6) solve3x2_fullpiv(b0, b1, bb, xz);
      const double x = -xz[0], y = -xz[1];
      double e[9], m[9];
      const double sc = 1.0 / sqrt(x * x + y * y + z * z + 1.0);
#pragma unroll
      for (int k = 0; k < 9; ++k) e[k] = (N[k] * x + N[9 + k] * y + N[18 + k] * z + N[27 + k]) * sc;
#pragma unroll
      for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int cc = 0; cc < 3; ++cc) m[3 * r + cc] = e[3 * cc + r];
      if (f_orientation_valid_idx(m, P, s, 5)) {
#pragma unroll
        for (int i = 0; i < 9; ++i) out[9 * kept + i] = m[i];
        ++kept;
      }
    }
  }
  for (int k = 0; k < 10; ++k) mstatus[10 * cand + k] = k < kept ? 2 : 0;
  nmodels[cand] = (int8_t)kept;
}

int64_t e5_slab(int64_t num_cand) {
  return std::min<int64_t>((std::max<int64_t>(num_cand, 1) + kTile - 1) / kTile * kTile, kE5SlabMax);
}

void launch_e5_solve(hipStream_t st, const double* pts, const int64_t* pair_pt_off, const int32_t* cand_pair,
                     const int32_t* samples, int64_t num_cand, double* models, int8_t* mstatus, int8_t* nmodels,
                     double* scratch) {
  const int64_t slab = e5_slab(num_cand);
  for (int64_t c0 = 0; c0 < num_cand; c0 += slab) {
    const int count = (int)std::min<int64_t>(slab, num_cand - c0);
    const unsigned waves = (unsigned)((count + 63) / 64);
    hipLaunchKernelGGL(k_e5_null_space, dim3(waves), dim3(64), 0, st, pts, pair_pt_off, cand_pair, samples, c0, count,
                       scratch, nmodels);
    hipLaunchKernelGGL(k_e5_constraints, dim3(waves), dim3(64), 0, st, c0, count, scratch, nmodels);
    hipLaunchKernelGGL(k_e5_eliminate, dim3((unsigned)((4 * (int64_t)count + 255) / 256)), dim3(256), 0, st, scratch, count);
    hipLaunchKernelGGL(k_e5_roots, dim3(waves), dim3(64), 0, st, pts, pair_pt_off, cand_pair, samples, c0, count,
                       scratch, models, mstatus, nmodels);
  }
}

}  // namespace gcr
