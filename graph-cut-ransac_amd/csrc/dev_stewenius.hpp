// Stewenius five-point solver on one wavefront (gfx950): the dense steps of
// the essential matrix's non-minimal fit (EssentialMatrixFivePointStewenius-
// Solver, ...stewenius.h:114-231).
//
// Every matrix is spread over the lanes -- a column per lane in registers
// where the row indices are compile-time constants (QR, elimination, null
// vectors), in LDS where they are not (eigenvalues) -- and every element keeps
// the operations and the order of the sequential solver, so results are its
// bits.
//
// What bounds it: one wave's chain of dependent divisions, square roots and
// LDS round trips (the QR steps of the eigenvalues above all).  With the dense
// steps on lane 0 and their arrays in scratch memory a launch of fits took
// 1,830 us on MI355X (one pair of 1,500 points), now 129 us; the call 19.4 ->
// 3.9 ms together with the minimal solver's kernels.
#pragma once

#include "dev_essential.hpp"

namespace gcr {

// Products of degree-1 polynomials (degree 2: at most two terms per
// coefficient) and of a degree-2 with a degree-1 polynomial (at most three), as
// the terms of each coefficient in the order the sequential product adds them:
// 16 * index in the first factor + index in the second, -1: none.
struct TermTable {
  int16_t t11[10][2];
  int16_t t21[20][3];
};
constexpr TermTable make_terms(const MulTable& m) {
  TermTable t{};
  for (int k = 0; k < 10; ++k) {
    int c = 0;
    t.t11[k][0] = t.t11[k][1] = -1;
    for (int e = 0; e < 16; ++e)
      if (m.m11[e] == k) t.t11[k][c++] = (int16_t)(16 * (e / 4) + e % 4);
  }
  for (int k = 0; k < 20; ++k) {
    int c = 0;
    t.t21[k][0] = t.t21[k][1] = t.t21[k][2] = -1;
    for (int e = 0; e < 40; ++e)
      if (m.m21[e] == k) t.t21[k][c++] = (int16_t)(16 * (e / 4) + e % 4);
  }
  return t;
}
struct StewShared {
  double ee[3][3][4];    // coefficients of E(i, j) = x N0 + y N1 + z N2 + N3
  double eet[9][10];     // 2 E E^T
  double tr[10];         // its trace
  double cof[3][10];     // cofactors of the third row
  double a[10][10];      // action matrix
  double h[10][10];      // its Hessenberg form, then the QR iterations
  double ev[10], evs[10];
  double vec[10][10];    // null vectors
  int pos[10];
};

// The sum over at most nine terms in the wave's 64-lane order: partials of
// terms 0 .. 8 combined as p[l] += p[l + s], s = 8 .. 1.
template <int BEGIN, class F>
__device__ __forceinline__ double tree9(F term) {
  double p[9];
#pragma unroll
  for (int i = 0; i < 9; ++i) p[i] = i >= BEGIN ? 0.0 + term(i) : 0.0;
  const double a = ((p[0] + p[8]) + p[4]) + (p[2] + p[6]);
  const double b = (p[1] + p[5]) + (p[3] + p[7]);
  return a + b;
}

// One step of the column-pivoted Householder QR: lane j holds column j.
template <int K>
__device__ __forceinline__ void qr9_step(double (&col)[9], double& norm, double (&hv)[9], double& tau) {
  const int lane = lane_id();
  int p = K;
  double np = readlane_f64(norm, K);
#pragma unroll
  for (int j = K + 1; j < 9; ++j) {
    const double nj = readlane_f64(norm, j);
    if (nj > np) {
      np = nj;
      p = j;
    }
  }
  p = __builtin_amdgcn_readfirstlane(p);
  if (p != K) {
    const int src = lane == K ? p : (lane == p ? K : lane);
#pragma unroll
    for (int i = 0; i < 9; ++i) col[i] = __shfl(col[i], src, 64);
    norm = __shfl(norm, src, 64);
  }
  const double alpha = readlane_f64(col[K], K);
  const double sigma = readlane_f64(tree9<K + 1>([&](int i) { return col[i] * col[i]; }), K);
  tau = 0.0;
#pragma unroll
  for (int i = 0; i < 9; ++i) hv[i] = i == K ? 1.0 : 0.0;
  if (sigma != 0.0) {
    const double nrm = sqrt(alpha * alpha + sigma);
    const double beta = alpha >= 0.0 ? -nrm : nrm;
    tau = (beta - alpha) / beta;
    const double scale = 1.0 / (alpha - beta);
#pragma unroll
    for (int i = K + 1; i < 9; ++i) hv[i] = readlane_f64(col[i] * scale, K);
    if (lane > K) {
      const double w = col[K] + tree9<K + 1>([&](int i) { return hv[i] * col[i]; });
      const double tw = tau * w;
      col[K] = col[K] - tw;
#pragma unroll
      for (int i = K + 1; i < 9; ++i) col[i] = col[i] - tw * hv[i];
    }
  }
  norm = tree9<K + 1>([&](int i) { return col[i] * col[i]; });
}

// Null space of the 9 x 9 matrix whose column `lane` is col: the last four
// columns of Q (the role of ColPivHouseholderQR::matrixQ) to NS.
__device__ __forceinline__ void wave_qr9_null_space(double (&col)[9], double (&NS)[9][4]) {
  const int lane = lane_id();
  double hv[9][9], tau[9];
  double norm = tree9<0>([&](int i) { return col[i] * col[i]; });
  qr9_step<0>(col, norm, hv[0], tau[0]);
  qr9_step<1>(col, norm, hv[1], tau[1]);
  qr9_step<2>(col, norm, hv[2], tau[2]);
  qr9_step<3>(col, norm, hv[3], tau[3]);
  qr9_step<4>(col, norm, hv[4], tau[4]);
  qr9_step<5>(col, norm, hv[5], tau[5]);
  qr9_step<6>(col, norm, hv[6], tau[6]);
  qr9_step<7>(col, norm, hv[7], tau[7]);
  qr9_step<8>(col, norm, hv[8], tau[8]);
  double q[9];
#pragma unroll
  for (int i = 0; i < 9; ++i) q[i] = i == lane ? 1.0 : 0.0;
#pragma unroll
  for (int k = 8; k >= 0; --k) {
    if (tau[k] == 0.0) continue;
    double w = 0.0;
#pragma unroll
    for (int i = k; i < 9; ++i) w += hv[k][i] * q[i];
    const double tw = tau[k] * w;
#pragma unroll
    for (int i = k; i < 9; ++i) q[i] = q[i] - tw * hv[k][i];
  }
  if (lane >= 5 && lane < 9) {
#pragma unroll
    for (int i = 0; i < 9; ++i) NS[i][lane - 5] = q[i];
  }
}

// The ten cubic constraints of the null space NS: column `lane` (< 20) of the
// 10 x 20 matrix in Stewenius order.
__device__ __forceinline__ void wave_constraints(const double (&NS)[9][4], StewShared& S, double (&col)[10]) {
  static constexpr TermTable T = make_terms(make_mul_table(kSteweniusOrder));
  const int lane = lane_id();
  if (lane < 36) {
    const int i = lane / 12, j = lane / 4 % 3, k = lane % 4;
    S.ee[i][j][k] = NS[3 * j + i][k];
  }
  __syncthreads();
  for (int e = lane; e < 120; e += 64) {
    const int k = e % 10;
    double v = 0.0;
    if (e < 90) {
      const int i = e / 30, j = e / 10 % 3;
#pragma unroll
      for (int m = 0; m < 3; ++m)
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const int c = T.t11[k][t];
          if (c >= 0) v = v + 2.0 * (S.ee[i][m][c >> 4] * S.ee[j][m][c & 15]);
        }
      S.eet[e / 10][k] = v;
    } else {
      // cofactor kk of the third row: entries (0, c1) (1, c2) - (0, c2) (1, c1)
      const int kk = e / 10 - 9;
      const int c1 = kk == 0 ? 1 : (kk == 1 ? 2 : 0), c2 = kk == 0 ? 2 : (kk == 1 ? 0 : 1);
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const int c = T.t11[k][t];
        if (c >= 0) v = v + 1.0 * (S.ee[0][c1][c >> 4] * S.ee[1][c2][c & 15]);
      }
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const int c = T.t11[k][t];
        if (c >= 0) v = v + -1.0 * (S.ee[0][c2][c >> 4] * S.ee[1][c1][c & 15]);
      }
      S.cof[kk][k] = v;
    }
  }
  __syncthreads();
  if (lane < 10) S.tr[lane] = S.eet[0][lane] + S.eet[4][lane] + S.eet[8][lane];
  __syncthreads();
  const int cl = lane < 20 ? lane : 19;
  const int c0 = T.t21[cl][0], c1 = T.t21[cl][1], c2 = T.t21[cl][2];
  auto add = [&](double v, const double* p, const double* q, double s) {
    v = v + s * (p[c0 >> 4] * q[c0 & 15]);
    if (c1 >= 0) v = v + s * (p[c1 >> 4] * q[c1 & 15]);
    if (c2 >= 0) v = v + s * (p[c2 >> 4] * q[c2 & 15]);
    return v;
  };
#pragma unroll
  for (int r = 0; r < 9; ++r) {
    const int i = r / 3, j = r % 3;
    double v = 0.0;
#pragma unroll
    for (int k = 0; k < 3; ++k) v = add(v, S.eet[3 * i + k], S.ee[k][j], 1.0);
    col[r] = add(v, S.tr, S.ee[i][j], -0.5);
  }
  {
    double v = 0.0;
#pragma unroll
    for (int k = 0; k < 3; ++k) v = add(v, S.cof[k], S.ee[2][k], 1.0);
    col[9] = v;
  }
}

// First maximum of |col[i]|, i >= K, in row order (strict >, from -1).
template <int K>
__device__ __forceinline__ void col_max(const double (&col)[10], double& best, int& bi) {
  best = -1.0;
  bi = K;
#pragma unroll
  for (int i = K; i < 10; ++i) {
    const bool take = fabs(col[i]) > best;
    best = take ? fabs(col[i]) : best;
    bi = take ? i : bi;
  }
}
template <int K>
__device__ __forceinline__ void row_swap(double (&col)[10], int p) {
#pragma unroll
  for (int i = K + 1; i < 10; ++i) {
    const bool sw = i == p;
    const double x = col[K];
    col[K] = sw ? col[i] : x;
    col[i] = sw ? x : col[i];
  }
}

// One step of the elimination with full pivoting (first maximum in row-major
// order): lanes 0 .. 9 the matrix, 10 .. 19 the right-hand sides.
template <int K>
__device__ __forceinline__ void lu_full_step(double (&col)[10], int& colp) {
  const int lane = lane_id();
  double best;
  int bi;
  col_max<K>(col, best, bi);
  const bool open = lane >= K && lane < 10;
  double gb;
  const int idx = wave_argmax_dpp(open ? best : -2.0, open ? 16 * bi + lane : 1024 + lane, gb);
  const int pr = idx >> 4, pc = idx & 15;
  row_swap<K>(col, pr);
  if (pc != K) {
    const int src = lane == K ? pc : (lane == pc ? K : lane);
#pragma unroll
    for (int i = 0; i < 10; ++i) col[i] = __shfl(col[i], src, 64);
    colp = __shfl(colp, src, 64);
  }
  if constexpr (K < 9) {
    // lane i > K forms row i's multiplier
    double num = 0.0;
#pragma unroll
    for (int i = K + 1; i < 10; ++i) {
      const double c = readlane_f64(col[i], K);
      num = lane == i ? c : num;
    }
    const double f = num / readlane_f64(col[K], K);
#pragma unroll
    for (int i = K + 1; i < 10; ++i) col[i] = col[i] - readlane_f64(f, i) * col[K];
  }
}

// Solves the 10 x 10 system with the ten right-hand sides; x[i]: row i of the
// permuted solution on lanes 10 .. 19; colp on lane i < 10: the unknown of
// that row.
__device__ __forceinline__ void wave_lu_full(double (&col)[10], double (&x)[10], int& colp) {
  colp = lane_id();
  lu_full_step<0>(col, colp);
  lu_full_step<1>(col, colp);
  lu_full_step<2>(col, colp);
  lu_full_step<3>(col, colp);
  lu_full_step<4>(col, colp);
  lu_full_step<5>(col, colp);
  lu_full_step<6>(col, colp);
  lu_full_step<7>(col, colp);
  lu_full_step<8>(col, colp);
  lu_full_step<9>(col, colp);
#pragma unroll
  for (int i = 9; i >= 0; --i) {
    double v = col[i];
#pragma unroll
    for (int k = i + 1; k < 10; ++k) v = v - readlane_f64(col[i], k) * x[k];
    x[i] = v / readlane_f64(col[i], i);
  }
}

// Real eigenvalues of the 10 x 10 matrix S.a, in diagonal order of the real
// Schur form, to S.evs; returns their number (-1: no convergence).
// Householder reduction to Hessenberg form, then Francis double-shift QR steps
// (Martin, Peters and Wilkinson, "The QR algorithm for real Hessenberg matrices",
// Numer. Math. 14, 1970).  The wave works on S.h: column operations with a lane
// per column, row operations with a lane per row, the searches with a lane per
// candidate; the scalar steps run on every lane alike.
__device__ inline int wave_real_eigenvalues(StewShared& S) {
  constexpr int n = 10;
  const int lane = lane_id();
  const int ln = lane < n ? lane : n - 1;
  const bool on = lane < n;
  double(&a)[10][10] = S.h;
  for (int e = lane; e < n * n; e += 64) a[e / n][e % n] = S.a[e / n][e % n];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < n - 2; ++k) {
    double v[10], sigma = 0.0;
#pragma unroll
    for (int i = k + 2; i < n; ++i) {
      v[i] = a[i][k];
      sigma += v[i] * v[i];
    }
    if (sigma == 0.0) continue;
    const double alpha = a[k + 1][k];
    const double nrm = sqrt(alpha * alpha + sigma);
    const double beta = alpha >= 0.0 ? -nrm : nrm;
    v[k + 1] = alpha - beta;
    double vv = 0.0;
#pragma unroll
    for (int i = k + 1; i < n; ++i) vv += v[i] * v[i];
    // A <- (I - 2 v v^T / vv) A (I - 2 v v^T / vv)
    {
      double c[10], s = 0.0;
#pragma unroll
      for (int i = k + 1; i < n; ++i) {
        c[i] = a[i][ln];
        s += v[i] * c[i];
      }
      s = 2.0 * s / vv;
      __syncthreads();
      if (on) {
#pragma unroll
        for (int i = k + 1; i < n; ++i) a[i][ln] = c[i] - s * v[i];
      }
    }
    __syncthreads();
    {
      double c[10], s = 0.0;
#pragma unroll
      for (int j = k + 1; j < n; ++j) {
        c[j] = a[ln][j];
        s += c[j] * v[j];
      }
      s = 2.0 * s / vv;
      __syncthreads();
      if (on) {
#pragma unroll
        for (int j = k + 1; j < n; ++j) a[ln][j] = c[j] - s * v[j];
        if (lane >= k + 2) a[lane][k] = 0.0;
      }
    }
    __syncthreads();
  }
  // double-shift QR on the active block, rows top .. bottom
  double size = 0.0;  // sum of the magnitudes, where a diagonal is all zero
  for (int i = 0; i < n; ++i)
    for (int j = (i - 1 > 0 ? i - 1 : 0); j < n; ++j) size += fabs(a[i][j]);
  const double eps = 2.220446049250313e-16;
  int nr = 0, steps = 0;
  double moved = 0.0;  // taken off the diagonal so far
  auto report = [&](int row, double value) {
    if (lane == 0) {
      S.pos[nr] = row;
      S.ev[nr] = value;
    }
    ++nr;
  };
  for (int bottom = n - 1; bottom >= 0;) {
    // the block begins below the last negligible subdiagonal entry
    int top;
    {
      bool small = false;
      if (lane >= 1 && lane <= bottom) {
        const double around = fabs(a[lane - 1][lane - 1]) + fabs(a[lane][lane]);
        small = fabs(a[lane][lane - 1]) <= eps * (around == 0.0 ? size : around);
      }
      const uint64_t b = ballot64(small);
      top = b ? 63 - __clzll((long long)b) : 0;
      if (b && lane == 0) a[top][top - 1] = 0.0;
    }
    __syncthreads();
    const double last = a[bottom][bottom];
    if (top == bottom) {
      report(bottom, last + moved);
      bottom -= 1;
      steps = 0;
      continue;
    }
    // the last 2 x 2 block (prev . ; . last): its product of off-diagonals
    const double prev = a[bottom - 1][bottom - 1], cross = a[bottom][bottom - 1] * a[bottom - 1][bottom];
    if (top + 1 == bottom) {
      const double half = 0.5 * (prev - last), disc = half * half + cross;
      if (disc >= 0.0) {
        // the root away from last first, the other by the product of both
        const double root = sqrt(disc), far = half >= 0.0 ? half + root : half - root, base = last + moved;
        report(bottom - 1, base + far);
        report(bottom, far != 0.0 ? base - cross / far : base + far);
      }
      bottom -= 2;
      steps = 0;
      continue;
    }
    if (steps == 30 * n) return -1;  // no convergence
    // the step's two shifts as the diagonal and the cross product of a block:
    // the last block, or after ten and twenty steps an ad hoc one
    double sh_last = last, sh_prev = prev, sh_cross = cross;
    if (steps == 10 || steps == 20) {
      moved += last;
      __syncthreads();
      if (lane <= bottom) a[lane][lane] -= last;
      __syncthreads();
      const double off = fabs(a[bottom][bottom - 1]) + fabs(a[bottom - 1][bottom - 2]);
      sh_last = sh_prev = 0.75 * off;
      sh_cross = -0.4375 * off * off;
    }
    ++steps;
    // first column of the shifted square, from the lowest row at which the
    // entries left of it hardly change under the step (a lane per row)
    int begin;
    double x0 = 0.0, x1 = 0.0, x2 = 0.0;
    {
      bool fits = false;
      if (lane >= top && lane <= bottom - 2) {
        const double at = a[lane][lane], dl = sh_last - at, dp = sh_prev - at;
        x0 = (dl * dp - sh_cross) / a[lane + 1][lane] + a[lane][lane + 1];
        x1 = a[lane + 1][lane + 1] - at - dl - dp;
        x2 = a[lane + 2][lane + 1];
        const double sum = fabs(x0) + fabs(x1) + fabs(x2);
        x0 /= sum;
        x1 /= sum;
        x2 /= sum;
        if (lane == top) {
          fits = true;
        } else {
          const double change = fabs(a[lane][lane - 1]) * (fabs(x1) + fabs(x2));
          const double diag = fabs(a[lane - 1][lane - 1]) + fabs(at) + fabs(a[lane + 1][lane + 1]);
          fits = change <= eps * (fabs(x0) * diag);
        }
      }
      begin = 63 - __clzll((long long)ballot64(fits));
      x0 = readlane_f64(x0, begin);
      x1 = readlane_f64(x1, begin);
      x2 = readlane_f64(x2, begin);
    }
    __syncthreads();
    if (lane >= begin + 2 && lane <= bottom) {
      a[lane][lane - 2] = 0.0;
      if (lane > begin + 2) a[lane][lane - 3] = 0.0;
    }
    __syncthreads();
    // chase: at every row a reflection of three (at the end two) rows and columns
    for (int row = begin; row < bottom; ++row) {
      const bool three = row + 1 < bottom;
      double scale = 0.0;
      if (row > begin) {
        x0 = a[row][row - 1];
        x1 = a[row + 1][row - 1];
        x2 = three ? a[row + 2][row - 1] : 0.0;
        scale = fabs(x0) + fabs(x1) + fabs(x2);
        if (scale != 0.0) {
          x0 /= scale;
          x1 /= scale;
          x2 /= scale;
        }
      }
      // I - u v^T with v = (1, v1, v2) takes x to (-length, 0, 0)
      const double norm = sqrt(x0 * x0 + x1 * x1 + x2 * x2), length = x0 >= 0.0 ? norm : -norm;
      if (length == 0.0) continue;
      if (lane == 0) {
        if (row > begin) a[row][row - 1] = -length * scale;
        else if (row > top) a[row][row - 1] = -a[row][row - 1];
      }
      const double head = x0 + length;
      const double u0 = head / length, u1 = x1 / length, u2 = x2 / length, v1 = x1 / head, v2 = x2 / head;
      __syncthreads();
      if (lane >= row && lane <= bottom) {
        double dot = a[row][lane] + v1 * a[row + 1][lane];
        if (three) {
          dot += v2 * a[row + 2][lane];
          a[row + 2][lane] -= dot * u2;
        }
        a[row + 1][lane] -= dot * u1;
        a[row][lane] -= dot * u0;
      }
      __syncthreads();
      if (lane >= top && lane <= (bottom < row + 3 ? bottom : row + 3)) {
        double dot = u0 * a[lane][row] + u1 * a[lane][row + 1];
        if (three) {
          dot += u2 * a[lane][row + 2];
          a[lane][row + 2] -= dot * v2;
        }
        a[lane][row + 1] -= dot * v1;
        a[lane][row] -= dot;
      }
      __syncthreads();
    }
  }
  __syncthreads();
  // diagonal order (top to bottom): the positions are distinct
  if (lane < nr) {
    int rank = 0;
    for (int j = 0; j < nr; ++j) rank += S.pos[j] < S.pos[lane] ? 1 : 0;
    S.evs[rank] = S.ev[lane];
  }
  __syncthreads();
  return nr;
}

// ---- null vectors: one matrix per row of 16 lanes -----------------------------
// (value, index) maximum over a row of 16 lanes (ties: smaller index), on every
// lane of the row.
__device__ __forceinline__ void row_argmax(double& v, int& idx) {
  argmax_step(v, idx, dpp_mov_f64<0x128>(v), dpp_mov_i32<0x128>(idx));
  argmax_step(v, idx, dpp_mov_f64<0x124>(v), dpp_mov_i32<0x124>(idx));
  argmax_step(v, idx, dpp_mov_f64<0x122>(v), dpp_mov_i32<0x122>(idx));
  argmax_step(v, idx, dpp_mov_f64<0x121>(v), dpp_mov_i32<0x121>(idx));
}

template <int K>
__device__ __forceinline__ void null_step(double (&col)[10], int& mine, int& rank, bool& open, double& first) {
  const int lane = lane_id(), c = lane & 15, row = lane & 48;
  double best;
  int bi;
  col_max<K>(col, best, bi);
  const bool elig = c >= K && c < 10;
  double v = elig ? best : -2.0;
  int idx = elig ? 16 * bi + c : 1024 + c;
  row_argmax(v, idx);
  if (K == 0) first = v;
  if (v <= 10.0 * 2.220446049250313e-16 * first || v == 0.0) open = false;
  const int pr = open ? idx >> 4 : K, pc = open ? idx & 15 : K;
  row_swap<K>(col, pr);
  const int src = row + (c == K ? pc : (c == pc ? K : c));
#pragma unroll
  for (int i = 0; i < 10; ++i) col[i] = __shfl(col[i], src, 64);
  mine = __shfl(mine, src, 64);
  if constexpr (K < 9) {
    // lane i > K of the row forms row i's multiplier
    double num = 0.0;
#pragma unroll
    for (int i = K + 1; i < 10; ++i) {
      const double t = __shfl(col[i], row + K, 64);
      num = c == i ? t : num;
    }
    const double f = num / __shfl(col[K], row + K, 64);
#pragma unroll
    for (int i = K + 1; i < 10; ++i) {
      const double fi = __shfl(f, row + i, 64);
      if (open && c > K) col[i] = col[i] - fi * col[K];
    }
  }
  rank += open ? 1 : 0;
}

// Null vectors of a - evs[q] I, q < ne, by elimination with full pivoting, to
// S.vec[q]; four eigenvalues at a time.
__device__ inline void wave_null_vectors(StewShared& S, int ne) {
  const int lane = lane_id(), c = lane & 15, row = lane & 48;
  for (int q0 = 0; q0 < ne; q0 += 4) {
    const int q = q0 + (lane >> 4);
    const double ev = S.evs[q < ne ? q : ne - 1];
    const int cc = c < 10 ? c : 9;
    double col[10];
#pragma unroll
    for (int i = 0; i < 10; ++i) {
      const double v = S.a[i][cc];
      col[i] = i == c ? v - ev : v;
    }
    int mine = cc, rank = 0;
    bool open = true;
    double first = 0.0;
    null_step<0>(col, mine, rank, open, first);
    null_step<1>(col, mine, rank, open, first);
    null_step<2>(col, mine, rank, open, first);
    null_step<3>(col, mine, rank, open, first);
    null_step<4>(col, mine, rank, open, first);
    null_step<5>(col, mine, rank, open, first);
    null_step<6>(col, mine, rank, open, first);
    null_step<7>(col, mine, rank, open, first);
    null_step<8>(col, mine, rank, open, first);
    null_step<9>(col, mine, rank, open, first);
    const int fr = rank < 10 ? rank : 9;  // the free unknown (in pivoted order)
    double z = c == fr ? 1.0 : 0.0;
#pragma unroll
    for (int k = 8; k >= 0; --k) {
      double s = 0.0;
#pragma unroll
      for (int j = k + 1; j < 10; ++j) {
        const double t = __shfl(col[k] * z, row + j, 64);
        s = j <= fr ? s + t : s;
      }
      const double zk = -s / __shfl(col[k], row + k, 64);
      if (c == k && k < fr) z = zk;
    }
    if (q < ne && c < 10) S.vec[q][mine] = z;
  }
  __syncthreads();
}

}  // namespace gcr
