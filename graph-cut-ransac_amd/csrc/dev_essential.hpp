// Device numerics of the essential-matrix path (gfx950).
//
// Thread-level routines (one thread runs each call): the monomial tables of
// both solvers, the five-point null space, the Sturm-sequence roots of the
// degree-10 polynomial and the relative-pose helpers of the bundle adjustment.
// They use only +, -, *, / and sqrt in a fixed order and
// are compiled without fused multiply-add, so results are reproducible
// bit for bit by a sequential host restatement of the same steps.
//
// Reference: inc/estimators/solver_essential_matrix_five_point_nister.h,
// solver_essential_matrix_five_point_stewenius.h,
// inc/maths/sturm_polynomial_solver.h, inc/relative_pose/{essential.cpp,
// bundle.cpp,bundle.h,jacobian_impl.h}.
#pragma once

#include "dev_common.hpp"
#include "dev_fundamental.hpp"

namespace gcr {

template <class T>
__device__ __forceinline__ void gswap(T& a, T& b) {
  T t = a;
  a = b;
  b = t;
}

// ---- monomials of x, y, z ----------------------------------------------------
// Nister order: degree 2 [x^2, xy, xz, x, y^2, yz, y, z^2, z, 1], degree 3
// [x^3, y^3, x^2y, xy^2, x^2z, x^2, y^2z, y^2, xyz, xy, xz^2, xz, x, yz^2,
// yz, y, z^3, z^2, z, 1]; Stewenius order: degree 2 [x^2, xy, y^2, xz, yz,
// z^2, x, y, z, 1], degree 3 [x^3, x^2y, xy^2, y^3, x^2z, xyz, y^2z, xz^2,
// yz^2, z^3, x^2, xy, y^2, xz, yz, z^2, x, y, z, 1].  Degree 1 is [x, y, z, 1].
// A monomial is encoded as 16 a + 4 b + c (exponents of x, y, z).
struct MonoOrder {
  int d2[10];
  int d3[20];
};
constexpr int mono_code(int a, int b, int c) { return 16 * a + 4 * b + c; }
constexpr int kDeg1Code[4] = {mono_code(1, 0, 0), mono_code(0, 1, 0), mono_code(0, 0, 1), mono_code(0, 0, 0)};
constexpr MonoOrder kNisterOrder = {
    {mono_code(2, 0, 0), mono_code(1, 1, 0), mono_code(1, 0, 1), mono_code(1, 0, 0), mono_code(0, 2, 0),
     mono_code(0, 1, 1), mono_code(0, 1, 0), mono_code(0, 0, 2), mono_code(0, 0, 1), mono_code(0, 0, 0)},
    {mono_code(3, 0, 0), mono_code(0, 3, 0), mono_code(2, 1, 0), mono_code(1, 2, 0), mono_code(2, 0, 1),
     mono_code(2, 0, 0), mono_code(0, 2, 1), mono_code(0, 2, 0), mono_code(1, 1, 1), mono_code(1, 1, 0),
     mono_code(1, 0, 2), mono_code(1, 0, 1), mono_code(1, 0, 0), mono_code(0, 1, 2), mono_code(0, 1, 1),
     mono_code(0, 1, 0), mono_code(0, 0, 3), mono_code(0, 0, 2), mono_code(0, 0, 1), mono_code(0, 0, 0)}};
constexpr MonoOrder kSteweniusOrder = {
    {mono_code(2, 0, 0), mono_code(1, 1, 0), mono_code(0, 2, 0), mono_code(1, 0, 1), mono_code(0, 1, 1),
     mono_code(0, 0, 2), mono_code(1, 0, 0), mono_code(0, 1, 0), mono_code(0, 0, 1), mono_code(0, 0, 0)},
    {mono_code(3, 0, 0), mono_code(2, 1, 0), mono_code(1, 2, 0), mono_code(0, 3, 0), mono_code(2, 0, 1),
     mono_code(1, 1, 1), mono_code(0, 2, 1), mono_code(1, 0, 2), mono_code(0, 1, 2), mono_code(0, 0, 3),
     mono_code(2, 0, 0), mono_code(1, 1, 0), mono_code(0, 2, 0), mono_code(1, 0, 1), mono_code(0, 1, 1),
     mono_code(0, 0, 2), mono_code(1, 0, 0), mono_code(0, 1, 0), mono_code(0, 0, 1), mono_code(0, 0, 0)}};

// Product index tables: out index of (degree-1 i) x (degree-1 j) and of
// (degree-2 i) x (degree-1 j) in each order (compile-time).
struct MulTable {
  int m11[16];
  int m21[40];
};
constexpr int find_code(const int* t, int n, int code) {
  for (int i = 0; i < n; ++i)
    if (t[i] == code) return i;
  return -1;
}
constexpr MulTable make_mul_table(const MonoOrder& o) {
  MulTable t{};
  for (int i = 0; i < 4; ++i)
    for (int j = 0; j < 4; ++j) t.m11[4 * i + j] = find_code(o.d2, 10, kDeg1Code[i] + kDeg1Code[j]);
  for (int i = 0; i < 10; ++i)
    for (int j = 0; j < 4; ++j) t.m21[4 * i + j] = find_code(o.d3, 20, o.d2[i] + kDeg1Code[j]);
  return t;
}

// Coefficient row of one correspondence for vec(E) stacked column by column:
// row . vec(E) = x2^T E x1.
__device__ __forceinline__ void e_row(const double* p, double w, double* r) {
  const double x0 = p[0], y0 = p[1], x1 = p[2], y1 = p[3];
  const double wx0 = w * x0, wx1 = w * x1, wy0 = w * y0, wy1 = w * y1;
  r[0] = wx0 * x1;
  r[1] = wx0 * y1;
  r[2] = wx0;
  r[3] = wy0 * x1;
  r[4] = wy0 * y1;
  r[5] = wy0;
  r[6] = wx1;
  r[7] = wy1;
  r[8] = w;
}

// Null space of the 5 x 9 coefficient matrix: N[9 k + j], k < 4.  False when
// the rank is below 5.
__device__ __forceinline__ bool null_space_5x9(double (&a)[5][9], double* N) {
  uint32_t used = 0, row_of_col = 0;  // 3 bits per pivot column: its row
  double max_pivot = 0.0;
  bool ok = true;
#pragma unroll
  for (int r = 0; r < 5; ++r) {
    double best = 0.0;
    int pr = -1, pc = -1;
#pragma unroll
    for (int i = r; i < 5; ++i)
#pragma unroll
      for (int j = 0; j < 9; ++j) {
        const double v = fabs(a[i][j]);
        const bool take = !((used >> j) & 1u) && v > best;
        best = take ? v : best;
        pr = take ? i : pr;
        pc = take ? j : pc;
      }
    if (r == 0) max_pivot = best;
    if (pr < 0 || best <= 5.0 * 2.220446049250313e-16 * max_pivot) ok = false;
    if (!ok) continue;
#pragma unroll
    for (int i = r + 1; i < 5; ++i) {
      const bool sw = i == pr;
#pragma unroll
      for (int j = 0; j < 9; ++j) {
        const double t = a[r][j];
        a[r][j] = sw ? a[i][j] : t;
        a[i][j] = sw ? t : a[i][j];
      }
    }
    double piv = a[r][0];
#pragma unroll
    for (int j = 1; j < 9; ++j) piv = j == pc ? a[r][j] : piv;
#pragma unroll
    for (int j = 0; j < 9; ++j) a[r][j] = a[r][j] / piv;
#pragma unroll
    for (int i = 0; i < 5; ++i) {
      if (i == r) continue;
      double f = a[i][0];
#pragma unroll
      for (int j = 1; j < 9; ++j) f = j == pc ? a[i][j] : f;
      const bool upd = f != 0.0;
#pragma unroll
      for (int j = 0; j < 9; ++j) a[i][j] = upd ? a[i][j] - f * a[r][j] : a[i][j];
    }
    used |= 1u << pc;
    row_of_col |= (uint32_t)r << (3 * pc);
  }
  if (!ok) return false;
  uint32_t freem = ~used & 0x1ffu;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int fc = __builtin_ctz(freem);
    freem &= freem - 1u;
    double v[5];
#pragma unroll
    for (int r = 0; r < 5; ++r) {
      double x = a[r][0];
#pragma unroll
      for (int j = 1; j < 9; ++j) x = j == fc ? a[r][j] : x;
      v[r] = -x;
    }
#pragma unroll
    for (int j = 0; j < 9; ++j) {
      const int r = (int)((row_of_col >> (3 * j)) & 7u);
      double x = v[0];
#pragma unroll
      for (int i = 1; i < 5; ++i) x = i == r ? v[i] : x;
      N[9 * k + j] = ((used >> j) & 1u) ? x : (j == fc ? 1.0 : 0.0);
    }
  }
  return true;
}

struct RelPose {
  double q[4];  // unit quaternion (w, x, y, z)
  double t[3];
};

__device__ inline double dot3(const double* a, const double* b) { return a[0] * b[0] + a[1] * b[1] + a[2] * b[2]; }

__device__ inline void solve3x2_fullpiv(const double* b0, const double* b1, const double* rhs, double* xz) {
  double a[3][2] = {{b0[0], b1[0]}, {b0[1], b1[1]}, {b0[2], b1[2]}};
  double r[3] = {rhs[0], rhs[1], rhs[2]};
  int col[2] = {0, 1};
  int rank = 0;
  double first = 0.0;
  for (int k = 0; k < 2; ++k) {
    int pr = k, pc = k;
    double best = -1.0;
    for (int i = k; i < 3; ++i)
      for (int j = k; j < 2; ++j)
        if (fabs(a[i][j]) > best) {
          best = fabs(a[i][j]);
          pr = i;
          pc = j;
        }
    if (k == 0) first = best;
    if (best <= 2.0 * 2.220446049250313e-16 * first || best == 0.0) break;
    if (pr != k) {
      for (int j = 0; j < 2; ++j) gswap(a[k][j], a[pr][j]);
      gswap(r[k], r[pr]);
    }
    if (pc != k) {
      for (int i = 0; i < 3; ++i) gswap(a[i][k], a[i][pc]);
      gswap(col[k], col[pc]);
    }
    for (int i = k + 1; i < 3; ++i) {
      const double f = a[i][k] / a[k][k];
      for (int j = k + 1; j < 2; ++j) a[i][j] = a[i][j] - f * a[k][j];
      r[i] = r[i] - f * r[k];
    }
    ++rank;
  }
  double z[2] = {0.0, 0.0};
  for (int k = rank - 1; k >= 0; --k) {
    double v = r[k];
    for (int j = k + 1; j < rank; ++j) v = v - a[k][j] * z[j];
    z[k] = v / a[k][k];
  }
  xz[col[0]] = z[0];
  xz[col[1]] = z[1];
}

__device__ inline void frobenius_normalise_sign(double* m) {
  double z = 0.0;
  for (int i = 0; i < 9; ++i) z += m[i] * m[i];
  if (z > 0.0) {
    const double s = sqrt(z);
    for (int i = 0; i < 9; ++i) m[i] /= s;
  }
  if (m[8] < 0)
    for (int i = 0; i < 9; ++i) m[i] = -m[i];
}

__device__ inline void quat_to_R(const double* q, double* R) {
  const double w = q[0], x = q[1], y = q[2], z = q[3];
  const double tx = 2 * x, ty = 2 * y, tz = 2 * z;
  const double twx = tx * w, twy = ty * w, twz = tz * w;
  const double txx = tx * x, txy = ty * x, txz = tz * x;
  const double tyy = ty * y, tyz = tz * y, tzz = tz * z;
  R[0] = 1 - (tyy + tzz);
  R[1] = txy - twz;
  R[2] = txz + twy;
  R[3] = txy + twz;
  R[4] = 1 - (txx + tzz);
  R[5] = tyz - twx;
  R[6] = txz - twy;
  R[7] = tyz + twx;
  R[8] = 1 - (txx + tyy);
}

__device__ inline void R_to_quat(const double* R, double* q) {
  auto m = [&](int i, int j) { return R[3 * i + j]; };
  double w, v[3];
  double t = m(0, 0) + m(1, 1) + m(2, 2);
  if (t > 0) {
    t = sqrt(t + 1.0);
    w = 0.5 * t;
    t = 0.5 / t;
    v[0] = (m(2, 1) - m(1, 2)) * t;
    v[1] = (m(0, 2) - m(2, 0)) * t;
    v[2] = (m(1, 0) - m(0, 1)) * t;
  } else {
    int i = 0;
    if (m(1, 1) > m(0, 0)) i = 1;
    if (m(2, 2) > m(i, i)) i = 2;
    const int j = (i + 1) % 3, k = (j + 1) % 3;
    t = sqrt(m(i, i) - m(j, j) - m(k, k) + 1.0);
    v[i] = 0.5 * t;
    t = 0.5 / t;
    w = (m(k, j) - m(j, k)) * t;
    v[j] = (m(j, i) + m(i, j)) * t;
    v[k] = (m(k, i) + m(i, k)) * t;
  }
  const double nrm = sqrt(w * w + v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
  q[0] = w / nrm;
  q[1] = v[0] / nrm;
  q[2] = v[1] / nrm;
  q[3] = v[2] / nrm;
}

__device__ inline void cross3(const double* a, const double* b, double* c) {
  c[0] = a[1] * b[2] - a[2] * b[1];
  c[1] = a[2] * b[0] - a[0] * b[2];
  c[2] = a[0] * b[1] - a[1] * b[0];
}

__device__ inline void normalise3(double* a) {
  const double n = sqrt(dot3(a, a));
  for (int i = 0; i < 3; ++i) a[i] /= n;
}

__device__ inline void essential_from_motion(const RelPose& p, double* E) {
  double R[9];
  quat_to_R(p.q, R);
  const double tx[9] = {0.0, -p.t[2], p.t[1], p.t[2], 0.0, -p.t[0], -p.t[1], p.t[0], 0.0};
  mat3_mul(tx, R, E);
}

__device__ inline bool check_cheirality(const RelPose& p, const double* x1, const double* x2) {
  double R[9], Rx1[3];
  quat_to_R(p.q, R);
  for (int i = 0; i < 3; ++i) Rx1[i] = R[3 * i] * x1[0] + R[3 * i + 1] * x1[1] + R[3 * i + 2] * x1[2];
  const double a = -dot3(Rx1, x2);
  const double b1 = -dot3(Rx1, p.t);
  const double b2 = dot3(x2, p.t);
  const double l1 = b1 - a * b2;
  const double l2 = -a * b1 + b2;
  const double md = 0.0 * (1 - a * a);
  return l1 > md && l2 > md;
}

__device__ inline double relpose_r2(const double* E, const double* p, double* JC, double* Cout) {
  const double x1 = p[0], y1 = p[1], x2 = p[2], y2 = p[3];
  const double e0 = E[0] * x1 + E[1] * y1 + E[2];
  const double e1 = E[3] * x1 + E[4] * y1 + E[5];
  const double e2 = E[6] * x1 + E[7] * y1 + E[8];
  const double C = x2 * e0 + y2 * e1 + e2;
  const double g0 = E[0] * x2 + E[3] * y2 + E[6];
  const double g1 = E[1] * x2 + E[4] * y2 + E[7];
  if (JC) {
    JC[0] = g0;
    JC[1] = g1;
    JC[2] = e0;
    JC[3] = e1;
  }
  if (Cout) *Cout = C;
  return (C * C) / ((e0 * e0 + e1 * e1) + (g0 * g0 + g1 * g1));
}

// The four (R, t) of E from cross products of its columns (essential.cpp:25-80),
// kept when the correspondence (x1, x2) is in front of both cameras, in the
// order (R_a, t), (R_a, -t), (R_b, t), (R_b, -t).  Returns their number.
__device__ inline int motion_from_essential_dev(const double* Erm, const double* x1, const double* x2,
                                                RelPose* out) {
  double c[3][3];  // columns of E
  for (int j = 0; j < 3; ++j)
    for (int i = 0; i < 3; ++i) c[j][i] = Erm[3 * i + j];
  double u12[3], u13[3], u23[3];
  cross3(c[0], c[1], u12);
  cross3(c[0], c[2], u13);
  cross3(c[1], c[2], u23);
  const double n12 = dot3(u12, u12), n13 = dot3(u13, u13), n23 = dot3(u23, u23);
  double UW[3][3];  // columns
  const double* col1;
  const double* u;
  double nu;
  if (n12 > n13) {
    if (n12 > n23) {
      col1 = c[0];
      u = u12;
      nu = n12;
    } else {
      col1 = c[1];
      u = u23;
      nu = n23;
    }
  } else {
    if (n13 > n23) {
      col1 = c[0];
      u = u13;
      nu = n13;
    } else {
      col1 = c[1];
      u = u23;
      nu = n23;
    }
  }
  {
    double v[3] = {col1[0], col1[1], col1[2]};
    normalise3(v);
    const double sq = sqrt(nu);
    for (int i = 0; i < 3; ++i) {
      UW[1][i] = v[i];
      UW[2][i] = u[i] / sq;
    }
  }
  double tmp[3];
  cross3(UW[2], UW[1], tmp);
  for (int i = 0; i < 3; ++i) UW[0][i] = -tmp[i];
  double Vt[3][3];
  for (int j = 0; j < 3; ++j) {
    Vt[0][j] = UW[1][0] * c[j][0] + UW[1][1] * c[j][1] + UW[1][2] * c[j][2];
    Vt[1][j] = -(UW[0][0] * c[j][0] + UW[0][1] * c[j][1] + UW[0][2] * c[j][2]);
  }
  normalise3(Vt[0]);
  const double d01 = dot3(Vt[0], Vt[1]);
  for (int j = 0; j < 3; ++j) Vt[1][j] -= d01 * Vt[0][j];
  normalise3(Vt[1]);
  cross3(Vt[0], Vt[1], Vt[2]);
  int cnt = 0;
  RelPose p;
  double R[9];
  for (int i = 0; i < 3; ++i)
    for (int j = 0; j < 3; ++j) R[3 * i + j] = UW[0][i] * Vt[0][j] + UW[1][i] * Vt[1][j] + UW[2][i] * Vt[2][j];
  R_to_quat(R, p.q);
  for (int i = 0; i < 3; ++i) p.t[i] = UW[2][i];
  if (check_cheirality(p, x1, x2)) out[cnt++] = p;
  for (int i = 0; i < 3; ++i) p.t[i] = -p.t[i];
  if (check_cheirality(p, x1, x2)) out[cnt++] = p;
  for (int k = 0; k < 2; ++k)
    for (int i = 0; i < 3; ++i) UW[k][i] = -UW[k][i];
  for (int i = 0; i < 3; ++i)
    for (int j = 0; j < 3; ++j) R[3 * i + j] = UW[0][i] * Vt[0][j] + UW[1][i] * Vt[1][j] + UW[2][i] * Vt[2][j];
  R_to_quat(R, p.q);
  if (check_cheirality(p, x1, x2)) out[cnt++] = p;
  for (int i = 0; i < 3; ++i) p.t[i] = -p.t[i];
  if (check_cheirality(p, x1, x2)) out[cnt++] = p;
  return cnt;
}

// ---- Sturm-sequence roots of a degree-10 polynomial ----------------------------
// The steps of this solver follow PoseLib's Sturm-sequence solver as the
// reference ships it (inc/maths/sturm_polynomial_solver.h), which carries
// this licence:
//   Copyright (c) 2020, Viktor Larsson.  All rights reserved.
//   Redistribution and use in source and binary forms, with or without
//   modification, are permitted provided that the following conditions are
//   met: (1) Redistributions of source code must retain the above copyright
//   notice, this list of conditions and the following disclaimer.
//   (2) Redistributions in binary form must reproduce the above copyright
//   notice, this list of conditions and the following disclaimer in the
//   documentation and/or other materials provided with the distribution.
//   (3) Neither the name of the copyright holder nor the names of its
//   contributors may be used to endorse or promote products derived from
//   this software without specific prior written permission.
//   THIS SOFTWARE IS PROVIDED BY THE COPYRIGHT HOLDERS AND CONTRIBUTORS "AS
//   IS" AND ANY EXPRESS OR IMPLIED WARRANTIES, INCLUDING, BUT NOT LIMITED TO,
//   THE IMPLIED WARRANTIES OF MERCHANTABILITY AND FITNESS FOR A PARTICULAR
//   PURPOSE ARE DISCLAIMED. IN NO EVENT SHALL THE COPYRIGHT HOLDER BE LIABLE
//   FOR ANY DIRECT, INDIRECT, INCIDENTAL, SPECIAL, EXEMPLARY, OR CONSEQUENTIAL
//   DAMAGES (INCLUDING, BUT NOT LIMITED TO, PROCUREMENT OF SUBSTITUTE GOODS OR
//   SERVICES; LOSS OF USE, DATA, OR PROFITS; OR BUSINESS INTERRUPTION) HOWEVER
//   CAUSED AND ON ANY THEORY OF LIABILITY, WHETHER IN CONTRACT, STRICT
//   LIABILITY, OR TORT (INCLUDING NEGLIGENCE OR OTHERWISE) ARISING IN ANY WAY
//   OUT OF THE USE OF THIS SOFTWARE, EVEN IF ADVISED OF THE POSSIBILITY OF
//   SUCH DAMAGE.
//
// Monic polynomial and normalised derivative, the Sturm sequence by
// pseudo-division with -|leading| scaling, sign changes by the three-term
// recurrence; the caller isolates the roots by bisection (depth <= 30, left
// half first); Ridders' method to width 1e-3, then up to ten Newton steps
// (tolerance 1e-10).  Every index is a compile-time constant, so the
// coefficients stay in registers.
struct SturmSeq10 {
  static constexpr int N = 10;
  double f[N + 1];  // monic, ascending
  double d[N];      // derivative / N
  double s[3 * N];

  template <int DEG>
  __device__ static __forceinline__ double eval(const double* p, double x) {
    double v = x + p[DEG - 1];
#pragma unroll
    for (int i = DEG - 2; i >= 0; --i) v = x * v + p[i];
    return v;
  }

  // one pseudo-division: f3 (N - 1 - I entries) from f1, f2
  template <int I>
  __device__ __forceinline__ void divide(const double* f1, const double* f2, double* f3) {
    const double q1 = f1[N - I] * f2[N - 1 - I];
    const double q0 = f1[N - 1 - I] * f2[N - 1 - I] - f1[N - I] * f2[N - 2 - I];
    f3[0] = f1[0] - q0 * f2[0];
#pragma unroll
    for (int j = 1; j < N - 1 - I; ++j) f3[j] = f1[j] - q1 * f2[j - 1] - q0 * f2[j];
    const double c = -fabs(f3[N - 2 - I]);
    const double ci = 1.0 / c;
#pragma unroll
    for (int j = 0; j < N - 1 - I; ++j) f3[j] = f3[j] * ci;
    s[3 * I] = q0;
    s[3 * I + 1] = q1;
    s[3 * I + 2] = c;
  }

  // coefficients ascending (11); false when the leading one is zero
  __device__ __forceinline__ bool init(const double* coeffs) {
    if (coeffs[N] == 0.0) return false;
    const double ci = 1.0 / coeffs[N];
#pragma unroll
    for (int i = 0; i < N; ++i) f[i] = coeffs[i] * ci;
    f[N] = 1.0;
#pragma unroll
    for (int i = 0; i < N - 1; ++i) d[i] = f[i + 1] * ((i + 1) / static_cast<double>(N));
    d[N - 1] = 1.0;
    double f3[9], f4[8], f5[7], f6[6], f7[5], f8[4], f9[3], f10[2], f11[1];
    divide<0>(f, d, f3);
    divide<1>(d, f3, f4);
    divide<2>(f3, f4, f5);
    divide<3>(f4, f5, f6);
    divide<4>(f5, f6, f7);
    divide<5>(f6, f7, f8);
    divide<6>(f7, f8, f9);
    divide<7>(f8, f9, f10);
    divide<8>(f9, f10, f11);
    s[3 * N - 3] = f10[0];
    s[3 * N - 2] = f10[1];
    s[3 * N - 1] = f11[0];
    return true;
  }

  // every real root lies within this distance of zero
  __device__ __forceinline__ double root_bound() const {
    double mx = 0.0;
#pragma unroll
    for (int i = 0; i < N; ++i) mx = fmax(mx, fabs(f[i]));
    return 1.0 + mx;
  }

  __device__ __forceinline__ int sign_changes(double x) const {
    double g2 = s[3 * N - 1];
    double g1 = s[3 * N - 3] + x * s[3 * N - 2];
    int cnt = (g1 < 0) != (g2 < 0) ? 1 : 0;
#pragma unroll
    for (int i = N - 2; i >= 0; --i) {
      const double g = (s[3 * i] + x * s[3 * i + 1]) * g1 + s[3 * i + 2] * g2;
      cnt += (g < 0) != (g1 < 0) ? 1 : 0;
      g2 = g1;
      g1 = g;
    }
    return cnt;
  }

  // the root in (a, b); false when the polynomial has the same sign at both
  __device__ __forceinline__ bool refine(double a, double b, double tol, double& root) const {
    double fa = eval<N>(f, a), fb = eval<N>(f, b);
    if (!((fa < 0) ^ (fb < 0))) return false;
    for (int it = 0; it < 30; ++it) {
      if (fabs(a - b) < 1e-3) break;
      const double c = (a + b) * 0.5;
      const double fc = eval<N>(f, c);
      const double sq = sqrt(fc * fc - fa * fb);
      if (!sq) break;
      const double x = (fa < fb) ? c + (a - c) * fc / sq : c + (c - a) * fc / sq;
      const double fx = eval<N>(f, x);
      if (fx >= 0 ? (fc < 0) : (fc > 0)) {
        a = c;
        fa = fc;
        b = x;
        fb = fx;
      } else if (fx >= 0 ? (fa < 0) : (fa > 0)) {
        b = x;
        fb = fx;
      } else {
        a = x;
        fa = fx;
      }
    }
    double x = (a + b) * 0.5;
    for (int it = 0; it < 10; ++it) {
      const double fx = eval<N>(f, x);
      if (fabs(fx) < tol) break;
      const double fpx = static_cast<double>(N) * eval<N - 1>(d, x);
      const double dx = fx / fpx;
      x = x - dx;
      if (fabs(dx) < tol) break;
    }
    root = x;
    return true;
  }
};

}  // namespace gcr
