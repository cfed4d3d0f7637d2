// Matrix-core scoring: the numbers of the rejection test (k_score_mx.hip has the
// reasons), before they are split into FP16 parts.
// Plain functions of numbers, for the kernels and for host code.
#pragma once

#include <cmath>

#if defined(__HIP__)
#define GCR_MX_FN __host__ __device__ __forceinline__
#else
#define GCR_MX_FN inline
#endif

namespace gcr {

constexpr double kMxDeltaRel = 0x1p-17;
constexpr double kMxDeltaAbs = 0x1p-20;
constexpr double kMxMargin = 1.0 + 0x1p-14;
constexpr double kMxEta = 0x1p-4;

// The scales of one pair's test: the quantities C (P, Q) are taken times sigma
// and the denominator form D times kappa, so that the test compares numbers
// near 1: sigma the power of two that brings kappa = 4 tau''^2 (1 + 2^-14)
// (1 + h) sigma^2 into [1, 4), at most 2^12 (FP16 coefficients).  Thresholds
// of half the points' range and more, and ones that are no numbers, drop nothing.
struct MxScale {
  double sigma, kappa;
  bool on;
};
GCR_MX_FN MxScale mx_scale(double sq_thr, double inv_scale) {
  MxScale r;
  const double q = 4.0 * (sq_thr * inv_scale * inv_scale) * kMxMargin * (1.0 + kMxEta);
  r.on = q >= 0.0 && q < 1.0;
  r.sigma = 1.0;
  r.kappa = r.on ? q : 0.0;
#pragma unroll 1
  for (int e = 0; e < 12 && r.kappa < 1.0; ++e) {
    r.sigma *= 2.0;
    r.kappa *= 4.0;
  }
  return r;
}

// One model's coefficient vectors over z (row-major 3x3 M): Sampson C;
// transfer P, Q.
template <int KIND>
GCR_MX_FN void mx_quantities(const double* F, double c[][9]) {
  constexpr int NQ = KIND == 1 ? 1 : 2;
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
  }
}

// A quarter of the denominator as a linear form in d = (x1^2, x1 y1, y1^2, x1,
// y1, the same of the second image, 1): (F x1)_0^2 + (F x1)_1^2 + (F^T x2)_0^2 +
// (F^T x2)_1^2, or W^2.  Every coefficient is at most 1 when |F| <= 1.
template <int KIND>
GCR_MX_FN void mx_denominator(const double* F, double g[11]) {
  g[10] = 0.0;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    double a[3], b[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      a[k] = KIND == 1 ? (h ? F[3 * k] : F[k]) : (h ? 0.0 : F[6 + k]);
      b[k] = KIND == 1 ? (h ? F[3 * k + 1] : F[3 + k]) : 0.0;
    }
    g[5 * h] = 0.25 * (a[0] * a[0] + b[0] * b[0]);
    g[5 * h + 1] = 0.5 * (a[0] * a[1] + b[0] * b[1]);
    g[5 * h + 2] = 0.25 * (a[1] * a[1] + b[1] * b[1]);
    g[5 * h + 3] = 0.5 * (a[0] * a[2] + b[0] * b[2]);
    g[5 * h + 4] = 0.5 * (a[1] * a[2] + b[1] * b[2]);
    g[10] += 0.25 * (a[2] * a[2] + b[2] * b[2]);
  }
}

// A scaled point's terms: z = x2 (x) x1 and the squared terms d.
GCR_MX_FN void mx_terms(double x1, double y1, double x2, double y2, double z[9], double d[11]) {
  const double zv[9] = {x2 * x1, x2 * y1, x2, y2 * x1, y2 * y1, y2, x1, y1, 1.0};
  const double dv[11] = {x1 * x1, x1 * y1, y1 * y1, x1, y1, x2 * x2, x2 * y2, y2 * y2, x2, y2, 1.0};
#pragma unroll
  for (int t = 0; t < 9; ++t) z[t] = zv[t];
#pragma unroll
  for (int t = 0; t < 11; ++t) d[t] = dv[t];
}

// The slack of a scaled point's test.
GCR_MX_FN float mx_slack(const MxScale& sc, double x1, double y1, double x2, double y2) {
  const double ax = fabs(x1), ay = fabs(y1), bx = fabs(x2), by = fabs(y2);
  const double sa = 1.0 + ax + ay, sb = 1.0 + bx + by;
  const double sd = 1.0 + ax * sa + ay * (1.0 + ay) + bx * sb + by * (1.0 + by);
  const double dc = sc.sigma * (kMxDeltaRel * (sa * sb) + kMxDeltaAbs);
  const double dd = (sc.kappa > 1.0 ? sc.kappa : 1.0) * (kMxDeltaRel * sd + kMxDeltaAbs);
  const double k = kMxMargin * (dd + (1.0 + 1.0 / kMxEta) * dc * dc);
  return k < 1e30 ? (float)k : 1.0f;
}

// A row-major 3 x 3 model in the scaled coordinates (x' = x / s on the scale of
// its pair, s a power of two), normalised to max |F| = 1: S F S, S = diag(s, s,
// 1), for the Sampson distance (KIND 1), S^-1 H S for the transfer error (KIND
// 0).  Nine zeros, with which nothing is dropped, for a model that is not to be
// tested, has an entry that is not finite, here or scaled, or is so near zero that
// 1 / max |F| is not finite.
template <int KIND>
GCR_MX_FN void mx_normalise(const double* M, double s, bool test, double* F) {
  const double sc[3] = {s, s, 1.0};
  double mx = 0.0;
  bool finite = true;
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const double v = KIND == 1 ? M[3 * i + k] * sc[i] * sc[k] : M[3 * i + k] / sc[i] * sc[k];
      finite = finite && fabs(v) <= 1e300;
      mx = fabs(v) > mx ? fabs(v) : mx;
      F[3 * i + k] = v;
    }
  const bool ok = test && finite && mx >= 1e-300;
  const double inv_mx = ok ? 1.0 / mx : 0.0;
#pragma unroll
  for (int k = 0; k < 9; ++k) F[k] = ok ? F[k] * inv_mx : 0.0;
}

}  // namespace gcr
