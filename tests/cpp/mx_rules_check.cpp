// The numbers of the matrix-core rejection (csrc/mx_rules.hpp) for a host test:
// models' and points' operands before they are split, the slack and the scales.
#include <cstdint>

#include "mx_rules.hpp"

using namespace gcr;

extern "C" {

// out per model: 9 normalised entries, 2 x 9 quantity coefficients (the second
// zero for the Sampson distance), 11 denominator coefficients
void mx_models(int32_t kind, int64_t count, const double* models, double s, double sq_thr, double* out) {
  const MxScale sc = mx_scale(sq_thr, 1.0 / s);
  for (int64_t m = 0; m < count; ++m) {
    double* o = out + 38 * m;
    double cq[2][9] = {};
    if (kind == 1) {
      mx_normalise<1>(models + 9 * m, s, sc.on, o);
      mx_quantities<1>(o, cq);
      mx_denominator<1>(o, o + 27);
    } else {
      mx_normalise<0>(models + 9 * m, s, sc.on, o);
      mx_quantities<0>(o, cq);
      mx_denominator<0>(o, o + 27);
    }
    for (int k = 0; k < 18; ++k) o[9 + k] = cq[k / 9][k % 9];
  }
}

// out per point: 9 terms z, 11 squared terms, the slack
void mx_points(int64_t count, const double* pts, double s, double sq_thr, double* out) {
  const MxScale sc = mx_scale(sq_thr, 1.0 / s);
  for (int64_t i = 0; i < count; ++i) {
    const double x1 = pts[4 * i] / s, y1 = pts[4 * i + 1] / s, x2 = pts[4 * i + 2] / s, y2 = pts[4 * i + 3] / s;
    double* o = out + 21 * i;
    mx_terms(x1, y1, x2, y2, o, o + 9);
    o[20] = mx_slack(sc, x1, y1, x2, y2);
  }
}

// on, sigma, kappa
void mx_scales(double s, double sq_thr, double* out) {
  const MxScale sc = mx_scale(sq_thr, 1.0 / s);
  out[0] = sc.on;
  out[1] = sc.sigma;
  out[2] = sc.kappa;
}
}
