// Matrix-core scoring: the model's side of the rejection test (k_score_mx.hip).
// Plain functions of numbers, for the kernels and for host code.
#pragma once

#include <cmath>

#if defined(__HIP__)
#define GCR_MX_FN __host__ __device__ __forceinline__
#else
#define GCR_MX_FN inline
#endif

namespace gcr {

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
