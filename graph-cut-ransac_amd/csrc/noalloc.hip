// gcr_score_models_noalloc: MSAC scoring of k models over n points with no
// device allocation.  Inputs and outputs are the caller's device buffers, the
// call is one kernel launch (which can be recorded into a HIP graph) and uses no
// other device memory.
#include <hip/hip_runtime.h>

#include <string>

#include "engine.hpp"
#include "kernels.hpp"

namespace {
constexpr int64_t kMaxModels = GCR_SCORE_NOALLOC_MAX_MODELS;
}

extern "C" int32_t gcr_score_models_noalloc(int32_t kind, const double* pts, int64_t n, const double* models,
                                            int64_t k, double sq_thr, int64_t* counts, double* values,
                                            uint8_t* masks, void* stream) {
  if (!pts || !models || !counts || !values) {
    gcr::set_last_error("null pointer argument");
    return GCR_ERR_INVALID_ARGUMENT;
  }
  if (kind != 0 && kind != 1) {
    gcr::set_last_error("kind must be 0 (homography) or 1 (Sampson)");
    return GCR_ERR_INVALID_ARGUMENT;
  }
  if (n <= 0 || n > (int64_t)INT32_MAX) {
    gcr::set_last_error("n must be in [1, 2^31 - 1]");
    return GCR_ERR_INVALID_ARGUMENT;
  }
  if (k <= 0 || k > kMaxModels) {
    gcr::set_last_error("k must be in [1, " + std::to_string(kMaxModels) + "]");
    return GCR_ERR_INVALID_ARGUMENT;
  }
  if (masks && k > INT64_MAX / n) {
    gcr::set_last_error("k * n overflows");
    return GCR_ERR_INVALID_ARGUMENT;
  }
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0) {
    gcr::set_last_error("no current HIP device");
    return GCR_ERR_DEVICE;
  }
  gcr::launch_score_direct(static_cast<hipStream_t>(stream), kind, pts, (int)n, sq_thr, models, k, counts, values,
                           masks);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    gcr::set_last_error(std::string("scoring launch: ") + hipGetErrorString(e));
    return GCR_ERR_DEVICE;
  }
  return GCR_OK;
}
