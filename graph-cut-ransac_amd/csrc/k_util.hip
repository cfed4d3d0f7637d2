// Small utility kernels: model-slot copies, range zeroing and IRLS weights.
#include <algorithm>
#include <atomic>

#include "dev_common.hpp"
#include "kernels.hpp"

namespace gcr {

__global__ void k_copy_models(const double* const* __restrict__ src, double* const* __restrict__ dst, int count) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const int c = t / 9, k = t % 9;
  if (c >= count) return;
  dst[c][k] = src[c][k];
}

int lds_limit_bytes() {
  static std::atomic<int> cached[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 64 * 1024;
  int v = cached[dev].load(std::memory_order_relaxed);
  if (v == 0) {
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess || v <= 0)
      v = 64 * 1024;
    cached[dev].store(v, std::memory_order_relaxed);
  }
  return v;
}

void launch_copy_models(hipStream_t st, const double* const* src, double* const* dst, int count) {
  if (count <= 0) return;
  const int th = count * 9;
  hipLaunchKernelGGL(k_copy_models, dim3((th + 255) / 256), dim3(256), 0, st, src, dst, count);
}

// Zeroes the ranges [off[r], off[r] + len[r]) of a; blockIdx.y = range.
__global__ void k_zero_ranges(double* __restrict__ a, const int64_t* __restrict__ off,
                              const int32_t* __restrict__ len) {
  const int r = blockIdx.y;
  const int64_t n = len[r];
  double* const dst = a + off[r];
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (int64_t)gridDim.x * blockDim.x)
    dst[k] = 0.0;
}

void launch_zero_ranges(hipStream_t st, double* a, const int64_t* off, const int32_t* len, int count, int max_len) {
  if (count <= 0 || max_len <= 0) return;
  const dim3 grid((unsigned)std::min(16, (max_len + 255) / 256), (unsigned)count);
  hipLaunchKernelGGL(k_zero_ranges, grid, dim3(256), 0, st, a, off, len);
}

// Tukey bisquare weights of the current inliers, stored by point index
// (GCRANSAC.h:655-667): w = max(0, 1 - r2 / tau2)^2.  zero != 0 resets the
// entries of the listed inliers to 0 instead (GCRANSAC.h:677-679).
template <int KIND>
__global__ void k_irls_weights(const double* __restrict__ pts, const int64_t* __restrict__ pair_pt_off,
                               const double* __restrict__ pair_sq_thr, const int32_t* __restrict__ item_pair,
                               const double* const* __restrict__ item_model, const int32_t* __restrict__ inliers,
                               const int64_t* __restrict__ inl_off, const int32_t* __restrict__ inl_n,
                               double* __restrict__ weights, int zero) {
  const int it = blockIdx.y;
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= inl_n[it]) return;
  const int pair = item_pair[it];
  const int64_t base = pair_pt_off[pair];
  const int idx = inliers[inl_off[it] + k];
  if (zero) {
    weights[base + idx] = 0.0;
    return;
  }
  double M[9];
#pragma unroll
  for (int j = 0; j < 9; ++j) M[j] = item_model[it][j];
  const double r2 = sq_residual<KIND>(pts + 4 * (base + idx), M);
  const double w0 = 1.0 - r2 / pair_sq_thr[pair];
  const double w = 0.0 > w0 ? 0.0 : w0;
  weights[base + idx] = w * w;
}

void launch_irls_weights(hipStream_t st, int kind, const double* pts, const int64_t* pair_pt_off,
                         const double* pair_sq_thr, const int32_t* item_pair, const double* const* item_model,
                         const int32_t* inliers, const int64_t* inl_off, const int32_t* inl_n, double* weights,
                         int num_items, int zero, int max_n) {
  if (num_items <= 0 || max_n <= 0) return;
  const dim3 grid((max_n + 255) / 256, num_items);
  if (kind == 0)
    hipLaunchKernelGGL(k_irls_weights<0>, grid, dim3(256), 0, st, pts, pair_pt_off, pair_sq_thr, item_pair, item_model,
                       inliers, inl_off, inl_n, weights, zero);
  else
    hipLaunchKernelGGL(k_irls_weights<1>, grid, dim3(256), 0, st, pts, pair_pt_off, pair_sq_thr, item_pair, item_model,
                       inliers, inl_off, inl_n, weights, zero);
}

// ---- candidate results filtered on the device --------------------------------
// One thread per candidate (blockIdx.y = item): the last model's count goes to
// last_count[c]; the slots whose value beats the item's best become records,
// appended in any order (the host puts each item's records back in slot
// order; few slots beat a pair's best).  One block per item walking its slots
// in order, 1,024 a round, was a serial chain of up to 160 rounds: 670 us per
// chunk of essential candidates on MI355X.
__global__ void __launch_bounds__(256)
    k_chunk_filter(int h, int S, const int64_t* __restrict__ item_base, const int32_t* __restrict__ item_ncand,
                   const double* __restrict__ item_best, const int8_t* __restrict__ status, int8_t* nmodels,
                   const int32_t* __restrict__ counts, const double* __restrict__ values,
                   const int32_t* __restrict__ sym, const int8_t* __restrict__ valid,
                   const int32_t* __restrict__ samples, int m, int32_t* __restrict__ last_count,
                   SlotRec* __restrict__ recs, uint32_t* __restrict__ rec_count, int first_item) {
  const int it = first_item + (int)blockIdx.y;
  const int q = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  const bool live = q < item_ncand[it];
  const int64_t c = item_base[it] + (live ? q : 0);
  const double best = item_best[it];
  int nm = 0;
  if (live) {
    if (h) {
      nm = status[c] == 2 ? 1 : 0;
      nmodels[c] = (int8_t)nm;
    } else {
      nm = nmodels[c];
    }
    if (nm > 0) last_count[c] = counts[c * S + nm - 1];
  }
  for (int j = 0; ballot64(j < nm) != 0; ++j) {
    const int64_t g = c * S + j;
    const double v = j < nm ? values[g] : 0.0;
    const bool keep = j < nm && v > best;
    const uint64_t b = ballot64(keep);
    if (b == 0) continue;
    uint32_t at = 0;
    if (lane_id() == 0) at = atomicAdd(rec_count, (uint32_t)__popcll(b));
    at = (uint32_t)__builtin_amdgcn_readfirstlane((int)at);
    if (keep) {
      SlotRec r;
      r.slot = q * S + j;
      r.count = counts[g];
      r.value = v;
      r.sym = h ? 0 : sym[g];
      r.valid = h ? valid[c] : 1;
      r.degen = 0;
      r.pad[0] = r.pad[1] = 0;
      r.sample0 = samples[c * m];
      r.item = it;
      recs[at + __popcll(b & ((1ull << lane_id()) - 1ull))] = r;
    }
  }
}

// cand_pair[base[i] + c] = pair[i] for c < count[i] (one block per item); *zero
// = 0 when given
__global__ void __launch_bounds__(256) k_fill_cand_pair(const int64_t* __restrict__ base,
                                                        const int32_t* __restrict__ count,
                                                        const int32_t* __restrict__ pair, int32_t* __restrict__ cand_pair,
                                                        uint32_t* __restrict__ zero) {
  const int it = blockIdx.x;
  if (zero && it == 0 && threadIdx.x == 0) *zero = 0u;
  const int64_t b = base[it];
  const int32_t n = count[it], p = pair[it];
  for (int32_t c = threadIdx.x; c < n; c += 256) cand_pair[b + c] = p;
}

void launch_fill_cand_pair(hipStream_t st, int num_items, const int64_t* base, const int32_t* count,
                           const int32_t* pair, int32_t* cand_pair, uint32_t* zero) {
  if (num_items <= 0) return;
  hipLaunchKernelGGL(k_fill_cand_pair, dim3(num_items), dim3(256), 0, st, base, count, pair, cand_pair, zero);
}

void launch_chunk_filter(hipStream_t st, int h, int S, int num_items, int max_cand, const int64_t* item_base,
                         const int32_t* item_ncand, const double* item_best, const int8_t* status, int8_t* nmodels,
                         const int32_t* counts, const double* values, const int32_t* sym, const int8_t* valid,
                         const int32_t* samples, int m, int32_t* last_count, SlotRec* recs, uint32_t* rec_count) {
  if (num_items <= 0 || max_cand <= 0) return;
  // blockIdx.y holds at most 65,535 items
  for (int i = 0; i < num_items; i += 65535) {
    const int k = std::min(65535, num_items - i);
    hipLaunchKernelGGL(k_chunk_filter, dim3((unsigned)((max_cand + 255) / 256), (unsigned)k), dim3(256), 0, st, h, S,
                       item_base, item_ncand, item_best, status, nmodels, counts, values, sym, valid, samples, m,
                       last_count, recs, rec_count, i);
  }
}

}  // namespace gcr
