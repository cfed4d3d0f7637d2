// Device kernels of the learned inlier-probability network.
//
// There is no reference counterpart: the reference's hook for a learned
// quality score is the PROSAC sampler, which draws from prefixes of the
// points sorted by quality (inc/samplers/prosac_sampler.h:51-237).  These
// kernels compute that score per correspondence:
//   k_knn_bin, k_knn_scatter, k_knn_query
//                    8-nearest-neighbour features (per-pair grid of cells,
//                    one thread per query walking rings of cells)
//   k_mlp_predict    forward pass on the matrix cores
//   k_mlp_train      forward, backward and weight-gradient pass of one
//                    mini-batch, a partial gradient per workgroup
//   k_mlp_reduce     deterministic sum of the partials, Adam and the packed
//                    weights of the next step
//
// Matrix-core formulation.  Activations are kept transposed: a wave owns 32
// points (the N = 32 columns of a 32x32x8 BF16 MFMA) and computes
// Z^T = W H^T, with W in the A operand (32 output neurons x 8 inputs per
// instruction) and H^T in B.  The 16 FP32 results a lane holds for one
// 32-neuron tile are the neurons 8*(r/4) + 4*(lane/32) + r%4 of point
// lane%32 -- exactly the B-operand slots of the next layer's k-blocks, so a
// layer's output (bias, GELU, BF16 rounding applied in registers) feeds the
// next layer with no data movement.  Weights live in LDS with a 132-element
// row stride (no bank conflicts on the 8-byte A-operand reads).
//
// Training has a few thousand points per step, too few for a wave per 32
// points to fill the chip, so there the four waves of a workgroup share 32
// points and own 32 neurons of every layer each (k_mlp_train).
#include <hip/hip_runtime.h>

#include "mlp_kernels.hpp"

namespace gcr {
namespace mlp {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

namespace {

constexpr int RS = 132;  // LDS row stride (elements) of the 128-wide matrices

struct FwdLds {
  uint16_t w1[HID * IN];
  uint16_t w2[HID * RS];
  uint16_t w3[HID * RS];
  float b1[HID], b2[HID], b3[HID], w4[HID];
  float b4, pad_[3];
};
static_assert(sizeof(FwdLds) % 16 == 0, "LDS layout");

// Training: activations and deltas of a workgroup's 32 points, BF16.
// Point-major rows (the next layer's B operand, 8 neurons per read) and
// neuron-major rows (the weight gradient's operands, 8 points per read); row
// strides of 17 and 5 16-byte units keep both free of bank conflicts.
constexpr int PS = 136, NS = 40;
struct TrainLds {
  uint16_t h1p[32][PS], h2p[32][PS], d3p[32][PS], d2p[32][PS];
  uint16_t x[16][NS];  // input rows 0 .. 7, row 8: ones (the bias gradient)
  uint16_t h1[HID][NS], h2[HID][NS];
  uint16_t d1[HID][NS], d2[HID][NS], d3[HID][NS];
  float z4[4][32];     // the waves' parts of the logits
  float b1[HID], b2[HID], b3[HID], w4[HID];
};
static_assert(sizeof(TrainLds) % 16 == 0, "LDS layout");

__device__ inline uint16_t f2bf(float f) {
  uint32_t u = __float_as_uint(f);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
__device__ inline float bf2f(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }

// GELU (tanh form), operations in the oracle's order
__device__ inline float gelu_f(float z) {
  const float c = 0.7978845608028654f;
  const float u = c * (z + 0.044715f * (z * z * z));
  return 0.5f * z * (1.0f + tanhf(u));
}
// GELU and its derivative from one tanh
__device__ inline float gelu_both(float z, float& grad) {
  const float c = 0.7978845608028654f;
  const float z2 = z * z;
  const float t = tanhf(c * (z + 0.044715f * (z2 * z)));
  grad = 0.5f * (1.0f + t) + 0.5f * z * ((1.0f - t * t) * (c * (1.0f + 0.134145f * z2)));
  return 0.5f * z * (1.0f + t);
}
__device__ inline float sigmoid_f(float z) { return 1.0f / (1.0f + expf(-z)); }
__device__ inline float softplus_f(float z) {
  const float a = z < 0.0f ? -z : z;
  return (z > 0.0f ? z : 0.0f) + log1pf(expf(-a));
}

__device__ inline uint64_t mix64(uint64_t x) {
  x += 0x9E3779B97F4A7C15ull;
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  return x ^ (x >> 31);
}

__device__ inline f32x16 zero16() {
  f32x16 z;
#pragma unroll
  for (int r = 0; r < 16; ++r) z[r] = 0.0f;
  return z;
}

__device__ inline f32x16 mfma(const bf16x4& a, const bf16x4& b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(a, b, c, 0, 0, 0);
}
// 16 values of the reduction dimension: lane l holds 8 (l / 32) .. + 7 of row /
// column l % 32
__device__ inline f32x16 mfma16(const bf16x8& a, const bf16x8& b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
__device__ inline bf16x8 load8(const uint16_t* p) { return *reinterpret_cast<const bf16x8*>(p); }
__device__ inline bf16x8 fill8(uint16_t v) {
  union {
    uint16_t u[8];
    bf16x8 b;
  } x;
#pragma unroll
  for (int e = 0; e < 8; ++e) x.u[e] = v;
  return x.b;
}

// 128 x 128 BF16 matrix (row-major) -> LDS rows of RS elements
__device__ inline void stage_matrix(uint16_t* dst, const uint16_t* src) {
  for (int e = threadIdx.x; e < HID * (HID / 4); e += blockDim.x) {
    const int r = e >> 5, c4 = e & 31;
    *reinterpret_cast<uint2*>(dst + r * RS + c4 * 4) = *reinterpret_cast<const uint2*>(src + r * HID + c4 * 4);
  }
}

__device__ inline void stage_forward(FwdLds& s, const uint16_t* wpk, const float* bias) {
  for (int e = threadIdx.x; e < HID * IN / 4; e += blockDim.x)
    *reinterpret_cast<uint2*>(s.w1 + 4 * e) = *reinterpret_cast<const uint2*>(wpk + PK_W1 + 4 * e);
  stage_matrix(s.w2, wpk + PK_W2);
  stage_matrix(s.w3, wpk + PK_W3);
  for (int i = threadIdx.x; i < HID; i += blockDim.x) {
    s.b1[i] = bias[i];
    s.b2[i] = bias[HID + i];
    s.b3[i] = bias[2 * HID + i];
    s.w4[i] = bf2f(wpk[PK_W4 + i]);
  }
  if (threadIdx.x == 0) s.b4 = bias[3 * HID];
}

// bias + GELU + BF16 of one 32-neuron tile; the rounded activations go to
// the next layer's B operand (k-blocks 4*MT .. 4*MT+3)
template <int MT>
__device__ __attribute__((always_inline)) inline void epilogue(const f32x16& acc, const float* bias, int half,
                                                               bf16x4* hout) {
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int i = 32 * MT + 8 * (r >> 2) + 4 * half + (r & 3);
    const float z = acc[r] + bias[i];
    hout[4 * MT + (r >> 2)][r & 3] = (short)f2bf(gelu_f(z));
  }
}

template <int MT>
__device__ __attribute__((always_inline)) inline void hidden_tile(const uint16_t* w, const float* bias,
                                                                  const bf16x4* hin, int j, int half, bf16x4* hout) {
  f32x16 acc = zero16();
  const uint16_t* wrow = w + (32 * MT + j) * RS + 4 * half;
#pragma unroll
  for (int kb = 0; kb < 16; ++kb) {
    const bf16x4 a = *reinterpret_cast<const bf16x4*>(wrow + 8 * kb);
    acc = mfma(a, hin[kb], acc);
  }
  epilogue<MT>(acc, bias, half, hout);
}

// Forward pass of the wave's 32 points (lane % 32 = point, lane / 32 = half
// of the k-block); returns the logit (both halves hold it).  fptr: this
// lane's feature row, nullptr for a padding column.
// wj: lane % 32 as the weight-row index; the persistent inference loop
// passes it through an empty asm so the weight reads stay inside the loop
// (hoisted, the 128 weight registers per layer would spill).
__device__ __attribute__((always_inline)) inline float forward_wave(const FwdLds& s, const float* fptr, int lane,
                                                                    int wj) {
  const int j = wj, half = lane >> 5;
  float4 f = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  if (fptr) f = *reinterpret_cast<const float4*>(fptr + 4 * half);
  bf16x4 xb;
  xb[0] = (short)f2bf(f.x);
  xb[1] = (short)f2bf(f.y);
  xb[2] = (short)f2bf(f.z);
  xb[3] = (short)f2bf(f.w);
  bf16x4 ha[16], hb[16];
  // layer 1: one k-block (8 inputs)
  {
    const uint16_t* wrow = s.w1 + j * IN + 4 * half;
    f32x16 acc0 = mfma(*reinterpret_cast<const bf16x4*>(wrow), xb, zero16());
    epilogue<0>(acc0, s.b1, half, ha);
    f32x16 acc1 = mfma(*reinterpret_cast<const bf16x4*>(wrow + 32 * IN), xb, zero16());
    epilogue<1>(acc1, s.b1, half, ha);
    f32x16 acc2 = mfma(*reinterpret_cast<const bf16x4*>(wrow + 64 * IN), xb, zero16());
    epilogue<2>(acc2, s.b1, half, ha);
    f32x16 acc3 = mfma(*reinterpret_cast<const bf16x4*>(wrow + 96 * IN), xb, zero16());
    epilogue<3>(acc3, s.b1, half, ha);
  }
  hidden_tile<0>(s.w2, s.b2, ha, j, half, hb);
  hidden_tile<1>(s.w2, s.b2, ha, j, half, hb);
  hidden_tile<2>(s.w2, s.b2, ha, j, half, hb);
  hidden_tile<3>(s.w2, s.b2, ha, j, half, hb);
  hidden_tile<0>(s.w3, s.b3, hb, j, half, ha);
  hidden_tile<1>(s.w3, s.b3, hb, j, half, ha);
  hidden_tile<2>(s.w3, s.b3, hb, j, half, ha);
  hidden_tile<3>(s.w3, s.b3, hb, j, half, ha);
  // output unit: this half's 64 neurons in ascending order, then the halves
  float sum = 0.0f;
#pragma unroll
  for (int kb = 0; kb < 16; ++kb) {
#pragma unroll
    for (int e = 0; e < 4; ++e) sum = sum + s.w4[8 * kb + 4 * half + e] * bf2f((uint16_t)ha[kb][e]);
  }
  const float other = __shfl_xor(sum, 32);
  return (half == 0 ? sum + other : other + sum) + s.b4;
}

}  // namespace

int lds_forward_bytes() { return (int)sizeof(FwdLds); }
int lds_train_bytes() { return (int)sizeof(TrainLds); }

// ---- features --------------------------------------------------------------
//
// Per correspondence: normalised coordinates, the descriptor ratio and the
// mean displacement (x2 - x1, y2 - y1) of its 8 nearest first-image
// neighbours minus its own, as the oracle's index-order scan defines them.
// The neighbour search is restricted by a grid: a pair's
// first-image points are binned into square cells (about four points per
// cell, indices clamped to the grid), sorted by cell, and each query walks
// rings of cells around its own cell until its eighth-best distance is below
// a lower bound of the distance of every point outside the rings.  Candidates
// are ranked by (distance, index): the index-order scan keeps, among
// equal distances, the earlier index, so both build the same ordered list of
// the 8 smallest (distance, index) pairs and the same sums.
//
// Lower bound: a point in a cell of column index below c has
// fl(x * inv_cs) < c, so x < c / inv_cs up to one rounding of the product;
// one in a column above c has x >= (c + 1) / inv_cs likewise (clamping moves
// a point only into the edge cell on its own side, which keeps both
// inequalities).  The bound is reduced by a margin far above those roundings
// and the float rounding of the distance, and the search stops only when the
// eighth distance is strictly below it, so no point outside the rings can
// enter the list.

__device__ __forceinline__ int knn_axis_cell(float v, float inv_cs, int g) {
  const float f = floorf(v * inv_cs);
  if (!(f >= 0.0f)) return 0;  // negative or NaN
  if (f >= (float)g) return g - 1;
  return (int)f;
}

__global__ __launch_bounds__(256) void k_knn_bin(const double* __restrict__ corr, const int64_t* __restrict__ pair_off,
                                                 const KnnGrid* __restrict__ grids,
                                                 const int32_t* __restrict__ tile_pair,
                                                 const int32_t* __restrict__ tile_start, int32_t* __restrict__ cell_count,
                                                 int32_t* __restrict__ cell_of, int32_t* __restrict__ rank) {
  const int p = tile_pair[blockIdx.x];
  const int64_t base = pair_off[p];
  const int64_t n = pair_off[p + 1] - base;
  const int64_t q = (int64_t)tile_start[blockIdx.x] + threadIdx.x;
  if (q >= n) return;
  const KnnGrid g = grids[p];
  const double* r = corr + 4 * (base + q);
  const float x = (float)r[0], y = (float)r[1];
  const int c = knn_axis_cell(y, g.inv_cs, g.gy) * g.gx + knn_axis_cell(x, g.inv_cs, g.gx);
  cell_of[base + q] = c;
  rank[base + q] = atomicAdd(cell_count + g.cell_base + c, 1);
}

__global__ __launch_bounds__(256) void k_knn_scatter(const double* __restrict__ corr,
                                                     const int64_t* __restrict__ pair_off,
                                                     const KnnGrid* __restrict__ grids,
                                                     const int32_t* __restrict__ tile_pair,
                                                     const int32_t* __restrict__ tile_start,
                                                     const int32_t* __restrict__ cell_off,
                                                     const int32_t* __restrict__ cell_of,
                                                     const int32_t* __restrict__ rank, float4* __restrict__ spts,
                                                     int32_t* __restrict__ sidx) {
  const int p = tile_pair[blockIdx.x];
  const int64_t base = pair_off[p];
  const int64_t n = pair_off[p + 1] - base;
  const int64_t q = (int64_t)tile_start[blockIdx.x] + threadIdx.x;
  if (q >= n) return;
  const KnnGrid g = grids[p];
  const double* r = corr + 4 * (base + q);
  const float x = (float)r[0], y = (float)r[1];
  const int64_t pos = (int64_t)cell_off[g.cell_base + cell_of[base + q]] + rank[base + q];
  spts[pos] = make_float4(x, y, (float)r[2] - x, (float)r[3] - y);
  sidx[pos] = (int32_t)q;
}

// one thread per sorted position (neighbouring threads query neighbouring
// cells); writes the features of the point at that position
__global__ __launch_bounds__(256) void k_knn_query(const double* __restrict__ corr,
                                                   const int64_t* __restrict__ pair_off,
                                                   const int32_t* __restrict__ sizes, const double* __restrict__ ratio,
                                                   const KnnGrid* __restrict__ grids,
                                                   const int32_t* __restrict__ tile_pair,
                                                   const int32_t* __restrict__ tile_start,
                                                   const int32_t* __restrict__ cell_off,
                                                   const float4* __restrict__ spts, const int32_t* __restrict__ sidx,
                                                   float* __restrict__ feat) {
  const int p = tile_pair[blockIdx.x];
  const int64_t base = pair_off[p];
  const int64_t n = pair_off[p + 1] - base;
  const int64_t sp = (int64_t)tile_start[blockIdx.x] + threadIdx.x;
  if (sp >= n) return;
  const KnnGrid g = grids[p];
  const float4 me = spts[base + sp];
  const int32_t q = sidx[base + sp];
  const float xq = me.x, yq = me.y, uxq = me.z, uyq = me.w;
  const int cx = knn_axis_cell(xq, g.inv_cs, g.gx), cy = knn_axis_cell(yq, g.inv_cs, g.gy);
  const double cs = 1.0 / (double)g.inv_cs;
  const double margin = 1e-5 * (fabs((double)xq) + fabs((double)yq) + cs * (double)(g.gx + g.gy + 2)) + 1e-3;
  const int32_t* coff = cell_off + g.cell_base;
  float td[8], tx[8], ty[8];
  int32_t ti[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    td[k] = INFINITY;
    ti[k] = -1;
    tx[k] = 0.0f;
    ty[k] = 0.0f;
  }
  auto visit = [&](int cell) {
    const int32_t b0 = coff[cell], b1 = coff[cell + 1];
    for (int32_t s = b0; s < b1; ++s) {
      const float4 cj = spts[s];
      const int32_t j = sidx[s];
      const float dx = xq - cj.x, dy = yq - cj.y;
      const float d = dx * dx + dy * dy;
      if (j == q || !(d < td[7] || (d == td[7] && j < ti[7]))) continue;
#pragma unroll
      for (int k = 7; k > 0; --k) {
        if (d < td[k - 1] || (d == td[k - 1] && j < ti[k - 1])) {
          td[k] = td[k - 1];
          ti[k] = ti[k - 1];
          tx[k] = tx[k - 1];
          ty[k] = ty[k - 1];
        } else if (d < td[k] || (d == td[k] && j < ti[k])) {
          td[k] = d;
          ti[k] = j;
          tx[k] = cj.z;
          ty[k] = cj.w;
        }
      }
      if (d < td[0] || (d == td[0] && j < ti[0])) {
        td[0] = d;
        ti[0] = j;
        tx[0] = cj.z;
        ty[0] = cj.w;
      }
    }
  };
  const int rmax = g.gx > g.gy ? g.gx : g.gy;
  for (int R = 0; R <= rmax; ++R) {
    const int i0 = cx - R, i1 = cx + R, j0 = cy - R, j1 = cy + R;
    for (int j = j0 < 0 ? 0 : j0; j <= (j1 < g.gy ? j1 : g.gy - 1); ++j) {
      if (j == j0 || j == j1) {
        for (int i = i0 < 0 ? 0 : i0; i <= (i1 < g.gx ? i1 : g.gx - 1); ++i) visit(j * g.gx + i);
      } else {
        if (i0 >= 0) visit(j * g.gx + i0);
        if (i1 < g.gx && i1 != i0) visit(j * g.gx + i1);
      }
    }
    // lower bound of the distance of every point outside rings 0..R
    const bool lo_x = i0 > 0, hi_x = i1 < g.gx - 1, lo_y = j0 > 0, hi_y = j1 < g.gy - 1;
    if (!(lo_x || hi_x || lo_y || hi_y)) break;  // every cell visited
    double b = INFINITY;
    if (lo_x) b = fmin(b, (double)xq - (double)i0 * cs);
    if (hi_x) b = fmin(b, (double)(i1 + 1) * cs - (double)xq);
    if (lo_y) b = fmin(b, (double)yq - (double)j0 * cs);
    if (hi_y) b = fmin(b, (double)(j1 + 1) * cs - (double)yq);
    b -= margin;
    if (b > 0.0 && (double)td[7] < b * b * (1.0 - 1e-5)) break;
  }
  float sx = 0.0f, sy = 0.0f;
  int c = 0;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    if (ti[k] >= 0) {
      sx = sx + tx[k];
      sy = sy + ty[k];
      ++c;
    }
  }
  const int h1 = sizes[4 * p + 0], w1 = sizes[4 * p + 1], h2 = sizes[4 * p + 2], w2 = sizes[4 * p + 3];
  const float s1x = 2.0f / (float)w1, s1y = 2.0f / (float)h1, s2x = 2.0f / (float)w2, s2y = 2.0f / (float)h2;
  const float sd = 2.0f / (float)(w1 > h1 ? w1 : h1);
  float f5 = 0.0f, f6 = 0.0f;
  if (c > 0) {
    const float fc = (float)c;
    f5 = (sx / fc - uxq) * sd;
    f6 = (sy / fc - uyq) * sd;
  }
  const double* r = corr + 4 * (base + q);
  const float x2q = (float)r[2], y2q = (float)r[3];
  float4* out = reinterpret_cast<float4*>(feat + IN * (base + q));
  out[0] = make_float4(xq * s1x - 1.0f, yq * s1y - 1.0f, x2q * s2x - 1.0f, y2q * s2y - 1.0f);
  out[1] = make_float4((float)ratio[base + q], f5, f6, 0.0f);
}

void launch_knn_bin(hipStream_t st, const double* corr, const int64_t* pair_off, const KnnGrid* grids,
                    const int32_t* tile_pair, const int32_t* tile_start, int tiles, int32_t* cell_count,
                    int32_t* cell_of, int32_t* rank) {
  if (tiles <= 0) return;
  hipLaunchKernelGGL(k_knn_bin, dim3(tiles), dim3(256), 0, st, corr, pair_off, grids, tile_pair, tile_start,
                     cell_count, cell_of, rank);
}

void launch_knn_scatter(hipStream_t st, const double* corr, const int64_t* pair_off, const KnnGrid* grids,
                        const int32_t* tile_pair, const int32_t* tile_start, int tiles, const int32_t* cell_off,
                        const int32_t* cell_of, const int32_t* rank, float4* spts, int32_t* sidx) {
  if (tiles <= 0) return;
  hipLaunchKernelGGL(k_knn_scatter, dim3(tiles), dim3(256), 0, st, corr, pair_off, grids, tile_pair, tile_start,
                     cell_off, cell_of, rank, spts, sidx);
}

void launch_knn_query(hipStream_t st, const double* corr, const int64_t* pair_off, const int32_t* sizes,
                      const double* ratio, const KnnGrid* grids, const int32_t* tile_pair, const int32_t* tile_start,
                      int tiles, const int32_t* cell_off, const float4* spts, const int32_t* sidx, float* feat) {
  if (tiles <= 0) return;
  hipLaunchKernelGGL(k_knn_query, dim3(tiles), dim3(256), 0, st, corr, pair_off, sizes, ratio, grids, tile_pair,
                     tile_start, cell_off, spts, sidx, feat);
}


// ---- packing, forward, training -------------------------------------------

__global__ __launch_bounds__(256) void k_mlp_pack(const float* __restrict__ p, uint16_t* __restrict__ wpk,
                                                  float* __restrict__ bias) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < HID * HID) {
    const int r = t / HID, c = t % HID;
    const uint16_t a = f2bf(p[OFF_W2 + t]), b = f2bf(p[OFF_W3 + t]);
    wpk[PK_W2 + t] = a;
    wpk[PK_W2T + c * HID + r] = a;
    wpk[PK_W3 + t] = b;
    wpk[PK_W3T + c * HID + r] = b;
  }
  if (t < HID * IN) wpk[PK_W1 + t] = f2bf(p[OFF_W1 + t]);
  if (t < HID) {
    wpk[PK_W4 + t] = f2bf(p[OFF_W4 + t]);
    bias[t] = p[OFF_B1 + t];
    bias[HID + t] = p[OFF_B2 + t];
    bias[2 * HID + t] = p[OFF_B3 + t];
  }
  if (t == 0) bias[3 * HID] = p[OFF_B4];
}

__global__ __launch_bounds__(256) void k_mlp_predict(const uint16_t* __restrict__ wpk, const float* __restrict__ bias,
                                                     const float* __restrict__ feat, int64_t n,
                                                     float* __restrict__ logit, float* __restrict__ prob) {
  extern __shared__ __align__(16) unsigned char mlp_lds_f[];
  FwdLds& s = *reinterpret_cast<FwdLds*>(mlp_lds_f);
  stage_forward(s, wpk, bias);
  __syncthreads();
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  for (int64_t b0 = (int64_t)blockIdx.x * POINTS_PER_BLOCK; b0 < n; b0 += (int64_t)gridDim.x * POINTS_PER_BLOCK) {
    const int64_t col = b0 + 32 * w + (lane & 31);
    const bool valid = col < n;
    int wj = lane & 31;
    asm volatile("" : "+v"(wj));
    const float z = forward_wave(s, valid ? feat + IN * col : nullptr, lane, wj);
    if ((lane >> 5) == 0 && valid) {
      logit[col] = z;
      if (prob) prob[col] = sigmoid_f(z);
    }
  }
}

// One mini-batch: forward, backward and weight gradients.  A workgroup takes
// tiles of 32 points; wave w owns neurons 32 w .. 32 w + 31 of every hidden
// layer: its rows of W2, W3 and of their transposes are the A operands, the
// layers' outputs pass between the waves through LDS, and
// the tile's deltas and activations are contracted into the workgroup's
// gradient accumulators (the points are the reduction dimension; the bias
// gradients are one more column of ones).  One partial gradient per workgroup
// goes to memory.
//
// What bounds it: the latency of one tile's chain of nine dependent layer
// products and their tanh epilogues, with one wave per SIMD.  A wave per 32
// points for all 128 neurons, the activations written to memory for a second
// kernel of 16 workgroups, took 135 + 115 us per step of 8,192 rows on MI355X;
// this kernel 31.8 us (128 workgroups of two tiles 55 us, with 5.9 us in the
// reduction against 9.2).
__global__ __launch_bounds__(256, 1) void k_mlp_train(const uint16_t* __restrict__ wpk, const float* __restrict__ bias,
                                                      const float* __restrict__ feat,
                                                      const float* __restrict__ labels, int64_t batch,
                                                      int64_t sample_n, uint64_t seed, int64_t step, float inv_batch,
                                                      float* __restrict__ part) {
  extern __shared__ __align__(16) unsigned char mlp_lds_t[];
  TrainLds& s = *reinterpret_cast<TrainLds*>(mlp_lds_t);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, j = lane & 31, half = lane >> 5;
  // this wave's neuron of accumulator slot r
  auto neuron = [&](int r) { return 32 * w + 8 * (r >> 2) + 4 * half + (r & 3); };
  // A operand of this wave's rows of a 128 x 128 matrix, fetched (from the L2)
  // a layer ahead of its use; the empty asm keeps the fetch inside the tile
  // loop (all four matrices held over it, 128 registers, spilled)
  auto fetch = [&](bf16x8* A, int matrix) {
    int at = matrix + (32 * w + j) * HID + 8 * half;
    asm volatile("" : "+v"(at));
#pragma unroll
    for (int kb = 0; kb < 8; ++kb) A[kb] = load8(wpk + at + 16 * kb);
  };
  for (int i = threadIdx.x; i < HID; i += 256) {
    s.b1[i] = bias[i];
    s.b2[i] = bias[HID + i];
    s.b3[i] = bias[2 * HID + i];
    s.w4[i] = bf2f(wpk[PK_W4 + i]);
  }
  const float b4 = bias[3 * HID];
  for (int e = threadIdx.x; e < 16 * NS; e += 256) s.x[e / NS][e % NS] = e / NS == 8 ? (uint16_t)0x3F80 : (uint16_t)0;
  f32x16 g1 = zero16(), gb2 = zero16(), gb3 = zero16();
  f32x16 g2[4] = {zero16(), zero16(), zero16(), zero16()}, g3[4] = {zero16(), zero16(), zero16(), zero16()};
  float gw4[16], gb4 = 0.0f, loss = 0.0f;
#pragma unroll
  for (int r = 0; r < 16; ++r) gw4[r] = 0.0f;
  const bf16x8 ones = fill8(j == 0 ? (uint16_t)0x3F80 : (uint16_t)0);
  // four neurons of a point at a time, and one by one neuron-major
  auto put = [&](uint16_t (*pm)[PS], uint16_t (*nm)[NS], const uint16_t* v) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      if (pm) {
        uint2 q;
        q.x = (uint32_t)v[4 * g] | ((uint32_t)v[4 * g + 1] << 16);
        q.y = (uint32_t)v[4 * g + 2] | ((uint32_t)v[4 * g + 3] << 16);
        *reinterpret_cast<uint2*>(&pm[j][32 * w + 8 * g + 4 * half]) = q;
      }
      if (nm) {
#pragma unroll
        for (int e = 0; e < 4; ++e) nm[neuron(4 * g + e)][j] = v[4 * g + e];
      }
    }
  };
  auto layer = [&](const bf16x8* A, uint16_t (*in)[PS]) {
    f32x16 acc = zero16();
#pragma unroll
    for (int kb = 0; kb < 8; ++kb) acc = mfma16(A[kb], load8(&in[j][16 * kb + 8 * half]), acc);
    return acc;
  };
  const int64_t tiles = (batch + 31) / 32;
  for (int64_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
    const int64_t col = 32 * tile + j;
    const bool valid = col < batch;
    int64_t idx = col;
    if (valid && sample_n > 0)
      idx = (int64_t)(mix64(seed ^ mix64((uint64_t)step * 0x100000001B3ull + (uint64_t)col)) % (uint64_t)sample_n);
    const float y = valid ? labels[idx] : 0.0f;
    float gr1[16], gr2[16], gr3[16], h3[16];
    uint16_t v[16];
    bf16x8 A1 = fill8(0), Aa[8], Ab[8];
    if (half == 0) A1 = load8(wpk + PK_W1 + (32 * w + j) * IN);
    fetch(Aa, PK_W2);
    __syncthreads();  // the last tile's operands have been read
    {
      union {
        uint16_t u[8];
        bf16x8 b;
      } x;
#pragma unroll
      for (int e = 0; e < 8; ++e) x.u[e] = 0;
      if (half == 0 && valid) {
        const float4 f0 = *reinterpret_cast<const float4*>(feat + IN * idx);
        const float4 f1 = *reinterpret_cast<const float4*>(feat + IN * idx + 4);
        x.u[0] = f2bf(f0.x);
        x.u[1] = f2bf(f0.y);
        x.u[2] = f2bf(f0.z);
        x.u[3] = f2bf(f0.w);
        x.u[4] = f2bf(f1.x);
        x.u[5] = f2bf(f1.y);
        x.u[6] = f2bf(f1.z);
        x.u[7] = f2bf(f1.w);
      }
      if (w == 0 && half == 0) {
#pragma unroll
        for (int e = 0; e < 8; ++e) s.x[e][j] = x.u[e];
      }
      const f32x16 acc = mfma16(A1, x.b, zero16());
#pragma unroll
      for (int r = 0; r < 16; ++r) v[r] = f2bf(gelu_both(acc[r] + s.b1[neuron(r)], gr1[r]));
    }
    put(s.h1p, s.h1, v);
    __syncthreads();
    {
      fetch(Ab, PK_W3);
      const f32x16 acc = layer(Aa, s.h1p);
#pragma unroll
      for (int r = 0; r < 16; ++r) v[r] = f2bf(gelu_both(acc[r] + s.b2[neuron(r)], gr2[r]));
    }
    put(s.h2p, s.h2, v);
    __syncthreads();
    {
      fetch(Aa, PK_W3T);
      const f32x16 acc = layer(Ab, s.h2p);
      float sum = 0.0f;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        h3[r] = bf2f(f2bf(gelu_both(acc[r] + s.b3[neuron(r)], gr3[r])));
        sum = sum + s.w4[neuron(r)] * h3[r];
      }
      const float other = __shfl_xor(sum, 32);
      if (half == 0) s.z4[w][j] = sum + other;
    }
    __syncthreads();
    const float z4 = ((s.z4[0][j] + s.z4[1][j]) + (s.z4[2][j] + s.z4[3][j])) + b4;
    const float d4 = valid ? (sigmoid_f(z4) - y) * inv_batch : 0.0f;
    if (w == 0 && half == 0 && valid) {
      gb4 += d4;
      loss += (softplus_f(z4) - y * z4) * inv_batch;
    }
    // D3 = w4 d4 * gelu'(Z3)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      gw4[r] += d4 * h3[r];
      v[r] = f2bf((s.w4[neuron(r)] * d4) * gr3[r]);
    }
    put(s.d3p, s.d3, v);
    __syncthreads();
    {
      fetch(Ab, PK_W2T);
      const f32x16 acc = layer(Aa, s.d3p);
#pragma unroll
      for (int r = 0; r < 16; ++r) v[r] = f2bf(acc[r] * gr2[r]);
    }
    put(s.d2p, s.d2, v);
    __syncthreads();
    {
      const f32x16 acc = layer(Ab, s.d2p);
#pragma unroll
      for (int r = 0; r < 16; ++r) v[r] = f2bf(acc[r] * gr1[r]);
    }
    put(nullptr, s.d1, v);
    __syncthreads();
    // G = D H^T over the tile's 32 points
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      const int at = 16 * kb + 8 * half;
      const bf16x8 a3 = load8(&s.d3[32 * w + j][at]), a2 = load8(&s.d2[32 * w + j][at]);
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) {
        g3[nt] = mfma16(a3, load8(&s.h2[32 * nt + j][at]), g3[nt]);
        g2[nt] = mfma16(a2, load8(&s.h1[32 * nt + j][at]), g2[nt]);
      }
      gb3 = mfma16(a3, ones, gb3);
      gb2 = mfma16(a2, ones, gb2);
      const bf16x8 xb = j < 16 ? load8(&s.x[j & 15][at]) : fill8(0);
      g1 = mfma16(load8(&s.d1[32 * w + j][at]), xb, g1);
    }
  }
  float* out = part + (int64_t)blockIdx.x * PART_STRIDE;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int k = neuron(r);
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {
      out[OFF_W3 + k * HID + 32 * nt + j] = g3[nt][r];
      out[OFF_W2 + k * HID + 32 * nt + j] = g2[nt][r];
    }
    if (j < IN) out[OFF_W1 + k * IN + j] = g1[r];
    if (j == IN) out[OFF_B1 + k] = g1[r];
    if (j == 0) {
      out[OFF_B2 + k] = gb2[r];
      out[OFF_B3 + k] = gb3[r];
    }
    float q = gw4[r];
#pragma unroll
    for (int d = 16; d >= 1; d >>= 1) q += __shfl_xor(q, d);
    if (j == 0) out[OFF_W4 + k] = q;
  }
  if (w == 0) {
#pragma unroll
    for (int d = 16; d >= 1; d >>= 1) {
      gb4 += __shfl_xor(gb4, d);
      loss += __shfl_xor(loss, d);
    }
    if (lane == 0) {
      out[OFF_B4] = gb4;
      out[NPARAM] = loss;
    }
  }
}

// Where parameter q goes in the packed weights.
__device__ inline void pack_param(int q, float p, uint16_t* __restrict__ wpk, float* __restrict__ bias) {
  if (q < OFF_B1) {
    wpk[PK_W1 + q] = f2bf(p);
  } else if (q < OFF_W2) {
    bias[q - OFF_B1] = p;
  } else if (q < OFF_B2) {
    const int t = q - OFF_W2;
    const uint16_t b = f2bf(p);
    wpk[PK_W2 + t] = b;
    wpk[PK_W2T + (t % HID) * HID + t / HID] = b;
  } else if (q < OFF_W3) {
    bias[HID + q - OFF_B2] = p;
  } else if (q < OFF_B3) {
    const int t = q - OFF_W3;
    const uint16_t b = f2bf(p);
    wpk[PK_W3 + t] = b;
    wpk[PK_W3T + (t % HID) * HID + t / HID] = b;
  } else if (q < OFF_W4) {
    bias[2 * HID + q - OFF_B3] = p;
  } else if (q < OFF_B4) {
    wpk[PK_W4 + q - OFF_W4] = f2bf(p);
  } else {
    bias[3 * HID] = p;
  }
}

// Four threads per parameter, each summing a quarter of the partials in
// workgroup order (the quarters' sums are added in order); the first applies
// Adam and packs the new weight for the next step.
__global__ __launch_bounds__(256) void k_mlp_reduce(const float* __restrict__ part, int chunks,
                                                    float* __restrict__ grad, float* __restrict__ loss_out, int adam,
                                                    float* __restrict__ params, float* __restrict__ m,
                                                    float* __restrict__ v, float lr, float c1, float c2,
                                                    uint16_t* __restrict__ wpk, float* __restrict__ bias) {
  __shared__ float sums[4][64];
  const int quarter = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int q = blockIdx.x * 64 + lane;
  const int lo = chunks * quarter / 4, hi = chunks * (quarter + 1) / 4;
  float g = 0.0f;
  if (q <= NPARAM) {
#pragma unroll 8
    for (int c = lo; c < hi; ++c) g = g + part[(int64_t)c * PART_STRIDE + q];
  }
  sums[quarter][lane] = g;
  __syncthreads();
  if (quarter != 0 || q > NPARAM) return;
  g = ((sums[0][lane] + sums[1][lane]) + sums[2][lane]) + sums[3][lane];
  if (q == NPARAM) {
    if (loss_out) *loss_out = g;
    return;
  }
  if (grad) grad[q] = g;
  if (adam) {
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    const float mm = b1 * m[q] + (1.0f - b1) * g;
    const float vv = b2 * v[q] + (1.0f - b2) * (g * g);
    m[q] = mm;
    v[q] = vv;
    const float mh = mm / c1, vh = vv / c2;
    const float p = params[q] - lr * mh / (sqrtf(vh) + eps);
    params[q] = p;
    pack_param(q, p, wpk, bias);
  }
}

// ---- guided-batch helpers ----------------------------------------------------

__device__ inline int find_pair(const int64_t* pair_off, int num_pairs, int64_t k) {
  int lo = 0, hi = num_pairs - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (pair_off[mid] <= k)
      lo = mid;
    else
      hi = mid - 1;
  }
  return lo;
}

__global__ void k_local_iota(const int64_t* __restrict__ pair_off, int num_pairs, int64_t total,
                             int32_t* __restrict__ out) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= total) return;
  const int p = find_pair(pair_off, num_pairs, pair_off[0] + k);
  out[k] = (int32_t)(pair_off[0] + k - pair_off[p]);
}

__global__ void k_gather_rows(const double* __restrict__ corr, const int32_t* __restrict__ perm,
                              const int64_t* __restrict__ pair_off, int num_pairs, int64_t total,
                              double* __restrict__ sorted) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= total) return;
  const int p = find_pair(pair_off, num_pairs, pair_off[0] + k);
  const int64_t src = pair_off[p] - pair_off[0] + perm[k];
#pragma unroll
  for (int c = 0; c < 4; ++c) sorted[4 * k + c] = corr[4 * src + c];
}

// ---- launchers ------------------------------------------------------------------

void launch_pack(hipStream_t st, const float* params, uint16_t* wpk, float* bias) {
  hipLaunchKernelGGL(k_mlp_pack, dim3(HID * HID / 256), dim3(256), 0, st, params, wpk, bias);
}

void launch_predict(hipStream_t st, const uint16_t* wpk, const float* bias, const float* feat, int64_t n,
                    float* logit, float* prob) {
  if (n <= 0) return;
  int64_t blocks = (n + POINTS_PER_BLOCK - 1) / POINTS_PER_BLOCK;
  if (blocks > 2048) blocks = 2048;
  hipLaunchKernelGGL(k_mlp_predict, dim3((unsigned)blocks), dim3(256), sizeof(FwdLds), st, wpk, bias, feat, n,
                     logit, prob);
}

int train_blocks(int64_t batch) {
  const int64_t tiles = (batch + 31) / 32;
  return (int)(tiles < kTrainBlocks ? tiles : kTrainBlocks);
}

void launch_train(hipStream_t st, const uint16_t* wpk, const float* bias, const float* feat, const float* labels,
                  int64_t batch, int64_t sample_n, uint64_t seed, int64_t step, float inv_batch, float* part) {
  hipLaunchKernelGGL(k_mlp_train, dim3((unsigned)train_blocks(batch)), dim3(256), sizeof(TrainLds), st, wpk, bias,
                     feat, labels, batch, sample_n, seed, step, inv_batch, part);
}

void launch_reduce_adam(hipStream_t st, const float* part, int chunks, float* grad, float* loss_out, int adam,
                        float* params, float* m, float* v, float lr, float c1, float c2, uint16_t* wpk, float* bias) {
  hipLaunchKernelGGL(k_mlp_reduce, dim3((NPARAM + 1 + 63) / 64), dim3(256), 0, st, part, chunks, grad, loss_out, adam,
                     params, m, v, lr, c1, c2, wpk, bias);
}

void launch_local_iota(hipStream_t st, const int64_t* pair_off, int num_pairs, int64_t total, int32_t* out) {
  if (total <= 0) return;
  hipLaunchKernelGGL(k_local_iota, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, pair_off, num_pairs,
                     total, out);
}

void launch_gather_rows(hipStream_t st, const double* corr, const int32_t* perm, const int64_t* pair_off,
                        int num_pairs, int64_t total, double* sorted) {
  if (total <= 0) return;
  hipLaunchKernelGGL(k_gather_rows, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, corr, perm, pair_off,
                     num_pairs, total, sorted);
}

}  // namespace mlp
}  // namespace gcr
