// Learned presizing kernels: per-cloud features, MLP inference, and the
// forward / backward / Adam kernels that train the network on the GPU.
// All FP32 except the feature moments (f64 accumulation).
#include <algorithm>
#include <cstring>

#include "kernels.h"
#include "mlp.h"

namespace wtet {

namespace {

__device__ __forceinline__ uint32_t gtid() { return blockIdx.x * blockDim.x + threadIdx.x; }

// spread the low 10 bits of v to every third bit
__device__ __forceinline__ uint32_t expand10(uint32_t v) {
  v &= 0x3FFu;
  v = (v | (v << 16)) & 0x030000FFu;
  v = (v | (v << 8)) & 0x0300F00Fu;
  v = (v | (v << 4)) & 0x030C30C3u;
  v = (v | (v << 2)) & 0x09249249u;
  return v;
}

constexpr int kMom = 9;

__device__ __forceinline__ double wave_sum(double v) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  return v;
}

}  // namespace

// Histogram counts (u32) and coordinate moments (f64) per cloud.  Each
// block accumulates the points of its first cloud in LDS (histogram and
// moments) and adds them to the global arrays once at the end; points of
// other clouds go straight to the global arrays.  One cloud: a grid-stride
// loop over a few hundred blocks, so that the global adds are per block
// and not per point (a global atomic per point on 512 words serializes at
// the memory side).  Many clouds: one point per thread, so that a block's
// points mostly share a cloud.
__global__ void __launch_bounds__(kBlock) k_feat_accum(const float* xyz, uint32_t n, const uint32_t* off,
                                                       uint32_t C, const uint32_t* mm, uint32_t* hist,
                                                       double* mom) {
  __shared__ uint32_t lh[kHistBins];
  __shared__ double lm[kMom];
  for (int b = threadIdx.x; b < kHistBins; b += blockDim.x) lh[b] = 0u;
  if (threadIdx.x < kMom) lm[threadIdx.x] = 0.0;
  const uint32_t first = blockIdx.x * blockDim.x;
  const uint32_t cb = (C > 1 && first < n) ? cloud_of_point(off, C, first) : 0u;
  __syncthreads();
  double m[kMom] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  const uint32_t stride = gridDim.x * blockDim.x;
  for (uint32_t i = gtid(); i < n; i += stride) {
    uint32_t c = C > 1 ? cloud_of_point(off, C, i) : 0u;
    const uint32_t* b = mm + 6 * (size_t)c;
    float u[3];
    uint32_t q[3];
    for (int k = 0; k < 3; ++k) {
      float lo = unord_f32(b[k]), hi = unord_f32(b[3 + k]);
      float ext = hi - lo;
      float v = ext > 0.0f ? (xyz[3 * (size_t)i + k] - lo) / ext : 0.0f;
      v = v < 0.0f ? 0.0f : (v > 1.0f ? 1.0f : v);
      u[k] = v;
      q[k] = (uint32_t)(v * 1023.0f);
    }
    uint32_t code = (expand10(q[2]) << 2) | (expand10(q[1]) << 1) | expand10(q[0]);
    double pm[kMom] = {u[0], u[1], u[2], (double)u[0] * u[0], (double)u[1] * u[1], (double)u[2] * u[2],
                       (double)u[0] * u[1], (double)u[0] * u[2], (double)u[1] * u[2]};
    if (c == cb) {
      atomicAdd(&lh[code >> 21], 1u);
      for (int k = 0; k < kMom; ++k) m[k] += pm[k];
    } else {
      atomicAdd(&hist[(size_t)c * kHistBins + (code >> 21)], 1u);
      for (int k = 0; k < kMom; ++k) atomicAdd(&mom[(size_t)c * kMom + k], pm[k]);
    }
  }
  // the block's own cloud: wave sums into LDS, then one global add each
  for (int k = 0; k < kMom; ++k) {
    double w = wave_sum(m[k]);
    if (__lane_id() == 0 && w != 0.0) atomicAdd(&lm[k], w);
  }
  __syncthreads();
  if (first < n) {
    for (int b = threadIdx.x; b < kHistBins; b += blockDim.x)
      if (lh[b]) atomicAdd(&hist[(size_t)cb * kHistBins + b], lh[b]);
    if (threadIdx.x < kMom && lm[threadIdx.x] != 0.0)
      atomicAdd(&mom[(size_t)cb * kMom + threadIdx.x], lm[threadIdx.x]);
  }
}

__global__ void k_feat_finish(const uint32_t* off, uint32_t C, const uint32_t* hist,
                              const double* mom, float* feat) {
  uint32_t g = gtid();
  if (g >= (uint64_t)C * kFeat) return;
  uint32_t c = g / kFeat, k = g - c * kFeat;
  double n = (double)(off[c + 1] - off[c]);
  const double* M = mom + (size_t)c * kMom;
  float v;
  if (k < (uint32_t)kHistBins) {
    v = (float)(hist[(size_t)c * kHistBins + k] / n);
  } else if (k < (uint32_t)kHistBins + 3) {
    v = (float)(M[k - kHistBins] / n);
  } else if (k < (uint32_t)kHistBins + 9) {
    // covariance: xx, yy, zz, xy, xz, yz
    const int a[6] = {0, 1, 2, 0, 0, 1}, b[6] = {0, 1, 2, 1, 2, 2};
    int j = (int)k - kHistBins - 3;
    v = (float)(M[3 + j] / n - (M[a[j]] / n) * (M[b[j]] / n));
  } else {
    v = (float)log(n);
  }
  feat[g] = v;
}

void launch_features(const float* xyz, uint32_t n, const uint32_t* off, uint32_t C,
                     const uint32_t* mm, double* acc, float* feat, hipStream_t s) {
  uint32_t* hist = reinterpret_cast<uint32_t*>(acc);  // C * kHistBins u32 at the front
  double* mom = acc + ((size_t)C * kHistBins + 1) / 2;
  launch_fill_u32(hist, 0u, (uint64_t)C * kHistBins, s);
  launch_fill_u64(reinterpret_cast<uint64_t*>(mom), 0ull, (uint64_t)C * kMom, s);
  uint32_t grid = C > 1 ? nblocks(n) : std::min(nblocks(n), 512u);
  if (n) k_feat_accum<<<grid, kBlock, 0, s>>>(xyz, n, off, C, mm, hist, mom);
  k_feat_finish<<<nblocks((uint64_t)C * kFeat), kBlock, 0, s>>>(off, C, hist, mom, feat);
}

// one block of kHidden threads per cloud
__global__ void __launch_bounds__(kHidden) k_mlp_predict(const float* P, const float* feat,
                                                         uint32_t C, float* pred) {
  __shared__ float x[kFeat];
  __shared__ float h1[kHidden];
  __shared__ float h2[kHidden];
  uint32_t c = blockIdx.x;
  int t = threadIdx.x;
  if (c >= C) return;
  for (int k = t; k < kFeat; k += kHidden)
    x[k] = (feat[(size_t)c * kFeat + k] - P[kOffFeatMean + k]) / P[kOffFeatStd + k];
  __syncthreads();
  float a = P[kOffB1 + t];
  for (int k = 0; k < kFeat; ++k) a += x[k] * P[kOffW1 + (size_t)k * kHidden + t];
  h1[t] = a > 0.0f ? a : 0.0f;
  __syncthreads();
  a = P[kOffB2 + t];
  for (int k = 0; k < kHidden; ++k) a += h1[k] * P[kOffW2 + (size_t)k * kHidden + t];
  h2[t] = a > 0.0f ? a : 0.0f;
  __syncthreads();
  if (t < kOut) {
    a = P[kOffB3 + t];
    for (int k = 0; k < kHidden; ++k) a += h2[k] * P[kOffW3 + (size_t)k * kOut + t];
    pred[(size_t)c * kOut + t] = a * P[kOffTgtStd + t] + P[kOffTgtMean + t] + P[kOffMargin + t];
  }
}

void launch_mlp_predict(const float* params, const float* feat, uint32_t C, float* pred,
                        hipStream_t s) {
  if (C) k_mlp_predict<<<C, kHidden, 0, s>>>(params, feat, C, pred);
}

// ---------------------------------------------------------------------------
// training
//
// What bounds it: a minibatch is 0.3 to 3 GFLOP of small products (128 wide),
// a few microseconds on the matrix cores, so launches, dependent round trips
// and idle CUs set the time.  Hence three launches a step: everything local
// to a row in one (a workgroup holds its 16 rows' activations in LDS), the
// weight gradients split over rows to fill the chip, and their sum.  FP32
// MFMA, FP32 accumulation.  2,048 rows: 12 launches and 1,440 us of kernel
// time (a thread per column summed 2,048 rows for the bias gradients, 355 us
// each); now 3 launches and 64 us (rows 47, gradients 13, sum 4).
// ---------------------------------------------------------------------------
typedef float f32x4 __attribute__((ext_vector_type(4)));
// the same at any float's address (the parameter blob is packed)
typedef float f32x4_packed __attribute__((ext_vector_type(4), aligned(4)));

// v_mfma_f32_16x16x4_f32: lane l holds A[l % 16][l / 16] and B[l / 16][l % 16]
// and receives D[4 (l / 16) + r][l % 16] in register r
__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

constexpr int kXPad = 528;     // kFeat up to a multiple of 16
constexpr int kXStride = 532;  // LDS rows 16-byte aligned, spread over the banks
constexpr int kHStride = 132;
static_assert(kXPad >= kFeat + 1 && kXPad % 16 == 0, "room for the bias row");

// A (16 x 16 KC, rows of `stride` floats in LDS) times columns col..col + 15 of
// W (K x kHidden row-major, or with TW its transpose).  Of the 16 k of a step,
// lane quarter q takes k = 4 q .. 4 q + 3, one per MFMA.
template <int KC, bool TW>
__device__ __forceinline__ f32x4 rows_times(const float* a, int stride, const float* W, int K, int col) {
  const int i = __lane_id() & 15, q = __lane_id() >> 4;
  f32x4 acc = {};
#pragma unroll 8
  for (int c = 0; c < KC; ++c) {
    const int k = 16 * c + 4 * q;
    const f32x4 av = *reinterpret_cast<const f32x4*>(a + i * stride + k);
    f32x4 b;
    if (TW) {
      b = *reinterpret_cast<const f32x4_packed*>(W + (size_t)(col + i) * kHidden + k);
    } else {
#pragma unroll
      for (int s = 0; s < 4; ++s) b[s] = k + s < K ? W[(size_t)(k + s) * kHidden + col + i] : 0.0f;
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) acc = mfma4(av[s], b[s], acc);
  }
  return acc;
}

// One workgroup takes 16 rows through the network and back: eight waves, 16 of
// the 128 hidden columns each.
constexpr int kRowThreads = 512;

__global__ void __launch_bounds__(kRowThreads) k_mlp_rows(const float* P, const float* feat, const float* tgt,
                                                          const uint32_t* idx, uint32_t B, MlpWork w) {
  __shared__ __align__(16) float xs[kRowTile * kXStride];  // later the deltas of layer 2
  __shared__ __align__(16) float h1s[kRowTile * kHStride];
  __shared__ __align__(16) float h2s[kRowTile * kHStride];
  __shared__ float d3s[kRowTile * 4];
  __shared__ float ls[kRowThreads / 64];
  const uint32_t r0 = blockIdx.x * kRowTile;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  // 32 threads per row
  {
    const int r = t / 32;
    const uint32_t row = r0 + r, src = row < B ? (idx ? idx[row] : row) : 0u;
    for (int k = t & 31; k < kXPad; k += 32) {
      float v = 0.0f;
      if (row < B && k < kFeat) {
        v = (feat[(size_t)src * kFeat + k] - P[kOffFeatMean + k]) / P[kOffFeatStd + k];
        w.x[(size_t)row * kFeat + k] = v;
      }
      xs[r * kXStride + k] = v;
    }
  }
  __syncthreads();
  const int j = lane & 15, q = lane >> 4, cl = 16 * wave + j;
  // relu(acc + bias) to LDS and memory
  auto hidden = [&](f32x4 acc, const float* bias, float* hs, float* h) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = 4 * q + r;
      float v = acc[r] + bias[cl];
      v = v > 0.0f ? v : 0.0f;
      hs[row * kHStride + cl] = v;
      if (r0 + row < B) h[(size_t)(r0 + row) * kHidden + cl] = v;
    }
  };
  hidden(rows_times<kXPad / 16, false>(xs, kXStride, P + kOffW1, kFeat, 16 * wave), P + kOffB1, h1s, w.h1);
  __syncthreads();
  hidden(rows_times<kHidden / 16, false>(h1s, kHStride, P + kOffW2, kHidden, 16 * wave), P + kOffB2, h2s, w.h2);
  __syncthreads();
  // outputs, loss and their deltas: eight lanes per (row, output)
  float sq = 0.0f;
  if (t < kRowTile * kOut * 8) {
    const int part = t & 7, ro = t >> 3, row = ro / kOut, o = ro - row * kOut;
    float a = 0.0f;
#pragma unroll
    for (int k = 0; k < kHidden / 8; ++k)
      a += h2s[row * kHStride + 8 * k + part] * P[kOffW3 + (size_t)(8 * k + part) * kOut + o];
    a += __shfl_xor(a, 1);
    a += __shfl_xor(a, 2);
    a += __shfl_xor(a, 4);
    float d = 0.0f;
    if (r0 + row < B) {
      const uint32_t src = idx ? idx[r0 + row] : r0 + row;
      const float y = (tgt[(size_t)src * kOut + o] - P[kOffTgtMean + o]) / P[kOffTgtStd + o];
      const float e = a + P[kOffB3 + o] - y;
      d = 2.0f * e / (float)(B * kOut);
      if (part == 0) {
        w.d3[(size_t)(r0 + row) * kOut + o] = d;
        sq = e * e;
      }
    }
    if (part == 0) d3s[row * 4 + o] = d;
  }
  for (int off = 32; off > 0; off >>= 1) sq += __shfl_xor(sq, off);
  if (lane == 0) ls[wave] = sq;
  __syncthreads();
  if (t == 0) {
    float a = 0.0f;
    for (int k = 0; k < kRowThreads / 64; ++k) a += ls[k];
    w.lpart[blockIdx.x] = a;
  }
  float* d2s = xs;
  for (int e = t; e < kRowTile * kHidden; e += kRowThreads) {
    const int row = e / kHidden, k = e - row * kHidden;
    float v = 0.0f;
    for (int o = 0; o < kOut; ++o) v += d3s[row * 4 + o] * P[kOffW3 + (size_t)k * kOut + o];
    if (!(h2s[row * kHStride + k] > 0.0f)) v = 0.0f;
    d2s[row * kHStride + k] = v;
    if (r0 + row < B) w.d2[(size_t)(r0 + row) * kHidden + k] = v;
  }
  __syncthreads();
  const f32x4 acc = rows_times<kHidden / 16, true>(d2s, kHStride, P + kOffW2, kHidden, 16 * wave);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int row = 4 * q + r;
    const float v = h1s[row * kHStride + cl] > 0.0f ? acc[r] : 0.0f;
    if (r0 + row < B) w.d1[(size_t)(r0 + row) * kHidden + cl] = v;
  }
}

// Gradient of one weight matrix, G = A^T D over a slice of rows: 16 inputs by
// 16 NT outputs per workgroup, its four waves a quarter of the slice each.
// The input after the last is constant 1: its row is the bias gradient, which
// follows the weights in the parameters.
template <int NT>
__device__ __forceinline__ void grad_tile(const float* A, int F, const float* D, int N, int f0, int col,
                                          uint32_t rb, uint32_t re, float* G, float* red) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, i = lane & 15, q = lane >> 4;
  const int f = f0 + i;
  f32x4 acc[NT] = {};
  const uint32_t w0 = rb + wave * (kGradSlice / 4);
#pragma unroll
  for (uint32_t c = 0; c < kGradSlice / 4; c += 16) {
    float a[4], b[NT][4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const uint32_t r = w0 + c + 4 * q + s;
      const bool in = r < re;
      a[s] = in ? (f < F ? A[(size_t)r * F + f] : (f == F ? 1.0f : 0.0f)) : 0.0f;
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        const int h = col + 16 * n + i;
        b[n][s] = in && h < N ? D[(size_t)r * N + h] : 0.0f;
      }
    }
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int n = 0; n < NT; ++n) acc[n] = mfma4(a[s], b[n][s], acc[n]);
  }
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int r = 0; r < 4; ++r) red[((wave * NT + n) * 4 + r) * 64 + lane] = acc[n][r];
  __syncthreads();
  // thread (wave, lane) adds the four waves' sums of tiles wave, wave + 4, ..
  for (int n = wave; n < NT; n += 4)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float v = 0.0f;
#pragma unroll
      for (int u = 0; u < 4; ++u) v += red[((u * NT + n) * 4 + r) * 64 + lane];
      const int fo = f0 + 4 * q + r, h = col + 16 * n + i;
      if (fo <= F && h < N) G[(size_t)fo * N + h] = v;
    }
}

constexpr int kW1Tiles = kXPad / 16, kW2Tiles = kHidden / 16 + 1, kW3Tiles = kHidden / 16 + 1;

// blockIdx.x: gradient tile (W1 and W2 in halves of 64 outputs, W3 whole);
// blockIdx.y: slice of rows
__global__ void __launch_bounds__(256) k_mlp_grads(MlpWork w, uint32_t B) {
  __shared__ float red[4 * 4 * 4 * 64];
  const uint32_t rb = blockIdx.y * kGradSlice, re = min(B, rb + kGradSlice);
  float* G = w.part + (size_t)blockIdx.y * kTrainCount;
  int t = blockIdx.x;
  if (t < 2 * kW1Tiles) {
    grad_tile<4>(w.x, kFeat, w.d1, kHidden, 16 * (t >> 1), 64 * (t & 1), rb, re, G, red);
    return;
  }
  t -= 2 * kW1Tiles;
  if (t < 2 * kW2Tiles) {
    grad_tile<4>(w.h1, kHidden, w.d2, kHidden, 16 * (t >> 1), 64 * (t & 1), rb, re, G + (kOffW2 - kTrainBegin), red);
    return;
  }
  t -= 2 * kW2Tiles;
  grad_tile<1>(w.h2, kHidden, w.d3, kOut, 16 * t, 0, rb, re, G + (kOffW3 - kTrainBegin), red);
}
static_assert(kOffB1 == kOffW1 + (size_t)kFeat * kHidden && kOffB2 == kOffW2 + (size_t)kHidden * kHidden &&
                  kOffB3 == kOffW3 + (size_t)kHidden * kOut,
              "each bias follows its weights");

struct AdamStep {
  float *p, *m, *v;
  float lr, b1, b2, eps, c1, c2;
};

// Sums the slices into the gradient, or, with ADAM, takes the step; block 0
// also adds up the loss.
template <bool ADAM>
__global__ void __launch_bounds__(kBlock) k_mlp_sum(MlpWork w, uint32_t B, uint32_t slices, float* grad, AdamStep A,
                                                    float* loss) {
  const uint32_t i = gtid();
  if (i < (uint32_t)kTrainCount) {
    float g = 0.0f;
    for (uint32_t s = 0; s < slices; ++s) g += w.part[(size_t)s * kTrainCount + i];
    if (ADAM) {
      const float mi = A.b1 * A.m[i] + (1.0f - A.b1) * g;
      const float vi = A.b2 * A.v[i] + (1.0f - A.b2) * g * g;
      A.m[i] = mi;
      A.v[i] = vi;
      A.p[i] -= A.lr * (mi / A.c1) / (sqrtf(vi / A.c2) + A.eps);
    } else {
      grad[i] = g;
    }
  }
  if (blockIdx.x == 0 && threadIdx.x < 64) {
    float a = 0.0f;
    const uint32_t tiles = (B + kRowTile - 1) / kRowTile;
    for (uint32_t k = threadIdx.x; k < tiles; k += 64) a += w.lpart[k];
    for (int off = 32; off > 0; off >>= 1) a += __shfl_xor(a, off);
    if (threadIdx.x == 0) loss[0] = a / (float)(B * kOut);
  }
}

void launch_mlp_forward_backward(const float* params, const float* feat, const float* tgt, const uint32_t* idx,
                                 const MlpWork& w, uint32_t B, hipStream_t s) {
  if (!B) return;
  k_mlp_rows<<<mlp_row_tiles(B), kRowThreads, 0, s>>>(params, feat, tgt, idx, B, w);
  k_mlp_grads<<<dim3(2 * kW1Tiles + 2 * kW2Tiles + kW3Tiles, mlp_slices(B)), 256, 0, s>>>(w, B);
}

void launch_mlp_gradient(const MlpWork& w, uint32_t B, float* grad, float* loss, hipStream_t s) {
  if (!B) return;
  k_mlp_sum<false><<<nblocks(kTrainCount), kBlock, 0, s>>>(w, B, mlp_slices(B), grad + kTrainBegin, AdamStep{}, loss);
}

void launch_mlp_adam(const MlpWork& w, uint32_t B, float* params, float* m, float* v, float lr, float b1,
                     float b2, float eps, uint32_t step, float* loss, hipStream_t s) {
  if (!B) return;
  const AdamStep A = {params + kTrainBegin, m + kTrainBegin, v + kTrainBegin, lr, b1, b2, eps,
                      1.0f - powf(b1, (float)step), 1.0f - powf(b2, (float)step)};
  k_mlp_sum<true><<<nblocks(kTrainCount), kBlock, 0, s>>>(w, B, mlp_slices(B), nullptr, A, loss);
}

}  // namespace wtet
