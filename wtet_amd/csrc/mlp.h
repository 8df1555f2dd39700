// Learned buffer presizing: per-cloud features and a small FP32 MLP.
//
// Features of a cloud (kFeat = 522): the 512-bin occupancy histogram of the
// top 9 bits of the 30-bit Morton code (10-bit floor quantization of each
// axis over the cloud's box, src/morton.rs:22-35), as fractions of the
// cloud's points; the mean (3) and covariance (6) of the box-normalized
// coordinates; log(n).  The network (kFeat -> 128 -> 128 -> 3, ReLU)
// predicts, in standardized log space, the tet slots the triangulation
// uses, the peak active-list length and the number of stuck faces, so that
// device buffers can be sized once.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace wtet {

constexpr int kHistBins = 512;
constexpr int kFeat = kHistBins + 3 + 6 + 1;
constexpr int kHidden = 128;
constexpr int kOut = 3;

// Parameter blob layout (floats): feature mean[kFeat], feature std[kFeat],
// target mean[kOut], target std[kOut], W1[kFeat*kHidden] (row-major, input
// major), b1[kHidden], W2[kHidden*kHidden], b2[kHidden], W3[kHidden*kOut],
// b3[kOut], margin[kOut] (log-space safety margin added to predictions).
constexpr size_t kOffFeatMean = 0;
constexpr size_t kOffFeatStd = kOffFeatMean + kFeat;
constexpr size_t kOffTgtMean = kOffFeatStd + kFeat;
constexpr size_t kOffTgtStd = kOffTgtMean + kOut;
constexpr size_t kOffW1 = kOffTgtStd + kOut;
constexpr size_t kOffB1 = kOffW1 + (size_t)kFeat * kHidden;
constexpr size_t kOffW2 = kOffB1 + kHidden;
constexpr size_t kOffB2 = kOffW2 + (size_t)kHidden * kHidden;
constexpr size_t kOffW3 = kOffB2 + kHidden;
constexpr size_t kOffB3 = kOffW3 + (size_t)kHidden * kOut;
constexpr size_t kOffMargin = kOffB3 + kOut;
constexpr size_t kParamCount = kOffMargin + kOut;
// trainable part: W1 .. b3
constexpr size_t kTrainBegin = kOffW1;
constexpr size_t kTrainEnd = kOffMargin;

// Per-cloud features from raw points (cloud c = points off[c]..off[c+1]).
// mm: per-cloud ordered-u32 min/max (as launch_prepare leaves it).
// acc: device scratch of C * (kHistBins + 9) doubles; feat: C * kFeat.
void launch_features(const float* xyz, uint32_t n, const uint32_t* off, uint32_t C,
                     const uint32_t* mm, double* acc, float* feat, hipStream_t s);

// Inference: pred[C * kOut] (un-standardized log targets + margin) from
// features feat[C * kFeat] with the parameter blob on the device.
void launch_mlp_predict(const float* params, const float* feat, uint32_t C, float* pred,
                        hipStream_t s);

// Training on a minibatch of B rows (mlp.hip): one kernel for what is local to
// a row (standardization, forward pass, loss, deltas), one for the weight
// gradients as partial sums over slices of kGradSlice rows, and one that adds
// the slices up.
constexpr int kRowTile = 16;      // rows a workgroup takes through the network
constexpr uint32_t kGradSlice = 256;
constexpr size_t kTrainCount = kTrainEnd - kTrainBegin;

struct MlpWork {
  float* x;     // B * kFeat (standardized features)
  float* h1;    // B * kHidden (post-ReLU)
  float* h2;    // B * kHidden
  float* d3;    // B * kOut
  float* d2;    // B * kHidden
  float* d1;    // B * kHidden
  float* part;  // mlp_slices(B) * kTrainCount: gradient slices
  float* lpart; // mlp_row_tiles(B): squared error of each row tile
};
inline uint32_t mlp_row_tiles(uint32_t B) { return (B + kRowTile - 1) / kRowTile; }
inline uint32_t mlp_slices(uint32_t B) { return (B + kGradSlice - 1) / kGradSlice; }

// rows idx[0..B) (null: 0..B-1) of the raw features and targets: forward pass,
// MSE loss and backward pass into w.part and w.lpart
void launch_mlp_forward_backward(const float* params, const float* feat, const float* tgt, const uint32_t* idx,
                                 const MlpWork& w, uint32_t B, hipStream_t s);
// the gradient (trainable range of grad) and the loss
void launch_mlp_gradient(const MlpWork& w, uint32_t B, float* grad, float* loss, hipStream_t s);
// the loss, and an Adam step on the trainable range with the gradient
void launch_mlp_adam(const MlpWork& w, uint32_t B, float* params, float* m, float* v, float lr, float b1,
                     float b2, float eps, uint32_t step, float* loss, hipStream_t s);

}  // namespace wtet
