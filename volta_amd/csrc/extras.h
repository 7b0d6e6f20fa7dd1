// Codegen extras of the generated step (LayerNorm, dropout, gradient
// clipping; mlp_train_rust_codegen.rs:745-788, :829-892, :936-955), as
// kernels around the GEMMs (extras.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "device_common.h"

namespace volta {

// One hidden layer's forward extras on act [B x c] (after the activation;
// with `softmax` act holds the pre-activation and the row softmax comes
// first).
struct HiddenFwdArgs {
  float* act;            // [B x c], updated in place
  int B, c;
  int softmax;           // 1: act = softmax(act) per row first
  const float* gamma;    // LayerNorm (null: off)
  const float* beta;
  float* mu;             // [B] per-row statistics kept for the backward
  float* inv_std;        // [B] (both null: not kept, inference)
  uint8_t* mask;         // dropout (null: off) [B x c]
  float p, keep_scale;
  uint64_t rng_offset;   // draws before this layer's first element in the step
  const DevScalars* scalars;  // rng = the step's starting state
};

// One hidden layer's backward extras (`din`: gradient w.r.t. the layer's
// final output): LayerNorm backward, dropout mask, activation derivative
// (softmax: the row form y * (d - dot(d, y))), in that order, and the
// LayerNorm gradients' column sums.
struct HiddenBwdArgs {
  const float* din;      // [B x c]: dL/d(layer output); with LayerNorm not `delta` itself
  float* delta;          // [B x c]: dL/d(pre-activation)
  const float* act;      // layer output (after LayerNorm / dropout)
  const float* pre;      // pre-activation
  int B, c, act_kind;
  const float* gamma;    // LayerNorm (null: off), pre-update values
  const float* beta;
  const float* inv_std;
  float* dgamma;         // [c] column sums (LayerNorm)
  float* dbeta;
  const uint8_t* mask;   // dropout (null: off)
  float keep_scale;
  DevScalars* scalars;   // rng_draws > 0: the dropout stream advances by that many draws (once per step)
  uint64_t rng_draws;
};

hipError_t launch_hidden_fwd(const HiddenFwdArgs& a, hipStream_t st);
// One launch; gamma and beta are left for the step's extras tail to update.
hipError_t launch_hidden_bwd(const HiddenBwdArgs& a, hipStream_t st);

// Gradient clipping over every layer's delta (up to 16 buffers): the global
// norm, scale = clip/norm when the norm exceeds clip (else 1, kept in
// scalars->clip_scale), then every delta multiplied by scale in place.
struct ClipArgs {
  int n;
  float* delta[16];
  int64_t count[16];
  float clip;
  float* partials;       // [kClipBlocks]
  DevScalars* scalars;   // receives clip_scale
};
constexpr int kClipBlocks = 256;
// The last pass of the clip (the partial sums are formed by the extras tail).
hipError_t launch_clip_apply(const ClipArgs& a, hipStream_t st);

// Sum of squares of every delta element, by block `block` of kClipBlocks (256
// threads): a fixed contiguous range of the layers' deltas taken in layer
// order; lanes add their strided elements, then a fixed butterfly and wave
// order.  Into partials[block].
__device__ __forceinline__ void clip_partial_block(const ClipArgs& a, int block, float* wave_part) {
  int64_t total = 0;
  for (int i = 0; i < a.n; ++i) total += a.count[i];
  const int64_t chunk = (total + kClipBlocks - 1) / kClipBlocks;
  const int64_t lo = (int64_t)block * chunk, hi = lo + chunk < total ? lo + chunk : total;
  float s = 0.0f;
  int layer = 0;
  int64_t layer_lo = 0;
  for (int64_t g = lo + threadIdx.x; g < hi; g += blockDim.x) {
    while (g >= layer_lo + a.count[layer]) {
      layer_lo += a.count[layer];
      ++layer;
    }
    const float v = a.delta[layer][g - layer_lo];
    s = s + v * v;
  }
  s = wave_sum(s);
  if ((threadIdx.x & 63) == 0) wave_part[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) a.partials[block] = wave_part[0] + wave_part[1] + wave_part[2] + wave_part[3];
}

}  // namespace volta
