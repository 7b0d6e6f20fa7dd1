// Host interface of the non-GEMM step kernels (step_kernels.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "device_common.h"
#include "recorder.h"

namespace volta {

// Parameter, gradient and optimizer-state buffers are flat, one segment per
// W_i and per b_i, each padded to kSegAlign floats so every optimizer
// workgroup stays inside one segment.
constexpr int kSegAlign = 1024;
constexpr int kMaxSegments = 2 * (VOLTA_MAX_LAYER_SIZES - 1);

struct SegTable {
  int n;
  int64_t off[kMaxSegments];    // first float of the segment in the flat buffer
  int64_t count[kMaxSegments];  // real (unpadded) element count
  float wd[kMaxSegments];       // weight decay applied to this segment
};

// What a stand-alone loss head needs beside its operands: where the step's
// loss goes, and for more than one block their partial sums (one float per
// block, loss_head_blocks of them) and an arrival counter (zero between
// launches).
struct LossHead {
  DevScalars* scalars = nullptr;
  const float2* bc_table = nullptr;  // Adam bias-correction table (null without Adam)
  int bc_len = 0;
  float* partials = nullptr;
  unsigned* counter = nullptr;
};
constexpr int kLossMaxBlocks = 1024;
int loss_head_blocks(int loss, int B, int C);
// delta [B x C] and the step's loss from z / yhat [B x C].
hipError_t launch_loss_mse(const float* yhat, const float* y, float* delta, int B, int C, const LossHead& h,
                           hipStream_t st);
hipError_t launch_loss_ce(const float* z, const int32_t* labels, float* delta, int B, int C, const LossHead& h,
                          hipStream_t st);
// A step's inputs into the resident batch by one launch: nx words of x and ny
// words of y (either count 0: not copied), from device memory or from pinned
// host memory.  With `done` set (pinned host memory), the launch stores `seq`
// there once every source word has been read; `ticket` (device, zero between
// launches) counts the blocks.
struct InputCopy {
  const uint32_t* x = nullptr;
  uint32_t* x_dst = nullptr;
  size_t nx = 0;
  const uint32_t* y = nullptr;
  uint32_t* y_dst = nullptr;
  size_t ny = 0;
  uint32_t* done = nullptr;
  uint32_t seq = 0;
  unsigned* ticket = nullptr;
};
hipError_t launch_input_copy(const InputCopy& c, hipStream_t st);

hipError_t launch_adam(float* w, float* m, float* v, const float* g, const SegTable& segs,
                       int64_t total, const DevScalars* sc, float b1, float b2, float eps,
                       hipStream_t st);
hipError_t launch_adagrad(float* w, float* G, const float* g, const SegTable& segs, int64_t total,
                          const DevScalars* sc, float eps, hipStream_t st);

}  // namespace volta
