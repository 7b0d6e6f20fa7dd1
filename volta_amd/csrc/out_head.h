// Row-level device code of the one-column output layer of a small batch,
// shared by skinny.hip's output launches and the last hidden layer's
// forward launch that also runs the output layer (gemm.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "device_common.h"
#include "skinny.h"

namespace volta {

// Output values z[g] of RG rows (rows[g], valid where rows[g] >= 0) of a
// one-column layer, computed by a whole wave: lane l sums k = l, l+64, ... in
// ascending order, then a fixed butterfly adds the lanes.  The k loop runs in
// chunks of C values per lane whose loads (W and all RG rows' activations) are
// issued before the chunk's first multiply, so a chunk costs one memory
// latency.  Every load is unconditional (clamped row and k; terms outside the
// matrix are not added), so no branch or wait separates them.
template <int RG, int C>
__device__ __forceinline__ void wave_rows(const OutLayerArgs& p, const int* rows, float (*z)[1]) {
  const int lane = threadIdx.x & 63;
  const int K = p.K;
  float acc[RG];
#pragma unroll
  for (int g = 0; g < RG; ++g) acc[g] = 0.0f;
  for (int kb = 0; kb < K; kb += 64 * C) {
    float x[RG][C], w[C];
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int kc = min(kb + 64 * c + lane, K - 1);
      w[c] = p.W[kc];
#pragma unroll
      for (int g = 0; g < RG; ++g) x[g][c] = p.act[(size_t)(rows[g] >= 0 ? rows[g] : 0) * K + kc];
    }
#pragma unroll
    for (int c = 0; c < C; ++c) {
#pragma unroll
      for (int g = 0; g < RG; ++g) {
        const float t = acc[g] + x[g][c] * w[c];
        acc[g] = kb + 64 * c + lane < K && rows[g] >= 0 ? t : acc[g];
      }
    }
  }
#pragma unroll
  for (int g = 0; g < RG; ++g) z[g][0] = wave_sum(acc[g]);
}

// Loss head of one row of a one-column layer: MSE (:792-798) d = z - y,
// loss += d^2, delta = 2d/nt; softmax-CE of one class (interpreter.rs:762-812,
// autograd.rs:467-534).  head_delta forms the row's delta and returns its loss
// without storing anything, so every lane of a wave can hold the delta;
// head_row also stores z and the delta.  `y` holds the row's target (MSE),
// `lab` its label (CE), both loaded before z was computed.
__device__ __forceinline__ float head_delta(const OutLayerArgs& p, const float* z, const float* y, int lab,
                                            float* d) {
  if (p.loss == VOLTA_LOSS_MSE) {
    const float dj = z[0] - y[0];
    d[0] = 2.0f * dj / (float)p.B;
    return 0.0f + dj * dj;
  }
  const float mx = fmaxf(-INFINITY, z[0]);
  const float sum = 0.0f + expf(z[0] - mx);
  const float lse = mx + logf(sum);
  const bool on = lab == 0;
  d[0] = (expf(z[0] - mx) / sum - (on ? 1.0f : 0.0f)) / (float)p.B;
  return on ? -(z[0] - lse) : __builtin_nanf("");
}

__device__ __forceinline__ float head_row(const OutLayerArgs& p, const float* z, const float* y, int lab, int m) {
  float d[1];
  const float l = head_delta(p, z, y, lab, d);
  p.out[m] = z[0];
  p.delta[m] = d[0];
  if (p.loss != VOLTA_LOSS_MSE && lab != 0) atomicOr(&p.scalars->flags, (uint32_t)VOLTA_STATUS_BAD_ARGUMENT);
  return l;
}

// Rows (waves) per block of the output launch that also forms dX_{n-1}.
constexpr int kOutDxRows = 4;
constexpr int kOutDxMaxBlocks = (kNarrowMaxB + kOutDxRows - 1) / kOutDxRows;

// Batch row m of a one-column output layer, computed by one wave: z =
// act_{n-1}[m] W + b, the loss head (z and delta_{n-1} stored by lane 0), and
// the row of delta_{n-2} = (delta_{n-1} W^T) * f'(layer n-2).  Returns the
// row's loss (0 for m >= B, whose loads are clamped and whose results are not
// stored).
__device__ __forceinline__ float out_dx_row(const OutLayerArgs& p, int m) {
  constexpr int C = 4;
  const int lane = threadIdx.x & 63;
  const int K = p.K;
  const bool has = m < p.B;
  const int mc = has ? m : p.B - 1;
  const bool mse = p.loss == VOLTA_LOSS_MSE;
  const float bias = p.bias[0];
  const float y[1] = {mse ? p.y[mc] : 0.0f};
  const int lab = mse ? 0 : p.labels[mc];
  const int rows[1] = {has ? m : -1};
  float z[1][1];
  wave_rows<1, C>(p, rows, z);
  z[0][0] = z[0][0] + bias;
  float d[1];
  const float row_loss = head_delta(p, z[0], y, lab, d);
  if (has && lane == 0) (void)head_row(p, z[0], y, lab, m);

  // delta_{n-2} of this row
  if (has) {
    const float* act = p.act + (size_t)m * K;
    const float* pre = p.dx_pre ? p.dx_pre + (size_t)m * K : act;
    float* out = p.dx_out + (size_t)m * K;
    for (int kb = 0; kb < K; kb += 64 * C) {
      float av[C], pv[C], wv[C];
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const int kc = min(kb + 64 * c + lane, K - 1);
        av[c] = act[kc];
        pv[c] = pre[kc];
        wv[c] = p.W[kc];
      }
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const int k = kb + 64 * c + lane;
        if (k < K) out[k] = (0.0f + d[0] * wv[c]) * act_derivative(p.dx_act, pv[c], av[c]);
      }
    }
  }
  return has ? row_loss : 0.0f;
}

// Rows rows[g] (g < RG) of a one-column output layer computed together by
// one wave, as out_dx_row computes each (wave_rows adds every row in the
// same k order whatever RG, then the same loss head), MSE only: lane 0
// writes each row's z to z_rows[g] and its delta_{n-1} to d_rows[g] (also
// for rows >= B), and every lane gets the row losses in losses[g] (0 for
// rows >= B).  Nothing is stored to global memory.
template <int RG>
__device__ __forceinline__ void out_head_rows(const OutLayerArgs& p, const int* rows, float* z_rows, float* d_rows,
                                              float* losses) {
  const int lane = threadIdx.x & 63;
  const float bias = p.bias[0];
  int wr[RG];
  float y[RG][1];
#pragma unroll
  for (int g = 0; g < RG; ++g) {
    const bool has = rows[g] < p.B;
    wr[g] = has ? rows[g] : -1;
    y[g][0] = p.y[has ? rows[g] : p.B - 1];
  }
  float z[RG][1];
  wave_rows<RG, 4>(p, wr, z);
#pragma unroll
  for (int g = 0; g < RG; ++g) {
    z[g][0] = z[g][0] + bias;
    float d[1];
    const float l = head_delta(p, z[g], y[g], 0, d);
    if (lane == 0) {
      z_rows[g] = z[g][0];
      d_rows[g] = d[0];
    }
    losses[g] = wr[g] >= 0 ? l : 0.0f;
  }
}

// The step's loss from the per-block partials (blocks of kOutDxRows rows,
// all loads issued together, added in block order), then the step counter
// and the arrival ticket reset; run by the one thread that arrived last.
__device__ __forceinline__ float out_dx_loss_sum(const float* partials, int nblocks) {
  float part[kOutDxMaxBlocks];
#pragma unroll
  for (int b = 0; b < kOutDxMaxBlocks; ++b) part[b] = partials[min(b, nblocks - 1)];
  float total = part[0];
#pragma unroll
  for (int b = 1; b < kOutDxMaxBlocks; ++b) {
    const float t = total + part[b];
    total = b < nblocks ? t : total;
  }
  return total;
}

__device__ __forceinline__ float out_dx_loss_denom(const OutLayerArgs& p) {
  return (float)p.B;  // B * 1 for MSE, B for CE
}

__device__ __forceinline__ void out_dx_finish(const OutLayerArgs& p, int nblocks, const StepNext& next) {
  step_finish(p.scalars, next, p.bc_table != nullptr, out_dx_loss_sum(p.partials, nblocks) / out_dx_loss_denom(p));
  *p.loss_counter = 0u;
}

// The deferred form: the loss of the partials an earlier output launch
// stored (launch_out_layer_dx with defer_loss), the same sum in block order,
// and its non-finite flag; the step counter was advanced by that launch.
__device__ __forceinline__ void deferred_loss_finish(DevScalars* sc, const float* partials, int nblocks,
                                                     float denom) {
  const float loss = out_dx_loss_sum(partials, nblocks) / denom;
  sc->loss = loss;
  if (!(fabsf(loss) <= 3.402823466e38f)) atomicOr(&sc->flags, (uint32_t)VOLTA_STATUS_NONFINITE_LOSS);
}

}  // namespace volta
