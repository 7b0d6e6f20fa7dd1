// Non-GEMM kernels of the MLP step: the stand-alone loss heads (used when the
// output layer is wider than one GEMM tile) and flat optimizer passes (the
// step fuses the optimizer into the dW epilogue; these run the same element
// functions over whole buffers for checks).  All reductions use a fixed
// association order and no floating-point atomics.
#include "step_kernels.h"

#include <algorithm>

namespace volta {

// The stand-alone loss heads: the output layer's logits are in memory, the
// rows (CE) or elements (MSE) are spread over the chip, and the step's loss is
// formed by whichever block finishes last.
//
// A block publishes its loss sum (publish_partial); the block that finishes
// last adds the partials (thread t: blocks t, t + 256, ... in order, then a
// fixed butterfly and the waves in order), so the sum does not depend on the
// arrival order.
constexpr int kLossThreads = 256;
constexpr int kLossWaves = kLossThreads / kWave;

// Block-wide sum with a fixed order: butterfly inside each wave, then wave
// partials added in wave order.  Result valid in thread 0.
__device__ __forceinline__ float block_sum_fixed(float v, float* lds) {
  v = wave_sum(v);
  const int wave = threadIdx.x >> 6;
  __syncthreads();  // earlier readers of lds are done
  if ((threadIdx.x & 63) == 0) lds[wave] = v;
  __syncthreads();
  float s = lds[0];
#pragma unroll
  for (int w = 1; w < kLossWaves; ++w) s = s + lds[w];
  return s;
}

// The block's sum `s` (thread 0) into the step's loss: sum / denom.  `next`:
// thread 0's step_prefetch from the kernel's start (only the block that
// finishes last writes the counter, after every block has started).
__device__ __forceinline__ void loss_finish(float s, float denom, const LossHead& h, const StepNext& next,
                                            float* lds) {
  if (gridDim.x == 1) {
    if (threadIdx.x == 0) step_finish(h.scalars, next, h.bc_table != nullptr, s / denom);
    return;
  }
  __shared__ unsigned last;
  if (threadIdx.x == 0) last = publish_partial(h.partials, h.counter, blockIdx.x, gridDim.x, s) ? 1u : 0u;
  __syncthreads();
  if (!last) return;  // block-uniform
  float t = 0.0f;
  for (unsigned b = threadIdx.x; b < gridDim.x; b += kLossThreads) t = t + published_partial(h.partials, b);
  t = block_sum_fixed(t, lds);
  if (threadIdx.x == 0) {
    step_finish(h.scalars, next, h.bc_table != nullptr, t / denom);
    *h.counter = 0u;  // for the next step's launch
  }
}

// MSE head (mlp_train_rust_codegen.rs:792-798): d = yhat - y,
// loss = sum(d^2)/nt, delta = 2*d/nt with nt = B*Ln.  Block b takes elements
// [b * per, (b + 1) * per).
__global__ void __launch_bounds__(kLossThreads)
loss_mse_kernel(const float* __restrict__ yhat, const float* __restrict__ y, float* __restrict__ delta, int nt,
                int per, LossHead h) {
  __shared__ float lds[kLossWaves];
  StepNext next{};
  if (threadIdx.x == 0) next = step_prefetch(h.scalars, h.bc_table, h.bc_len);
  const float ntf = (float)nt;
  const int64_t lo = (int64_t)blockIdx.x * per;
  const int64_t hi = lo + per < nt ? lo + per : nt;
  float acc = 0.0f;
  for (int64_t k = lo + threadIdx.x; k < hi; k += kLossThreads) {
    const float d = yhat[k] - y[k];
    acc = acc + d * d;
    delta[k] = 2.0f * d / ntf;
  }
  loss_finish(block_sum_fixed(acc, lds), ntf, h, next, lds);
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, kWave));
  return v;
}

// Softmax cross-entropy head with integer labels.
// Loss (interpreter.rs:762-812): per row max, sum of exp(z - max),
// lse = max + ln(sum), sample loss -(z_label - lse); mean over B.
// Gradient (autograd.rs:467-534): (softmax(z) - onehot) / B with
// softmax = exp(z - max) / sum (kernels/reduce.rs:203-213).
// One wave per row, rows_per_wave of them in turn: lane l takes columns l,
// l + 64, ... (a row of up to 64 * PER columns stays in registers with its
// exponentials; PER = 0 reads it again from the cache), the row's maximum and
// exp sum by butterflies.  An out-of-range label raises BAD_ARGUMENT and makes
// that row's loss NaN (it is never used as an index).
// Latency bound: one load round, two butterflies and one store per row.  One
// thread per row in a single block took 452 us of the 2961 us step of
// 1500-3000-3000-1000-100 at B=2000 (2505 us a step with this), and 42 us of
// the 61 us step of 800-384-100 at B=1 (24 us).
template <int PER>
__global__ void __launch_bounds__(kLossThreads)
loss_ce_kernel(const float* __restrict__ z, const int32_t* __restrict__ labels, float* __restrict__ delta, int B,
               int C, int rows_per_wave, LossHead h) {
  __shared__ float lds[kLossWaves];
  constexpr int R = PER > 0 ? PER : 1;
  StepNext next{};
  if (threadIdx.x == 0) next = step_prefetch(h.scalars, h.bc_table, h.bc_len);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const float bf = (float)B;
  float acc = 0.0f;  // lane 0: the wave's row losses in row order
  bool bad = false;
  const int row0 = (blockIdx.x * kLossWaves + wave) * rows_per_wave;
  for (int b = row0; b < min(B, row0 + rows_per_wave); ++b) {  // wave-uniform
    const float* zr = z + (size_t)b * C;
    float* dr = delta + (size_t)b * C;
    const int lab = labels[b];
    const bool ok = lab >= 0 && lab < C;
    const float zl = zr[ok ? lab : 0];
    float v[R];
    float mx = -INFINITY, sum = 0.0f;
    if constexpr (PER > 0) {
#pragma unroll
      for (int i = 0; i < R; ++i) v[i] = zr[min(lane + 64 * i, C - 1)];
#pragma unroll
      for (int i = 0; i < R; ++i) mx = fmaxf(mx, v[i]);  // a repeated last column changes no maximum
    } else {
      for (int j = lane; j < C; j += 64) mx = fmaxf(mx, zr[j]);
    }
    mx = wave_max(mx);
    if constexpr (PER > 0) {
#pragma unroll
      for (int i = 0; i < R; ++i) {
        v[i] = expf(v[i] - mx);
        sum = lane + 64 * i < C ? sum + v[i] : sum;
      }
    } else {
      for (int j = lane; j < C; j += 64) sum = sum + expf(zr[j] - mx);
    }
    sum = wave_sum(sum);
    auto grad = [&](int j, float e) { dr[j] = (e / sum - (j == lab ? 1.0f : 0.0f)) / bf; };
    if constexpr (PER > 0) {
#pragma unroll
      for (int i = 0; i < R; ++i)
        if (lane + 64 * i < C) grad(lane + 64 * i, v[i]);
    } else {
      for (int j = lane; j < C; j += 64) grad(j, expf(zr[j] - mx));
    }
    acc = acc + (ok ? -(zl - (mx + logf(sum))) : __builtin_nanf(""));
    bad |= !ok;
  }
  if (bad && lane == 0) atomicOr(&h.scalars->flags, (uint32_t)VOLTA_STATUS_BAD_ARGUMENT);
  __syncthreads();
  if (lane == 0) lds[wave] = acc;
  __syncthreads();
  float s = lds[0];
#pragma unroll
  for (int w = 1; w < kLossWaves; ++w) s = s + lds[w];
  __syncthreads();
  loss_finish(s, bf, h, next, lds);
}

// A step's inputs into the resident batch.  Blocks [0, xb) copy x, the rest y:
// 16-byte accesses where source and destination allow them, 4-byte ones
// otherwise and for the last words; a block's loads are all issued before its
// first store.  One launch of a few blocks: 2 us on the queue, where a
// hipMemcpyAsync each for x and y took 4 us of a 52 us step on the device and
// 14 us of host time, and one from pinned host memory, on a copy engine, 20 us
// of a 28 us step.
template <int U>
__device__ __forceinline__ void copy_words(const uint32_t* src, uint32_t* dst, size_t n, unsigned block,
                                           unsigned blocks) {
  const size_t t = (size_t)block * blockDim.x + threadIdx.x, all = (size_t)blocks * blockDim.x;
  size_t head = 0;  // words copied four at a time
  if ((((uintptr_t)src | (uintptr_t)dst) & 15) == 0) {
    const size_t n4 = n / 4;
    const uint4* s4 = reinterpret_cast<const uint4*>(src);
    uint4* d4 = reinterpret_cast<uint4*>(dst);
    for (size_t i = t; i < n4; i += U * all) {
      uint4 v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) v[u] = s4[i + u * all < n4 ? i + u * all : i];
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (i + u * all < n4) d4[i + u * all] = v[u];
    }
    head = n4 * 4;
  }
  for (size_t i = head + t; i < n; i += 4 * all) {
    uint32_t v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = src[i + u * all < n ? i + u * all : i];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (i + u * all < n) dst[i + u * all] = v[u];
  }
}

template <int U>
__global__ void __launch_bounds__(256) input_copy_kernel(InputCopy c, int xb) {
  if ((int)blockIdx.x < xb) copy_words<U>(c.x, c.x_dst, c.nx, blockIdx.x, xb);
  else copy_words<U>(c.y, c.y_dst, c.ny, blockIdx.x - xb, gridDim.x - xb);
  if (!c.done) return;
  // every load of the block has returned (its stores took the values) once
  // its memory counter is at zero
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x != 0) return;
  if (__hip_atomic_fetch_add(c.ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1u) {
    __hip_atomic_store(c.ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(c.done, c.seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// Find the segment holding flat element `base` (segments are padded to
// kSegAlign floats, so a whole block lies in one segment).
__device__ __forceinline__ int find_segment(const SegTable& t, int64_t base) {
  int s = 0;
  for (int i = 1; i < t.n; ++i)
    if (base >= t.off[i]) s = i;
  return s;
}

// Adam / AdamW over a flat segmented buffer (adam_update,
// mlp_train_rust_codegen.rs:326-388; the tail rule is per segment).
__global__ void __launch_bounds__(256)
adam_kernel(float* __restrict__ w, float* __restrict__ m, float* __restrict__ v,
            const float* __restrict__ g, SegTable segs, const DevScalars* __restrict__ sc,
            float b1, float b2, float eps) {
  const int64_t base = (int64_t)blockIdx.x * kSegAlign;
  const int s = find_segment(segs, base);
  const float lr = sc->lr;
  const AdamRcp rc = adam_rcp(sc->bc1, sc->bc2);
  const float wd = segs.wd[s];
  const int64_t count = segs.count[s];
  const int64_t vec_end = count - count % 8;
  for (int e = threadIdx.x; e < kSegAlign; e += 256) {
    const int64_t local = base - segs.off[s] + e;
    if (local >= count) continue;
    const int64_t k = base + e;
    adam_elem(w + k, m + k, v + k, g[k], local >= vec_end, lr, rc, b1, b2, eps, wd);
  }
}

// Adagrad over a flat segmented buffer (mlp_train_rust_codegen.rs:967-985).
__global__ void __launch_bounds__(256)
adagrad_kernel(float* __restrict__ w, float* __restrict__ G, const float* __restrict__ g,
               SegTable segs, const DevScalars* __restrict__ sc, float eps) {
  const int64_t base = (int64_t)blockIdx.x * kSegAlign;
  const int s = find_segment(segs, base);
  const float lr = sc->lr;
  const int64_t count = segs.count[s];
  for (int e = threadIdx.x; e < kSegAlign; e += 256) {
    const int64_t local = base - segs.off[s] + e;
    if (local >= count) continue;
    const int64_t k = base + e;
    adagrad_elem(w + k, G + k, g[k], lr, eps);
  }
}

// ---------------------------------------------------------------------------
// Elements a block of the MSE head takes: four per thread, and more once that
// is over kLossMaxBlocks blocks.
static int mse_per_block(int64_t nt) {
  const int64_t per = std::max<int64_t>(4 * kLossThreads, (nt + kLossMaxBlocks - 1) / kLossMaxBlocks);
  return (int)((per + kLossThreads - 1) / kLossThreads * kLossThreads);
}
// Rows a wave of the CE head takes in turn: one, until that is over
// kLossMaxBlocks blocks.
static int ce_rows_per_wave(int B) {
  return std::max(1, (B + kLossMaxBlocks * kLossWaves - 1) / (kLossMaxBlocks * kLossWaves));
}

int loss_head_blocks(int loss, int B, int C) {
  if (loss == VOLTA_LOSS_MSE) {
    const int per = mse_per_block((int64_t)B * C);
    return (int)(((int64_t)B * C + per - 1) / per);
  }
  const int rows = kLossWaves * ce_rows_per_wave(B);
  return (B + rows - 1) / rows;
}

hipError_t launch_loss_mse(const float* yhat, const float* y, float* delta, int B, int C, const LossHead& h,
                           hipStream_t st) {
  const int blocks = loss_head_blocks(VOLTA_LOSS_MSE, B, C);
  if (blocks > 1 && (!h.partials || !h.counter)) return hipErrorInvalidValue;
  hipLaunchKernelGGL(loss_mse_kernel, dim3(blocks), dim3(kLossThreads), 0, st, yhat, y, delta, B * C,
                     mse_per_block((int64_t)B * C), h);
  return hipGetLastError();
}

hipError_t launch_loss_ce(const float* z, const int32_t* labels, float* delta, int B, int C, const LossHead& h,
                          hipStream_t st) {
  const int blocks = loss_head_blocks(VOLTA_LOSS_SOFTMAX_CE, B, C), rows = ce_rows_per_wave(B);
  if (blocks > 1 && (!h.partials || !h.counter)) return hipErrorInvalidValue;
  const dim3 grid(blocks), block(kLossThreads);
  if (C <= 64) hipLaunchKernelGGL(loss_ce_kernel<1>, grid, block, 0, st, z, labels, delta, B, C, rows, h);
  else if (C <= 128) hipLaunchKernelGGL(loss_ce_kernel<2>, grid, block, 0, st, z, labels, delta, B, C, rows, h);
  else if (C <= 256) hipLaunchKernelGGL(loss_ce_kernel<4>, grid, block, 0, st, z, labels, delta, B, C, rows, h);
  else if (C <= 1024) hipLaunchKernelGGL(loss_ce_kernel<16>, grid, block, 0, st, z, labels, delta, B, C, rows, h);
  else hipLaunchKernelGGL(loss_ce_kernel<0>, grid, block, 0, st, z, labels, delta, B, C, rows, h);
  return hipGetLastError();
}

hipError_t launch_input_copy(const InputCopy& c, hipStream_t st) {
  if (!c.nx && !c.ny) return hipSuccess;
  if ((c.nx && (!c.x || !c.x_dst)) || (c.ny && (!c.y || !c.y_dst)) || (c.done && !c.ticket))
    return hipErrorInvalidValue;
  // four words per thread; from a megaword on 16, over at most 2048 blocks
  const bool big = c.nx + c.ny > ((size_t)1 << 20);
  const size_t per = big ? 256 * 16 : 256 * 4;
  auto blocks = [&](size_t n) { return (int)std::min<size_t>((n + per - 1) / per, 2048); };
  const int xb = blocks(c.nx), yb = blocks(c.ny);
  if (big) hipLaunchKernelGGL(input_copy_kernel<4>, dim3(xb + yb), dim3(256), 0, st, c, xb);
  else hipLaunchKernelGGL(input_copy_kernel<1>, dim3(xb + yb), dim3(256), 0, st, c, xb);
  return hipGetLastError();
}

hipError_t launch_adam(float* w, float* m, float* v, const float* g, const SegTable& segs,
                       int64_t total, const DevScalars* sc, float b1, float b2, float eps,
                       hipStream_t st) {
  const int blocks = (int)(total / kSegAlign);
  hipLaunchKernelGGL(adam_kernel, dim3(blocks), dim3(256), 0, st, w, m, v, g, segs, sc, b1, b2, eps);
  return hipGetLastError();
}

hipError_t launch_adagrad(float* w, float* G, const float* g, const SegTable& segs, int64_t total,
                          const DevScalars* sc, float eps, hipStream_t st) {
  const int blocks = (int)(total / kSegAlign);
  hipLaunchKernelGGL(adagrad_kernel, dim3(blocks), dim3(256), 0, st, w, G, g, segs, sc, eps);
  return hipGetLastError();
}

}  // namespace volta
