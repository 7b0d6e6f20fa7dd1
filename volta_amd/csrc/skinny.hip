// Kernels for the narrow output layer (the regression head of width 1, or a
// classifier head of up to 64 columns), whose products are too thin for 64-wide
// MFMA tiles:
//
//   out_strip_kernel     z = act_{n-1} W + b on 16-row MFMA strips, the loss
//                        head, delta_{n-1} and (up to 16 columns) dX_{n-1}
//   out_layer_dx_kernel  the same for one column and a small batch, as wave
//                        dot products (out_layer_kernel: without dX)
//   outer_dx_kernel      delta_{n-2} = (delta_{n-1} W^T) * f'   (K = L[n])
//   narrow_dw_kernel     one column: dW = act^T delta, db, optimizer update
//
// Every sum has a fixed order: MFMA k groups and pairwise trees (out_strip),
// per-lane k-strided partials then a fixed butterfly (out_layer), a
// sequential loop in the reference's order (outer_dx over k), or interleaved
// accumulators over the batch added pairwise (narrow_dw).
#include "skinny.h"

#include "narrow_dw.h"
#include "out_head.h"

namespace volta {

// The one-column output layer of a small batch in one block: wave w takes
// every (waves)-th row, four at a time (in increasing row order), the loss is
// the waves' row sums in wave order.  Lane 0 loads the bias, the targets or
// labels of its rows and the next step counter before the dot products.
__global__ void __launch_bounds__(1024) out_layer_kernel(OutLayerArgs p) {
  // rows per group and k per lane per chunk, sized to stay within the 128
  // registers a 1024-thread block allows
  constexpr int RG = 4, C = 4;
  __shared__ float wave_loss[16];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int waves = blockDim.x >> 6;
  StepNext next{};
  if (threadIdx.x == 0) next = step_prefetch(p.scalars, p.bc_table, p.bc_len);
  const float bias = p.bias[0];
  const bool mse = p.loss == VOLTA_LOSS_MSE;
  float wl = 0.0f;
  for (int m0 = wave; m0 < p.B; m0 += waves * RG) {
    int rows[RG], lab[RG];
    float y[RG][1], z[RG][1];
#pragma unroll
    for (int g = 0; g < RG; ++g) {
      const int m = m0 + g * waves, mc = min(m, p.B - 1);
      rows[g] = m < p.B ? m : -1;
      y[g][0] = mse ? p.y[mc] : 0.0f;
      lab[g] = mse ? 0 : p.labels[mc];
    }
    wave_rows<RG, C>(p, rows, z);
    if (lane == 0) {
#pragma unroll
      for (int g = 0; g < RG; ++g) {
        if (rows[g] < 0) continue;
        z[g][0] = z[g][0] + bias;
        wl = wl + head_row(p, z[g], y[g], lab[g], rows[g]);
      }
    }
  }
  if (lane == 0) wave_loss[wave] = wl;
  __syncthreads();
  if (threadIdx.x == 0) {
    float s = wave_loss[0];
    for (int w = 1; w < waves; ++w) s = s + wave_loss[w];
    step_finish(p.scalars, next, p.bc_table != nullptr, s / out_dx_loss_denom(p));
  }
}

// The one-column output layer, its loss head and its dX in one launch (B <=
// kNarrowMaxB).  Wave w of block b owns batch row m = 4b + w:
//   z = act_{n-1}[m] W + bias     (wave_rows: lane k-strided, fixed butterfly)
//   delta_{n-1}[m] and the row loss (head_delta, identical in every lane;
//                                     lane 0 stores z and the delta)
//   delta_{n-2}[m][k] = delta_{n-1}[m] W[k] * f'(pre, act)
//                                    for the lane's k = lane + 64c
// Everything but the loss is row-local.  The block's row losses are added in
// row order into partials[b].  With defer_loss (the small-batch step, whose
// grouped dW launch adds the partials later) block 0 only advances the Adam
// step counter; otherwise the last block to finish (integer ticket, an
// agent-scope release and acquire) adds the partials in block order and
// records the step's loss, the non-finite flag and the step counter.  A
// separate one-block output launch plus the outer-product dX launch cost
// more: one CU for 64 rows, and a dependent launch between them.
__global__ void __launch_bounds__(kOutDxRows * 64) out_layer_dx_kernel(OutLayerArgs p) {
  __shared__ float wave_loss[kOutDxRows];
  __shared__ unsigned last_block;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  // the next step counter and its bias corrections, in case this block
  // finishes last (nothing else in the launch writes them); with the loss
  // deferred, block 0 alone reads and advances the counter
  StepNext next{};
  if (threadIdx.x == 0 && (!p.defer_loss || blockIdx.x == 0)) next = step_prefetch(p.scalars, p.bc_table, p.bc_len);
  const float row_loss = out_dx_row(p, blockIdx.x * kOutDxRows + wave);
  if (lane == 0) wave_loss[wave] = row_loss;
  __syncthreads();
  if (threadIdx.x == 0) {
    float sb = wave_loss[0];
    for (int w = 1; w < kOutDxRows; ++w) sb = sb + wave_loss[w];
    p.partials[blockIdx.x] = sb;
    if (p.defer_loss) {
      // a later launch of the step adds the partials (deferred_loss_finish):
      // no agent-scope fence or ticket here
      if (blockIdx.x == 0 && p.bc_table) {
        p.scalars->t = next.t;
        p.scalars->bc1 = next.bc.x;
        p.scalars->bc2 = next.bc.y;
      }
      return;
    }
    __threadfence();
    last_block = atomicAdd(p.loss_counter, 1u) == gridDim.x - 1 ? 1u : 0u;
    if (last_block) {
      __threadfence();
      out_dx_finish(p, (int)gridDim.x, next);
    }
  }
}

// ---------------------------------------------------------------------------
// The output layer of up to 64 columns, its loss head and, for up to 16
// columns, its dX_{n-1}, on 16-row strips of the batch: one workgroup of 16
// waves per strip.
//   z      CT column tiles of v_mfma_f32_16x16x4f32, the K range of each split
//          over 16 / CT waves (the small-M tile's k order), the waves'
//          partial tiles added as a pairwise tree; + bias, into LDS
//   head   one wave per row, one lane per column: row maximum, exp sum or
//          squared error by butterflies; delta_{n-1} and the row's loss
//   dX     (DX) delta_{n-2}[m][k] = (sum_j delta_{n-1}[m][j] W[k][j]) * f',
//          j ascending (outer_dx_kernel's arithmetic), four rows per thread
//          With few strips several workgroups share one: each forms its z and
//          deltas and takes a part of dX's columns, the first stores the rest.
//   loss   the strip's rows in order, the strips' sums by the strip that
//          finishes last, or by a later launch (defer_loss)
// Latency bound up to a few hundred rows (one load round, the head's
// butterflies, one load round for dX); beyond that by the strips' reads of
// act_{n-1}.  Wave-wide dot products, one row per wave with every column's
// butterfly in turn and the head repeated in each lane, took 20.8 us for 16
// rows of 1088 x 10 and 1.8 ms where W (3392 x 10) did not fit in LDS and one
// block ran all rows; a 64-wide GEMM tile with one thread per row of the loss
// head took 18 us for 629 rows of 200 x 17.
constexpr int kStripRed = 80;  // LDS floats per (wave, register) row of partial tiles

// DXN: dX columns of W a thread holds (4 or 16; at least N), or 0 without dX.
template <int CT, bool VEC, int DXN>
__global__ void __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(4))) out_strip_kernel(OutLayerArgs p) {
  constexpr bool DX = DXN > 0;
  constexpr int NJ = DX ? DXN : 1;
  constexpr int KW = 16 / CT;       // waves per column tile
  constexpr int NC = 16 * CT;       // columns in LDS
  constexpr int CH = 4;             // 16-k groups per load round
  constexpr int ZS = NC + 1;
  __shared__ float red[16 * 4 * kStripRed];
  __shared__ float zrow[16 * ZS];   // z, then delta_{n-1}
  __shared__ float row_loss[16];
  __shared__ unsigned last;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, q = lane >> 4;
  const int B = p.B, K = p.K, N = p.N, m0 = blockIdx.x * 16;
  const bool writer = !DX || blockIdx.y == 0;  // stores z, delta_{n-1} and the loss of its strip
  StepNext next{};
  if (tid == 0 && writer && (!p.defer_loss || blockIdx.x == 0)) next = step_prefetch(p.scalars, p.bc_table, p.bc_len);
  const bool mse = p.loss == VOLTA_LOSS_MSE;
  // the head's operands of row m0 + wave, column `lane`
  const int hm = min(m0 + wave, B - 1), hc = min(lane, N - 1);
  const float y = mse ? p.y[(size_t)hm * N + hc] : 0.0f;
  const int lab = mse ? 0 : p.labels[hm];
  const int rows = min(16, B - m0);
  const int ct = wave % CT, kw = wave / CT;
  const int kq = (K + KW * 16 - 1) / (KW * 16) * 16;
  const int kbeg = kw * kq, kend = min(K, kbeg + kq);
  const int col = ct * 16 + r;
  const bool row_ok = m0 + r < B, col_ok = col < N;
  const float* pa = p.act + (size_t)(row_ok ? m0 + r : 0) * K;
  const float* pb = p.W + (col_ok ? col : 0);
  floatx4 acc[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) acc[c] = floatx4{0.f, 0.f, 0.f, 0.f};
  for (int kc = kbeg; kc < kend; kc += 16 * CH) {
    floatx4 fa[CH], fb[CH];
#pragma unroll
    for (int g = 0; g < CH; ++g) {
      if (kc + 16 * g >= kend) break;  // wave-uniform
      const int k = kc + 16 * g + 4 * q;
      if constexpr (VEC) {  // K % 4 == 0: every range bound is a multiple of 4
        const int kl = min(k, kend - 4);
        fa[g] = *reinterpret_cast<const floatx4*>(pa + kl);
#pragma unroll
        for (int s = 0; s < 4; ++s) fb[g][s] = pb[(size_t)(kl + s) * N];
      } else {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const int kl = min(k + s, kend - 1);
          fa[g][s] = pa[kl];
          fb[g][s] = pb[(size_t)kl * N];
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int g = 0; g < CH; ++g) {
      if (kc + 16 * g < kend) {
        const int k = kc + 16 * g + 4 * q;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const bool in = VEC ? k < kend : k + s < kend;
          acc[g] = __builtin_amdgcn_mfma_f32_16x16x4f32(in && row_ok ? fa[g][s] : 0.0f, in && col_ok ? fb[g][s] : 0.0f,
                                                        acc[g], 0, 0, 0);
        }
      }
    }
  }
#pragma unroll
  for (int v = 0; v < 4; ++v)
    red[(wave * 4 + v) * kStripRed + lane] = (acc[0][v] + acc[1][v]) + (acc[2][v] + acc[3][v]);
  __syncthreads();
  // element (i, j) of column tile t: lane 16*(i/4) + j, register i%4 of each of its waves
  if (tid < 256 * CT) {
    const int t = tid >> 8, i = (tid >> 4) & 15, j = tid & 15;
    const int src = (i & 3) * kStripRed + 16 * (i >> 2) + j;
    float v[KW];
#pragma unroll
    for (int w = 0; w < KW; ++w) v[w] = red[(w * CT + t) * 4 * kStripRed + src];
#pragma unroll
    for (int h = 1; h < KW; h *= 2)
#pragma unroll
      for (int w = 0; w < KW; w += 2 * h) v[w] = v[w] + v[w + h];
    const int n = t * 16 + j;
    zrow[i * ZS + n] = v[0] + p.bias[min(n, N - 1)];  // z = act_{n-1} W + b (:792-798)
  }
  __syncthreads();
  {  // the loss head of row m0 + wave
    const int m = m0 + wave;
    const bool in = lane < N;
    const float z = zrow[wave * ZS + hc];
    float d, loss;
    if (mse) {
      const float nt = (float)(B * N);
      const float dj = z - y;
      d = 2.0f * dj / nt;
      loss = wave_sum(in ? dj * dj : 0.0f);
    } else {
      float mx = in ? z : -INFINITY;
#pragma unroll
      for (int off = 32; off >= 1; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, kWave));
      const float e = expf(z - mx);
      const float sum = wave_sum(in ? e : 0.0f);
      d = (e / sum - (lane == lab ? 1.0f : 0.0f)) / (float)B;
      const bool ok = lab >= 0 && lab < N;
      const float zl = __shfl(z, ok ? lab : 0, kWave);
      loss = ok ? -(zl - (mx + logf(sum))) : __builtin_nanf("");
      if (!ok && m < B && lane == 0 && writer) atomicOr(&p.scalars->flags, (uint32_t)VOLTA_STATUS_BAD_ARGUMENT);
    }
    if (in) zrow[wave * ZS + lane] = d;  // (this wave's row only)
    if (in && m < B && writer) {
      p.out[(size_t)m * N + lane] = z;
      p.delta[(size_t)m * N + lane] = d;
    }
    if (lane == 0) row_loss[wave] = loss;
  }
  __syncthreads();
  if (tid == 0) {
    float s = row_loss[0];
    for (int w = 1; w < rows; ++w) s = s + row_loss[w];
    last = 0u;
    if (!writer) {
    } else if (p.defer_loss) {
      // a later launch of the step adds the partials
      p.partials[blockIdx.x] = s;
      if (blockIdx.x == 0 && p.bc_table) {
        p.scalars->t = next.t;
        p.scalars->bc1 = next.bc.x;
        p.scalars->bc2 = next.bc.y;
      }
    } else if (gridDim.x == 1) {
      row_loss[0] = s;
      last = 1u;
    } else {
      last = publish_partial(p.partials, p.loss_counter, blockIdx.x, gridDim.x, s) ? 1u : 0u;
    }
  }
  if constexpr (DX) {
    // four of the strip's rows per thread: column idx % K, rows 4 * (idx / K)
    // ..; workgroup y of the strip's gridDim.y takes every gridDim.y-th 1024
    const float* pre = p.dx_pre ? p.dx_pre : p.act;
    const int items = (rows + 3) / 4 * K;
    for (int idx = tid + 1024 * blockIdx.y; idx < items; idx += 1024 * gridDim.y) {
      const int g = idx / K, k = idx - g * K;
      float w[NJ], av[4], pv[4];
#pragma unroll
      for (int j = 0; j < NJ; ++j) w[j] = p.W[(size_t)k * N + min(j, N - 1)];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const size_t o = (size_t)min(m0 + 4 * g + i, B - 1) * K + k;
        av[i] = p.act[o];
        pv[i] = pre[o];
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float s = 0.0f;
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          const float u = s + zrow[(4 * g + i) * ZS + min(j, N - 1)] * w[j];
          s = j < N ? u : s;
        }
        if (m0 + 4 * g + i < B)
          p.dx_out[(size_t)(m0 + 4 * g + i) * K + k] = s * act_derivative(p.dx_act, pv[i], av[i]);
      }
    }
  }
  __syncthreads();
  if (!last || wave != 0) return;
  float s = row_loss[0];
  if (gridDim.x > 1) {
    const int strips = (int)gridDim.x;
    s = 0.0f;
    for (int b = lane; b < strips; b += 64) s = s + published_partial(p.partials, b);
    if (strips <= 16) {  // in strip order, as the dW group's deferred sum
      float t = __shfl(s, 0, kWave);
      for (int b = 1; b < strips; ++b) t = t + __shfl(s, b, kWave);
      s = t;
    } else {
      s = wave_sum(s);
    }
  }
  if (lane == 0) {
    step_finish(p.scalars, next, p.bc_table != nullptr, s / (mse ? (float)(B * N) : (float)B));
    if (gridDim.x > 1) *p.loss_counter = 0u;  // for the next step's launch
  }
}

int out_strip_blocks(int B) { return (B + 15) / 16; }

template <int CT, int DX>
static void launch_strip_t(const OutLayerArgs& p, hipStream_t st) {
  const bool vec = p.K % 4 == 0 && ((uintptr_t)p.act & 15) == 0;
  // dX: up to 8 workgroups a strip, until every thread has one group of rows
  // or the launch has a workgroup for each of 256 CUs
  const int strips = out_strip_blocks(p.B), groups = (std::min(p.B, 16) + 3) / 4;
  const int per = DX ? std::max(1, std::min({8, (groups * p.K + 1023) / 1024, 256 / strips})) : 1;
  const dim3 grid(strips, per), block(1024);
  if (vec) hipLaunchKernelGGL((out_strip_kernel<CT, true, DX>), grid, block, 0, st, p);
  else hipLaunchKernelGGL((out_strip_kernel<CT, false, DX>), grid, block, 0, st, p);
}

hipError_t launch_out_strip(const OutLayerArgs& p, bool dx, hipStream_t st) {
  const bool ok = p.B >= 1 && p.K >= 1 && p.N >= 1 && p.N <= kOutStripMaxN && p.act && p.W && p.bias && p.out &&
                  p.delta && p.scalars && p.partials && (p.loss_counter || p.defer_loss) &&
                  (p.loss == VOLTA_LOSS_MSE ? p.y != nullptr : p.labels != nullptr) &&
                  (!dx || (p.N <= 16 && p.dx_out));
  if (!ok) return hipErrorInvalidValue;
  if (p.N <= 16) {
    if (!dx) launch_strip_t<1, 0>(p, st);
    else if (p.N <= 4) launch_strip_t<1, 4>(p, st);
    else launch_strip_t<1, 16>(p, st);
  } else if (p.N <= 32) {
    launch_strip_t<2, 0>(p, st);
  } else {
    launch_strip_t<4, 0>(p, st);
  }
  return hipGetLastError();
}

int out_layer_dx_blocks(int B) { return (B + kOutDxRows - 1) / kOutDxRows; }

bool out_layer_dx_supported(int B, int K, int N) { return B >= 1 && B <= kNarrowMaxB && K >= 1 && N == 1; }

hipError_t launch_out_layer_dx(const OutLayerArgs& p, hipStream_t st) {
  if (!out_layer_dx_supported(p.B, p.K, p.N) || !p.partials || (!p.loss_counter && !p.defer_loss) || !p.dx_out)
    return hipErrorInvalidValue;
  hipLaunchKernelGGL(out_layer_dx_kernel, dim3(out_layer_dx_blocks(p.B)), dim3(kOutDxRows * 64), 0, st, p);
  return hipGetLastError();
}

// delta_out[b][j] = (sum_{k<K} delta[b][k] * W[j][k]) * f'(layer below)[b][j]
// for K <= KMAX <= 16 (reference order: k ascending, :919-929).  Thread j of
// a block keeps row j of W in registers for the block's RB batch rows, whose
// deltas are staged in LDS; its loads (W row, then the activation operands
// of all RB rows) are unconditional (clamped indices) and issued together.
// RB = 16 on large layers (the W row is loaded once per 16 outputs), 1 on
// small ones (more blocks).
template <int KMAX, int RB>
__global__ void __launch_bounds__(256)
outer_dx_kernel(const float* __restrict__ delta, const float* __restrict__ W, int B, int R, int K, int act,
                const float* __restrict__ aux_act, const float* __restrict__ aux_pre, float* __restrict__ out,
                LossDefer ld) {
  static_assert(RB * KMAX <= 256, "one staged delta per thread");
  __shared__ float sd[RB * KMAX];
  const int t = threadIdx.x;
  const int j = blockIdx.x * 256 + t, jc = min(j, R - 1);
  const int b0 = blockIdx.y * RB;
  const float dv = delta[(size_t)min(b0 + t / KMAX, B - 1) * K + min(t % KMAX, K - 1)];
  float wv[KMAX];
#pragma unroll
  for (int k = 0; k < KMAX; ++k) wv[k] = W[(size_t)jc * K + min(k, K - 1)];
  const float* pp = aux_pre ? aux_pre : aux_act;
  // block (0, 0) also forms the step's loss (below): its first 256 partials
  // are loaded now, so their latency runs under the block's products
  const bool loss_block = ld.partials && blockIdx.x == 0 && blockIdx.y == 0;  // block-uniform
  const float p0 = loss_block ? ld.partials[min(t, ld.blocks - 1)] : 0.0f;
  float y[RB], pr[RB];
  if (aux_pre) {  // uniform: f' from the kept pre-activation
#pragma unroll
    for (int r = 0; r < RB; ++r) {
      const size_t o = (size_t)min(b0 + r, B - 1) * R + jc;
      y[r] = aux_act[o];
      pr[r] = pp[o];
    }
  } else {  // f' from the output: one load per element
#pragma unroll
    for (int r = 0; r < RB; ++r) {
      y[r] = aux_act[(size_t)min(b0 + r, B - 1) * R + jc];
      pr[r] = y[r];
    }
  }
  if (t < RB * KMAX) sd[t] = dv;
  __syncthreads();
#pragma unroll
  for (int r = 0; r < RB; ++r) {
    float s = 0.0f;
#pragma unroll
    for (int k = 0; k < KMAX; ++k) {
      const float u = s + sd[r * KMAX + k] * wv[k];
      s = k < K ? u : s;
    }
    if (j < R && b0 + r < B) out[(size_t)(b0 + r) * R + j] = s * act_derivative(act, pr[r], y[r]);
  }
  if (loss_block) deferred_loss_tree(ld, p0, t);  // the step's loss
}

// Stand-alone launch: 64 rows of W per block.
__global__ void __launch_bounds__(kNarrowThreads) narrow_dw_kernel(NarrowDwArgs p) {
  extern __shared__ float lds[];
  narrow_dw_block(p, blockIdx.x, lds);
}

// ---------------------------------------------------------------------------
hipError_t launch_out_layer(const OutLayerArgs& p, hipStream_t st) {
  if (p.N != 1 || p.B < 1 || p.B > kNarrowMaxB) return hipErrorInvalidValue;
  hipLaunchKernelGGL(out_layer_kernel, dim3(1), dim3(1024), 0, st, p);
  return hipGetLastError();
}

template <int KMAX>
static void launch_outer_k(bool big, dim3 blocks, hipStream_t st, const float* delta, const float* W, int B, int R,
                           int K, int act, const float* aux_act, const float* aux_pre, float* out,
                           const LossDefer& ld) {
  if (big)
    hipLaunchKernelGGL((outer_dx_kernel<KMAX, 16>), blocks, dim3(256), 0, st, delta, W, B, R, K, act, aux_act,
                       aux_pre, out, ld);
  else
    hipLaunchKernelGGL((outer_dx_kernel<KMAX, 1>), blocks, dim3(256), 0, st, delta, W, B, R, K, act, aux_act,
                       aux_pre, out, ld);
}

hipError_t launch_outer_dx(const float* delta, const float* W, int B, int R, int K, int act, const float* aux_act,
                           const float* aux_pre, float* out, hipStream_t st, const LossDefer& ld) {
  if (K > 16 || K < 1) return hipErrorInvalidValue;
  if (ld.partials && (ld.blocks < 1 || !ld.scalars)) return hipErrorInvalidValue;
  // 16 batch rows per block once the layer has a million outputs
  const bool big = (size_t)B * R >= ((size_t)1 << 20);
  const dim3 blocks((R + 255) / 256, (B + (big ? 16 : 1) - 1) / (big ? 16 : 1));
  if (K <= 1) launch_outer_k<1>(big, blocks, st, delta, W, B, R, K, act, aux_act, aux_pre, out, ld);
  else if (K <= 4) launch_outer_k<4>(big, blocks, st, delta, W, B, R, K, act, aux_act, aux_pre, out, ld);
  else launch_outer_k<16>(big, blocks, st, delta, W, B, R, K, act, aux_act, aux_pre, out, ld);
  return hipGetLastError();
}

hipError_t launch_narrow_dw(const NarrowDwArgs& p, hipStream_t st) {
  if (p.N != 1 || p.B < 1 || p.B > kNarrowMaxB) return hipErrorInvalidValue;
  if (p.opt != VOLTA_OPT_SGD && p.opt != VOLTA_OPT_ADAM && p.opt != VOLTA_OPT_ADAGRAD) return hipErrorInvalidValue;
  const int blocks = (p.R + kNarrowRows - 1) / kNarrowRows;
  hipLaunchKernelGGL(narrow_dw_kernel, dim3(blocks), dim3(kNarrowThreads), narrow_lds_floats(p.B) * 4, st, p);
  return hipGetLastError();
}

}  // namespace volta
