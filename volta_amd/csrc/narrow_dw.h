// Device code of the one-column output layer's dW (also run beside a GEMM in
// one launch by gemm.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "device_common.h"
#include "skinny.h"

namespace volta {

// Rows of W a block of kNarrowThreads threads updates.
constexpr int kNarrowThreads = 256;
constexpr int kNarrowRows = 64;
static_assert(kNarrowMaxB <= kNarrowThreads, "each thread stages at most one delta");

// Floats of LDS a block uses: the B deltas (padded to 4), then the waves'
// partial sums.
__host__ __device__ inline int narrow_lds_floats(int B) { return (B + 3) / 4 * 4 + kNarrowThreads; }

// dW[j] = sum_b act[b][j] * delta[b] for the kNarrowRows rows j of W of this
// block: lane l of wave q takes row j = block*64 + l and, of every 64 batch
// rows, the 16 rows 16q..16q+15 (ascending; all chunks into one partial), and
// the four waves' partials are added as (P0 + P1) + (P2 + P3) by wave 0, which
// runs the optimizer on W.  Block 0 also forms db = sum_b delta[b] (:931-933)
// over four interleaved accumulators (b mod 4) added pairwise.  Latency: every
// global load is unconditional (clamped addresses; values outside the batch
// are never used); the delta's load goes first, so staging waits for it alone,
// then the activations (16 a thread for each of up to four 64-row chunks a
// round) and wave 0's optimizer state; the staged deltas are read from LDS in
// batches before the multiplies, and guards are selects.
// kU (64-row chunks whose loads one round issues together), kDbChunk (the
// bias's reads issued before their adds) and the batch of staged deltas read
// before the multiplies trade registers for memory latency: the stand-alone
// launches keep the widest settings; the grouped dW launch, whose small-K
// tiles share its register budget, takes the narrow ones (LEAN).
template <bool LEAN = false>
__device__ __forceinline__ void narrow_dw_block(const NarrowDwArgs& p, int block, float* lds) {
  constexpr int kQ = 16;  // batch rows per wave per 64-row chunk
  constexpr int kU = LEAN ? 1 : 4;         // 64-row chunks whose loads one round issues together
  constexpr int kDBatch = LEAN ? 8 : 16;   // batch rows per LDS read batch
  const int B = p.B, R = p.R;
  const int tid = threadIdx.x, lane = tid & 63, q = tid >> 6;
  const int j = block * kNarrowRows + lane;
  const bool own = j < R;
  const int jc = own ? j : 0;
  const bool sgd = p.opt == VOLTA_OPT_SGD, adam = p.opt == VOLTA_OPT_ADAM;
  float* sdelta = lds;
  float* part = lds + (B + 3) / 4 * 4;  // part[q*64 + lane]
  const float dst = p.delta[min(tid, B - 1)];
  // activations of a round: chunk u holds batch rows b0 + 64u + 16q + c
  float a[kU][kQ];
  auto load_round = [&](int b0) {
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      if (b0 + 64 * u >= B) break;  // wave-uniform
#pragma unroll
      for (int c = 0; c < kQ; ++c) a[u][c] = p.act[(size_t)min(b0 + 64 * u + kQ * q + c, B - 1) * R + jc];
    }
  };
  load_round(0);
  float w = p.w[jc];
  float s1 = (sgd ? p.w : p.m)[jc];
  float s2 = (adam ? p.v : p.w)[jc];
  // bias state (no bias work when p.b is null)
  const float* pb = p.b ? p.b : p.w;
  const float bw = pb[0];
  const float bs1 = (sgd || !p.b ? pb : p.bm)[0];
  const float bs2 = (adam && p.b ? p.bv : pb)[0];
  const float lr = p.scalars->lr;
  const AdamRcp rc = adam_rcp(p.scalars->bc1, p.scalars->bc2);
  if (tid < B) sdelta[tid] = dst;
  __syncthreads();

  float acc = 0.0f;
  for (int r0 = 0; r0 < B; r0 += 64 * kU) {
    if (r0 > 0) load_round(r0);
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int b0 = r0 + 64 * u;
      if (b0 >= B) break;  // wave-uniform
#pragma unroll
      for (int c0 = 0; c0 < kQ; c0 += kDBatch) {
        float d[kDBatch];
#pragma unroll
        for (int c = 0; c < kDBatch; ++c) d[c] = sdelta[min(b0 + kQ * q + c0 + c, B - 1)];
#pragma unroll
        for (int c = 0; c < kDBatch; ++c) {
          const float t = acc + a[u][c0 + c] * d[c];
          acc = b0 + kQ * q + c0 + c < B ? t : acc;
        }
      }
    }
  }
  part[q * 64 + lane] = acc;
  __syncthreads();
  if (q != 0) return;
  acc = (part[lane] + part[64 + lane]) + (part[128 + lane] + part[192 + lane]);
  if (own) {
    if (sgd) {
      const float nlr = -lr;
      w = w + nlr * acc;
    } else if (p.opt == VOLTA_OPT_ADAGRAD) {
      adagrad_elem(&w, &s1, acc, lr, p.eps);
    } else {
      adam_elem(&w, &s1, &s2, acc, j >= R - R % 8, lr, rc, p.b1, p.b2, p.eps, p.wd);
    }
    if (p.grad) p.grad[j] = acc;
    p.w[j] = w;
    if (!sgd) p.m[j] = s1;
    if (adam) p.v[j] = s2;
  }
  if (block == 0 && tid == 0 && p.b) {
    // four interleaved accumulators; each chunk's reads are issued before
    // its first add
    constexpr int kDbChunk = LEAN ? 16 : 64;
    float dba[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int b0 = 0; b0 < B; b0 += kDbChunk) {
      float d[kDbChunk];
#pragma unroll
      for (int c = 0; c < kDbChunk; ++c) d[c] = sdelta[min(b0 + c, B - 1)];
#pragma unroll
      for (int c = 0; c < kDbChunk; ++c) {
        const float t = dba[c & 3] + d[c];
        dba[c & 3] = b0 + c < B ? t : dba[c & 3];
      }
    }
    const float db = (dba[0] + dba[1]) + (dba[2] + dba[3]);
    if (p.bgrad) p.bgrad[0] = db;
    float x = bw, y1 = bs1, y2 = bs2;
    if (sgd) {
      x = x - lr * db;
    } else if (p.opt == VOLTA_OPT_ADAGRAD) {
      adagrad_elem(&x, &y1, db, lr, p.eps);
    } else {
      adam_elem(&x, &y1, &y2, db, true, lr, rc, p.b1, p.b2, p.eps, 0.0f);  // (one element: its own tail)
    }
    p.b[0] = x;
    if (!sgd) p.bm[0] = y1;
    if (adam) p.bv[0] = y2;
  }
}

}  // namespace volta
