// adam.h -- the Adam update of a batch of parameter tensors, shared by the
// training kernels (device code).
#pragma once

#include <hip/hip_runtime.h>

#include "mlp.h"

namespace bude {
namespace mlp {

// One Adam update of w, m and v by gradient g.  The contractions are written
// out, so that every kernel rounds the same way.
__device__ __forceinline__ void adam_update(float &w, float &m, float &v, float g, float lr, float bc1, float bc2,
                                            float b1, float b2, float eps) {
  m = __builtin_fmaf(1.f - b1, g, b1 * m);
  v = __builtin_fmaf((1.f - b2) * g, g, b2 * v);
  w -= lr * (m / bc1) / (sqrtf(v / bc2) + eps);
}

constexpr int kAdamWaves = 4;

// Entries 64 block .. 64 block + 63 of the flat index over the batch's
// tensors, by one work-group of four waves: partial sum p of the lane's entry
// is over slices p, p + P, ... (each load a coalesced row of 64 entries), the
// work-group adds the P partials in order, and the first wave applies Adam.
// Wave w forms partials w, w + 4, ...; P is 16 for the hundreds of slices of
// the learned field's step, 4 for the K splits of the GEMMs; the order of
// every sum is fixed.  hyper: the step's learning rates and bias corrections
// (schedule_hyper).
template <int P>
__device__ __forceinline__ void adam_tensors(const AdamBatch &b, int block, float b1, float b2, float eps,
                                             const float *__restrict__ hyper) {
  constexpr int kOwn = P / kAdamWaves;
  __shared__ float part[P][64];
  const float lr = hyper[0], bc1 = hyper[2], bc2 = hyper[3];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  size_t i = size_t(block) * 64 + lane;
  int t = 0;
  for (; t < b.count; t++) {
    const size_t n = size_t(b.t[t].rows) * b.t[t].cols;
    if (i < n) break;
    i -= n;
  }
  const bool valid = t < b.count;
  float gs[kOwn];
#pragma unroll
  for (int o = 0; o < kOwn; o++) gs[o] = 0.f;
  if (valid) {
    const float *g = b.t[t].g + i;
    const size_t stride = b.t[t].stride;
    const int splits = b.t[t].splits;
    // four slices of each partial in flight
    int z = wave;
    for (; z + 3 * P + (kOwn - 1) * kAdamWaves < splits; z += 4 * P) {
      float sl[4][kOwn];
#pragma unroll
      for (int u = 0; u < 4; u++)
#pragma unroll
        for (int o = 0; o < kOwn; o++) sl[u][o] = g[size_t(z + u * P + o * kAdamWaves) * stride];
#pragma unroll
      for (int u = 0; u < 4; u++)
#pragma unroll
        for (int o = 0; o < kOwn; o++) gs[o] += sl[u][o];
    }
    for (; z < splits; z += P)
#pragma unroll
      for (int o = 0; o < kOwn; o++)
        if (z + o * kAdamWaves < splits) gs[o] += g[size_t(z + o * kAdamWaves) * stride];
  }
#pragma unroll
  for (int o = 0; o < kOwn; o++) part[wave + o * kAdamWaves][lane] = gs[o];
  __syncthreads();
  if (wave != 0 || !valid) return;
  float gi = part[0][lane];
#pragma unroll
  for (int p = 1; p < P; p++) gi += part[p][lane];
  const AdamTensor &T = b.t[t];
  const size_t at = T.pitch ? i / T.cols * T.pitch + i % T.cols : i;
  float wi = T.w[at], mi = T.m[at], vi = T.v[at];
  adam_update(wi, mi, vi, gi, lr, bc1, bc2, b1, b2, eps);
  T.w[at] = wi;
  T.m[at] = mi;
  T.v[at] = vi;
  const bf16 h = __builtin_bit_cast(bf16, static_cast<__bf16>(wi));  // (round to nearest even)
  if (T.w16) T.w16[at] = h;
  if (T.w16t) T.w16t[size_t(i % T.cols) * T.rows + i / T.cols] = h;
  if (T.w16x) T.w16x[tiled_index(i / T.cols, i % T.cols, size_t(T.cols))] = h;
  if (T.w16tx) T.w16tx[tiled_index(i % T.cols, i / T.cols, size_t(T.rows))] = h;
}

// Entries of a batch's tensors.
inline size_t adam_entries(const AdamBatch &b) {
  size_t n = 0;
  for (int t = 0; t < b.count; t++) n += size_t(b.t[t].rows) * b.t[t].cols;
  return n;
}

}  // namespace mlp
}  // namespace bude
