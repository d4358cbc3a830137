// gate.hip -- validation statistics of a combined screen's pairs: one
// work-group per pair sorts its samples in LDS (bitonic, keys of value and
// index, so equal values keep their order) and reduces the sums in FP64 in a
// fixed order.  64 pairs of 1,024 samples take 40 us; the host took 5 ms,
// with the rescoring waiting for it.
#include <hip/hip_runtime.h>

#include <cmath>

#include "gate.h"

namespace bude {
namespace gate {

namespace {

constexpr int kThreads = 1024;

// float -> uint32 of the same order; equal values (both zeros) get equal keys.
__device__ __forceinline__ uint32_t order_key(float x) {
  const uint32_t u = __float_as_uint(x == 0.f ? 0.f : x);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

__device__ __forceinline__ float key_value(uint64_t k) {
  const uint32_t u = uint32_t(k >> 32);
  return __uint_as_float((u & 0x80000000u) ? (u & 0x7fffffffu) : ~u);
}

// Sorts keys[0 .. m) (m a power of two) ascending.
__device__ void sort_keys(uint64_t *keys, int m) {
  for (int size = 2; size <= m; size <<= 1)
    for (int stride = size >> 1; stride; stride >>= 1) {
      __syncthreads();
      for (int t = threadIdx.x; t < m / 2; t += kThreads) {
        const int i = 2 * t - (t & (stride - 1)), j = i + stride;
        const uint64_t a = keys[i], b = keys[j];
        if ((a > b) == ((i & size) == 0)) {
          keys[i] = b;
          keys[j] = a;
        }
      }
    }
  __syncthreads();
}

// Sum over the work-group, the same in every work-item.
__device__ double group_sum(double v, double *part) {
  for (int d = 32; d; d >>= 1) v += __shfl_xor(v, d);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
  __syncthreads();
  double s = 0;
  for (int w = 0; w < kThreads / 64; w++) s += part[w];
  return s;
}

__global__ __launch_bounds__(kThreads) void stats_kernel(const float *__restrict__ e, const float *__restrict__ p,
                                                         const uint32_t *__restrict__ off, int room, const Params q,
                                                         Stats *__restrict__ out) {
  extern __shared__ uint64_t keys[];  // room (a power of two), then a mark per sample
  __shared__ double part[kThreads / 64];
  auto *mark = reinterpret_cast<unsigned char *>(keys + room);
  const uint32_t b = off[blockIdx.x];
  const int n = int(off[blockIdx.x + 1] - b);
  const float *ee = e + b, *pp = p + b;
  if (n < 1) {
    if (threadIdx.x == 0) out[blockIdx.x] = Stats{0.0, 0.f, 0.f, 0.f, 0.f};
    return;
  }
  int m = 2;
  while (m < n) m <<= 1;
  const double dn = double(n);

  // the scores' lowest tenth, for the recall
  const int kt = max(1, int(lround(0.05 * dn))), ks = min(n, max(kt, int(lround(0.10 * dn))));
  for (int i = threadIdx.x; i < m; i += kThreads)
    keys[i] = i < n ? uint64_t(order_key(pp[i])) << 32 | uint32_t(i) : ~uint64_t(0);
  sort_keys(keys, m);
  for (int i = threadIdx.x; i < n; i += kThreads) mark[uint32_t(keys[i])] = i < ks;
  __syncthreads();
  for (int i = threadIdx.x; i < m; i += kThreads)
    keys[i] = i < n ? uint64_t(order_key(ee[i])) << 32 | uint32_t(i) : ~uint64_t(0);
  sort_keys(keys, m);

  auto quantile = [&](double f) {
    const double x = fmin(1.0, fmax(0.0, f)) * double(n - 1);
    const int i = int(x);
    const double t = x - double(i);
    return i + 1 < n ? double(key_value(keys[i])) * (1 - t) + double(key_value(keys[i + 1])) * t
                     : double(key_value(keys[n - 1]));
  };
  const double q_top = quantile(q.top), gap = quantile(q.keep) - q_top;
  // line of score on energy over the lowest samples, and its residual
  const int nt = min(n, max(8, int(ceil(q.tail_q * dn))));
  double s[6] = {0, 0, 0, 0, 0, 0};
  for (int i = threadIdx.x; i < nt; i += kThreads) {
    const double x = key_value(keys[i]), y = pp[uint32_t(keys[i])];
    s[0] += x;
    s[1] += y;
    s[2] += x * x;
    s[3] += x * y;
    s[4] += y * y;
  }
  for (int k = 0; k < 5; k++) s[k] = group_sum(s[k], part) / double(nt);
  const double ve = s[2] - s[0] * s[0], vp = s[4] - s[1] * s[1], cv = s[3] - s[0] * s[1];
  const double a = ve > 0 ? cv / ve : 0.0;
  const double sd = a > 0 ? sqrt(fmax(0.0, vp - a * cv)) / a : INFINITY;
  Stats r{};
  r.z = sd > 0 ? float(gap / sd) : (gap > 0 ? INFINITY : 0.f);
  const double thr = q_top + q.z_req * sd;
  double below = 0, hits = 0;
  for (int i = threadIdx.x; i < n; i += kThreads) below += double(key_value(keys[i])) <= thr;
  for (int i = threadIdx.x; i < kt; i += kThreads) hits += mark[uint32_t(keys[i])];
  below = group_sum(below, part);
  hits = group_sum(hits, part);
  r.need = isfinite(sd) ? below / dn : INFINITY;
  r.recall = float(hits / double(kt));
  if (n < 2) {
    r.z = r.recall = 0.f;
    r.need = INFINITY;
  }

  // clipped, standardised targets and scores
  const float clip = key_value(keys[min(n - 1, int(q.clip_q * dn))]);
  double s1 = 0, s2 = 0;
  for (int i = threadIdx.x; i < n; i += kThreads) {
    const double y = fminf(ee[i], clip);
    s1 += y;
    s2 += y * y;
  }
  s1 = group_sum(s1, part);
  s2 = group_sum(s2, part);
  const float mu = float(s1 / dn);
  const float sigma = float(sqrt(fmax(1e-12, s2 / dn - double(mu) * mu)));
  for (double &v : s) v = 0;
  for (int i = threadIdx.x; i < n; i += kThreads) {
    const double y = (double(fminf(ee[i], clip)) - mu) / sigma, x = (double(fminf(pp[i], clip)) - mu) / sigma;
    s[0] += (x - y) * (x - y);
    s[1] += y;
    s[2] += x;
    s[3] += y * y;
    s[4] += x * x;
    s[5] += x * y;
  }
  for (double &v : s) v = group_sum(v, part) / dn;
  const double vy = fmax(0.0, s[3] - s[1] * s[1]), vx = fmax(0.0, s[4] - s[2] * s[2]), cxy = s[5] - s[1] * s[2];
  r.rmse = float(sqrt(s[0]));
  r.rmse_cal = float(sqrt(vx > 0 && cxy > 0 ? fmax(0.0, vy - cxy * cxy / vx) : vy));
  if (threadIdx.x == 0) out[blockIdx.x] = r;
}

}  // namespace

hipError_t pair_stats(const float *e, const float *p, const uint32_t *off, size_t npairs, size_t most,
                      const Params &q, Stats *out, hipStream_t s) {
  if (npairs == 0) return hipSuccess;
  if (most > kMaxSamples || npairs > 0x7fffffffu) return hipErrorInvalidValue;
  int room = 2;
  while (size_t(room) < most) room <<= 1;
  hipLaunchKernelGGL(stats_kernel, dim3(unsigned(npairs)), dim3(kThreads), unsigned(room * 9), s, e, p, off, room, q,
                     out);
  return hipGetLastError();
}

}  // namespace gate
}  // namespace bude
