// gate.h -- validation statistics of a combined screen's pairs.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

namespace bude {
namespace gate {

struct Params {
  double keep, top, z_req;    // rescored and top fractions, required gap in error deviations
  double tail_q;              // samples (lowest by exact energy) the error is taken over
  double clip_q;              // target transform: energies above this quantile count as it
};

// One pair's statistics (the host's gate_stats and norm_of, and the RMSE of
// the standardised scores).
struct Stats {
  double need;
  float z, recall, rmse, rmse_cal;
};

// Samples per pair the kernel takes (they are sorted in LDS).
constexpr size_t kMaxSamples = 4096;

// Statistics of npairs pairs, pair l from samples off[l] .. off[l + 1] - 1 of
// exact energies e and scores p (energy units); at most kMaxSamples each.
hipError_t pair_stats(const float *e, const float *p, const uint32_t *off, size_t npairs, size_t most,
                      const Params &q, Stats *out, hipStream_t s);

}  // namespace gate
}  // namespace bude
