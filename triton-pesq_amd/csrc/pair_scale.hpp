// The common power of two of a pair of signals: 2^-e, 2^e <= peak < 2^(e + 1).
// Every bit of samples that are not far below the peak is kept by it, and what
// a scale invariant computation rounds afterwards is rounded as before, only
// away from the ends of the float32 range.
#pragma once

#include "common.hpp"

namespace pesq {

// partial peaks per pair, [pairs][kPairParts]: one per lane of the wavefronts
// that read them
constexpr int kPairParts = kWave;

// An infinite peak gives 0 (0 for the finite samples, NaN for the infinite ones)
// and a zero peak NaN, as division by the peak does.
__device__ __forceinline__ double pair_factor(float peak) {
    if (peak == 0.0f) return static_cast<double>(NAN);
    return isinf(peak) ? 0.0 : ldexp(1.0, -ilogb(static_cast<double>(peak)));
}
// the factor of a pair from its partial peaks (a whole wavefront's call)
__device__ __forceinline__ double pair_factor(const float *peaks, int64_t pair, int lane) {
    return pair_factor(wave_max(peaks[pair * kPairParts + lane]));
}

// peaks of the pairs (ref, deg) [batch, len] into `peaks` (elementwise.hip):
// one launch
int launch_pair_peaks(const float *ref, const float *deg, int64_t batch, int64_t len,
                      float *peaks, hipStream_t stream);

}  // namespace pesq
