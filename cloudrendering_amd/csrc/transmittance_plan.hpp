// How a transmittance query is split into launches and what workspace it takes (transmittance.hip, api.cpp). Plain
// integers, no device code.
#pragma once

#include <algorithm>
#include <cstddef>

namespace crvpt {

constexpr size_t kTransmittanceUnits = size_t(1) << 26;     // estimates per launch
constexpr size_t kTransmittanceUnitsMin = size_t(1) << 16;  // where memory is short

struct TransmittancePlan {
    size_t rays, samples;  // rays and samples per ray of a launch
    size_t sumBytes;       // running sums of the rays whose samples span launches (a launch holds one such ray)
    size_t recordBytes;    // a launch's estimates (none for one sample: the estimate is the result)
    size_t bytes() const { return sumBytes + recordBytes; }
};

// Launches of `units` estimates at most: as many rays with all their samples as fit, or a part of one ray's samples.
inline TransmittancePlan transmittancePlan(int nRays, int nSamples, size_t units) {
    TransmittancePlan p{};
    p.samples = std::min(size_t(nSamples), units);
    p.rays = std::min(size_t(nRays), std::max<size_t>(1, units / p.samples));
    if (nSamples > 1) {
        p.sumBytes = p.samples < size_t(nSamples) ? p.rays * 2 * sizeof(double) : 0;
        p.recordBytes = p.rays * p.samples * sizeof(float);
    }
    return p;
}

}  // namespace crvpt
