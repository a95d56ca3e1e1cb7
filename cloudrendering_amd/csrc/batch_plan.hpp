// Sizes of a batched launch (api.cpp): samples per unit, unit records and drain states. Plain integers, no device code.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>

namespace crvpt {

struct BatchSize {
    uint64_t npix;  // pixels of a request
    uint32_t spp;
};

// Unit records of 16 bytes that a launch whose units are cut down may need (4 GiB).
constexpr uint64_t kBatchMaxSplitUnits = uint64_t(1) << 28;

inline uint64_t batchUnits(const BatchSize* q, size_t n, uint32_t samplesPerUnit) {
    uint64_t units = 0;
    for (size_t i = 0; i < n; i++) units += q[i].npix * ((uint64_t(q[i].spp) + samplesPerUnit - 1) / samplesPerUnit);
    return units;
}

// Units of fewer samples than the setting where the batch is too small for them: a lane's unit is a chain of samples,
// and a launch lasts as long as its last chain, so one sample per 64 paths that a lane gets (8 requests of 6.6 M paths,
// 25 per lane: 90.3 / 57.1 / 47.7 ms with 16 / 4 / 1 samples per unit). A unit needs a record, so not below what keeps
// the records within kBatchMaxSplitUnits: with the workgroups of an explicit setting, lanes can outnumber the paths.
inline uint32_t batchSamplesPerUnit(const BatchSize* q, size_t n, uint32_t setting, uint64_t lanes) {
    uint64_t paths = 0;
    for (size_t i = 0; i < n; i++) paths += q[i].npix * q[i].spp;
    const uint64_t perLane = paths / std::max<uint64_t>(lanes, 1);
    uint64_t g = std::min<uint64_t>(setting, std::max<uint64_t>(perLane / 64, 1));
    while (g < setting && batchUnits(q, n, uint32_t(g)) > kBatchMaxSplitUnits) g = std::min<uint64_t>(setting, 2 * g);
    return uint32_t(g);
}

// Paths that the pool can hand to the drain (units of one sample): one per lane, and no more than there are.
inline uint64_t batchDrainStates(uint64_t units, uint64_t lanes) { return std::min(units, lanes); }

}  // namespace crvpt
