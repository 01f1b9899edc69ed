// How many workgroups the reactive path's kernels are launched with (host
// arithmetic; the kernels read what there is to do on the device and are
// right with any number).
#pragma once
#include <stdint.h>

#include <algorithm>

namespace mcg {

// Workgroups of 256 threads the chip holds at once: 256 CUs, eight each.
constexpr uint32_t kFullChip = 2048;

// The scatter into bin order also clears the bins: at most this many per
// thread before it gets workgroups beyond its molecules' (up to a full chip).
// 200 molecules in a 4 um cube of 0.02 um subpartitions (4.1e7 bins) take
// 0.15 ms an iteration; with one workgroup clearing they took 1.41.
constexpr uint32_t kBinsPerThread = 16;
inline uint32_t scatter_workgroups(uint32_t molecules, uint32_t bins) {
  const uint32_t own = std::max<uint32_t>(1u, molecules / 256u + (molecules % 256u != 0));
  const uint32_t share = 256u * kBinsPerThread;
  return std::max(own, std::min(kFullChip, bins / share + (bins % share != 0)));
}

}  // namespace mcg
