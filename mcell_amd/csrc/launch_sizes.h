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

// The list of movers that diffuse again is copied behind the products' by one
// workgroup, which updates the counts too, while that takes no longer than a
// grid and a second launch (4.3 us and the gap between them): 4.1 us at 8,000
// entries, 6.0 at 16,000, 10.2 at 32,000, 34 at 128,000, 272 at 1,000,000,
// where the grid takes 3.8.
constexpr uint32_t kAppendAlone = 16384;
inline uint32_t append_workgroups(uint32_t entries) {
  return entries <= kAppendAlone ? 1u : std::min(kFullChip, entries / 256u + (entries % 256u != 0));
}

// What the rounds of an iteration are expected to bring: proposals, and
// movers deferred for a larger exact_disk pool.  A phase's first round is
// expected to be like the first round the same phase had in the last
// iteration (the first moves by the drain's form, which decides what they
// defer; then the moves of products and of movers that diffuse again, phase
// by phase).  The later rounds of a phase repeat the moves of a list whose
// length is known, and say nothing about any first round.
struct RoundSizes {
  static constexpr uint32_t kUnknown = 0xFFFFFFFFu;
  static constexpr uint32_t kPhases = 8;  // list phases told apart; later ones are taken for the last of these
  uint32_t props[2 + kPhases], deferred[2 + kPhases];
  RoundSizes() {
    std::fill(props, props + 2 + kPhases, kUnknown);
    std::fill(deferred, deferred + 2 + kPhases, kUnknown);
  }
  // phase 0: the iteration's first moves with the drain's form 1 or 2
  static uint32_t slot(uint32_t phase, uint32_t form) { return phase == 0 ? form - 1 : 1 + std::min(phase, kPhases); }
  uint32_t expect_props(uint32_t phase, uint32_t form, uint32_t round, uint32_t movers) const {
    return round ? movers : std::min(movers, props[slot(phase, form)]);
  }
  uint32_t expect_deferred(uint32_t phase, uint32_t form, uint32_t round, uint32_t movers) const {
    return round ? movers : std::min(movers, deferred[slot(phase, form)]);
  }
  void first_round(uint32_t phase, uint32_t form, uint32_t proposals, uint32_t deferred_movers) {
    props[slot(phase, form)] = proposals;
    deferred[slot(phase, form)] = deferred_movers;
  }
};

// A length to launch for where `expected` was seen last and `bound` is the
// most there can be.
inline uint32_t room_for(uint32_t expected, uint32_t bound) {
  return (uint32_t)std::min<uint64_t>(bound, 64 + 2 * (uint64_t)expected);
}

}  // namespace mcg
