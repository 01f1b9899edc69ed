// Host build of the reactive path's counters (mcell_amd/csrc/device/header.h)
// for tests/test_header.py.
#include "../mcell_amd/csrc/device/header.h"

using namespace mcg;

extern "C" {

// A call's phases one after the other, from `reacted` reactions on: for each
// the log row of its first and its last reaction; returns the reactions of
// the call.
uint64_t book_phases(uint64_t reacted, uint64_t phases, const uint32_t* n, uint64_t* rows) {
  alignas(8) uint32_t hdr[kHdrWords] = {};
  hdr_u64(hdr, kHdrReacted) = reacted;
  for (uint64_t i = 0; i < phases; ++i) {
    hdr[kHdrAccepted] = n[i];
    book_batch(hdr, n[i], 0, 1u << 20);
    rows[2 * i] = log_row(hdr, 0);
    rows[2 * i + 1] = log_row(hdr, n[i] - 1);
  }
  return hdr_u64(static_cast<const uint32_t*>(hdr), kHdrReacted);
}

// Slots: the used ones after a phase of `total` new molecules, and its first.
uint32_t book_slots(uint32_t used, uint32_t total, uint32_t capacity, uint32_t* first) {
  alignas(8) uint32_t hdr[kHdrWords] = {};
  hdr[kHdrNumOut] = used;
  book_batch(hdr, 1, total, capacity);
  *first = hdr[kHdrOutBase];
  return hdr[kHdrNumOut];
}

}  // extern "C"
