// The reactive path's counters ("the header"): words the kernels of an
// iteration count in, and the host's copy of them.
#pragma once
#include <stdint.h>

#include "wallbox.h"

namespace mcg {

enum : uint32_t {
  kHdrNumOut = 0,         // used output slots (snapshot size + products)
  kHdrProposals = 1,      // proposals of the current round
  kHdrAccepted = 2,       // accepted reactions of the current phase
  kHdrProductMovers = 3,  // products that move in this iteration
  kHdrRerun0 = 4,         // movers queued for another round (two lists)
  kHdrRerun1 = 5,
  kHdrSnapshot = 6,       // molecules in the snapshot (the iteration's movers)
  kHdrLog = 7,            // events logged (snapshot mode)
  kHdrUnimolDue = 8,      // molecules whose unimolecular reaction falls in this phase
  kHdrErr = 9,            // error bits (ERR_*) of the call's kernels
  kHdrExd = 10,           // movers the full step deferred to its exact_disk pass
  kHdrContinue = 11,      // movers of the phase that diffuse again in this iteration
  kHdrSurfMovers = 13,    // surface phase: the first pass's movers
  kHdrSurfCont0 = 15,     // surface phase: molecules that step again in this iteration (two lists)
  kHdrSurfCont1 = 16,
  kHdrOutBase = 17,       // products: the first output slot of the phase's new molecules
  kHdrBatch = 18,         // products: the phase's reactions
  kHdrReacted = 20,       // (64 bits) reactions of the call: it may cover any number of iterations
  kHdrMoveStart = 22,     // (64 bits) device clock at the start of the iteration's first move
  kHdrMoveTicks = 24,     // (64 bits) device clock ticks the call's first moves took
  kHdrLogBase = 26,       // (64 bits) products: reactions of the call before the phase
  kHdrSurfChanged = 28,   // surface phase: ends changed by each round of a batch (kSurfBatch words)
  kHdrWords = 36,
};
constexpr uint32_t kSurfBatch = 8;
// The host's copy of the counters, written by the kernels that end a round:
// the words, then the number of the copy.
constexpr uint32_t kHdrSeq = 40;
constexpr uint32_t kHdrHostWords = 64;

// A 64-bit counter of the header (its word is even, the header 8-byte aligned).
typedef unsigned long long __attribute__((may_alias)) HdrWord64;
MCG_BOX_HD HdrWord64& hdr_u64(uint32_t* hdr, uint32_t word) { return *reinterpret_cast<HdrWord64*>(hdr + word); }
MCG_BOX_HD uint64_t hdr_u64(const uint32_t* hdr, uint32_t word) {
  return *reinterpret_cast<const HdrWord64*>(hdr + word);
}

// The header after the phase's reactions are in order (one thread): their
// `total` new molecules take the output slots from the used ones on, never
// past the capacity (k_products reports what does not fit).
MCG_BOX_HD void book_batch(uint32_t* hdr, uint32_t n, uint32_t total, uint32_t capacity) {
  const uint32_t base = hdr[kHdrNumOut];
  const uint64_t used = (uint64_t)base + total;
  hdr[kHdrOutBase] = base;
  hdr[kHdrNumOut] = used < capacity ? (uint32_t)used : capacity;
  hdr[kHdrBatch] = n;
  hdr_u64(hdr, kHdrLogBase) = hdr_u64(hdr, kHdrReacted);
  hdr_u64(hdr, kHdrReacted) += n;
  hdr[kHdrAccepted] = 0;
  hdr[kHdrUnimolDue] = 0;
  hdr[kHdrProductMovers] = 0;
}

// The row of the call's log for the phase's reaction k, or log_cap or more if
// the log is full.
MCG_BOX_HD uint64_t log_row(const uint32_t* hdr, uint32_t k) { return hdr_u64(hdr, kHdrLogBase) + k; }

}  // namespace mcg
