// Host-side interface of the surface-molecule diffusion phase
// (kernels_surface.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "device/surface.h"

namespace mcg {

// The arrays of one surface phase.  Tile slots are replica-major,
// [replica * total_tiles + tile_base + tile].
struct SurfPhase {
  const WallRec64* __restrict__ walls;
  const WallGrid* __restrict__ grids;
  const WallEdgeRec* __restrict__ edges;     // 3 per wall
  const uint32_t* __restrict__ tile_wall;    // per tile of one replica
  SpeciesTable species;
  uint32_t* tiles;                           // tile words (kTileEmpty: free)
  uint32_t* tile_id;
  uint32_t* tile_consumed;
  double* tu;                                // molecule positions in the wall's uv frame
  double* tv;
  double* ttoff;                             // diffusion-time offsets from the iteration's start
  double* birth;                             // birthdays (absolute)
  // Per slot, of this round and of the one before it: the smallest order key
  // of the movers whose step ends on the slot's tile, under the round's code
  // (kernels_surface.hip), ...
  unsigned long long *claim, *claim_prev;
  uint32_t *dest, *dest_prev;                // ... and the slot a mover's step ends on (kSurfNotDue: none this iteration)
  // Per place in the mover list, the first max_tries of them: the slots of the
  // tiles the mover's attempts fall on, in order (its own: it stays on its
  // tile; kSurfSpent: no attempt left; kSurfUnknown: not worked out), and the
  // positions there.
  uint32_t* tries;                           // [kSurfTries * place + k]
  double* tries_uv;                          // [2 * (kSurfTries * place + k)]
  uint32_t max_tries;
  // Per mover slot: the position its step ends at.
  double* pu;
  double* pv;
  uint32_t* flags;                           // per mover slot: error bits | the attempts before them << 16; while
                                             // moving, the tile word
  uint32_t* moved_id;                        // per mover slot, while moving: the molecule's id
  uint32_t* list;                            // the pass's movers
  const uint32_t* count;
  // per slot: the iteration's stamp, stamp_base | kDoneFinal when its
  // molecule has no further step in the iteration, stamp_base | (pass + 1)
  // when it steps again in the next pass
  uint32_t* done;
  uint32_t* clist;                           // slots of the molecules that step again (next pass)
  uint32_t* ccount;
  uint32_t* hdr;
  uint32_t* err;
  uint32_t total_tiles, num_replicas;
  uint64_t seed;
  uint32_t iteration;
  uint32_t pass;                             // the pass (a molecule's n-th step in the iteration)
  uint32_t stamp_base;                       // ((iteration + 1) mod 2^28) << 4
  double barrier;                            // time up to the next barrier from the iteration's start
  uint32_t round;                            // the round of the pass
  uint32_t slot;                             // its place in the batch of rounds queued together
  uint32_t code, code_prev;                  // the claims' codes of this round and the one before (0: none)
};

constexpr uint32_t kDoneFinal = 15u;
constexpr uint32_t kSurfPasses = 8;          // steps per iteration (time steps of at least 1/8)
constexpr uint32_t kSurfNotDue = 0xFFFFFFFFu, kSurfUnknown = 0xFFFFFFFFu, kSurfSpent = 0xFFFFFFFEu;
constexpr uint32_t kSurfTries = kSurfRetries + 1;
// Codes of a claim word's high 31 bits: newer rounds have smaller ones, down
// to 1; a pass starts with enough of them left for its rounds.
constexpr uint32_t kSurfFirstCode = 0x7FFFFFFEu;
constexpr uint32_t kSurfMaxRounds = 100000;

// One round of a pass: every mover's end, given the ends of the movers ahead
// of it that the round before worked out; hdr[kHdrSurfChanged + P.slot], zero
// on entry, gets the number of ends it changed.  The first pass's first round
// (n_all > 0) looks at every slot and lists the movers; max_movers bounds or
// estimates them.
hipError_t surf_round(hipStream_t s, const SurfPhase& P, uint32_t n_all, uint32_t max_movers);
// The movers move, if the round P stands for changed nothing.
hipError_t surf_commit(hipStream_t s, const SurfPhase& P, uint32_t max_movers);
hipError_t launch_fill_done(hipStream_t s, uint32_t* done, uint32_t n);
// Zeroes two words of the header.
hipError_t launch_clear_words(hipStream_t s, uint32_t* hdr, uint32_t a, uint32_t b);
hipError_t launch_fill_claims(hipStream_t s, unsigned long long* claim, uint32_t n);

}  // namespace mcg
