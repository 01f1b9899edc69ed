// A team: 1, 2, 4, ... 64 consecutive lanes of a wave that work on one mover.
//
// The full step is one serial chain per mover, and where the list of full
// steps is shorter than the lanes of the chip the chain's length is the
// pass's time.  The lanes of a team run the same step on the same values
// (they branch alike); the scans inside it -- wall boxes, candidate walls,
// partners -- are dealt out over the lanes and their results combined, and
// only the leader writes.  Every result equals that of a lone lane bit for
// bit: the scans' outcomes are the first entry in list order or the minimum
// of a total order, neither of which depends on how the scan is split.
//
// Team sizes are uniform over a grid, so a team's lanes are always active
// together.  Solo is the team of one lane: the same code without any exchange
// (the host's, too).
#pragma once
#include <stdint.h>

#include "wallbox.h"

namespace mcg {

struct Team {
  static constexpr bool kShared = true;
  uint32_t size;  // lanes, a power of two
  uint32_t rank;  // this lane's place
  MCG_BOX_HD bool leader() const { return rank == 0; }
};
struct Solo {
  static constexpr bool kShared = false;
  static constexpr uint32_t size = 1, rank = 0;
  MCG_BOX_HD bool leader() const { return true; }
};

// The lowest rank whose lane has `want` set, or 64 if none.
MCG_BOX_HD uint32_t team_first(const Solo&, bool want) { return want ? 0u : 64u; }
#if defined(__HIPCC__) || defined(__HIP__)
__device__ __forceinline__ uint32_t team_first(const Team& T, bool want) {
  const uint64_t m = (__ballot(want) >> (__lane_id() - T.rank)) & (~0ull >> (64u - T.size));
  return m ? (uint32_t)__ffsll((unsigned long long)m) - 1u : 64u;
}
#endif

// next_overlap with the team's lanes reading the boxes: entry k + u * size +
// rank of every group is this lane's.
MCG_BOX_HD uint32_t next_overlap(const Solo&, const uint32_t* __restrict__ box, uint32_t k, uint32_t k1, uint32_t sb) {
  return next_overlap(box, k, k1, sb);
}
#if defined(__HIPCC__) || defined(__HIP__)
__device__ __forceinline__ uint32_t next_overlap(const Team& T, const uint32_t* __restrict__ box, uint32_t k,
                                                 uint32_t k1, uint32_t sb) {
  for (; k < k1; k += kOverlapGroup * T.size) {
    uint32_t bx[kOverlapGroup];
#pragma unroll
    for (uint32_t u = 0; u < kOverlapGroup; ++u) {
      const uint32_t e = k + u * T.size + T.rank;
      bx[u] = box[e < k1 ? e : k1 - 1];
    }
#pragma unroll
    for (uint32_t u = 0; u < kOverlapGroup; ++u) {
      const uint32_t e = k + u * T.size;
      if (e >= k1) break;
      const uint32_t r = team_first(T, e + T.rank < k1 && boxes_overlap(bx[u], sb));
      if (r < T.size) return e + r;
    }
  }
  return k1;
}

// Lane `rank` of the team's value of v.
template <typename V>
__device__ __forceinline__ V team_get(const Team& T, V v, uint32_t rank) {
  return __shfl(v, (int)(__lane_id() - T.rank + rank));
}

// The sum of v over the team.
__device__ __forceinline__ uint32_t team_sum(const Team& T, uint32_t v) {
  for (uint32_t o = 1; o < T.size; o <<= 1) v += __shfl_xor(v, (int)o);
  return v;
}

__device__ __forceinline__ uint32_t team_min_u32(const Team& T, uint32_t v) {
  for (uint32_t o = 1; o < T.size; o <<= 1) {
    const uint32_t v2 = __shfl_xor(v, (int)o);
    v = v2 < v ? v2 : v;
  }
  return v;
}

// The rank holding the smallest (t, tie) among the lanes with `have` set
// (64 if none has).
__device__ __forceinline__ uint32_t team_min(const Team& T, bool have, double t, uint32_t tie) {
  uint32_t r = have ? T.rank : 64u;
  for (uint32_t o = 1; o < T.size; o <<= 1) {
    const double t2 = __shfl_xor(t, (int)o);
    const uint32_t tie2 = __shfl_xor(tie, (int)o), r2 = __shfl_xor(r, (int)o);
    if (r2 < 64u && (r >= 64u || t2 < t || (t2 == t && tie2 < tie))) {
      t = t2;
      tie = tie2;
      r = r2;
    }
  }
  return r;
}
#endif

}  // namespace mcg
