// The surface phase of an iteration: every surface molecule of a species
// that diffuses takes its step (diffuse_surf_molecule,
// diffuse_react_event.cpp:1071-1246) after the iteration's volume phases.  A
// molecule whose end point lies on its own tile moves within it; one whose
// end point lies on another tile moves there if that tile is free, else it
// draws again (move_sm_on_same_triangle / move_sm_to_new_triangle,
// diffusion_utils.inl:453-548).
//
// The reference moves one molecule at a time: those whose diffusion time
// falls on the iteration's start by id, then the delayed ones by id
// (diffuse_molecules, diffuse_react_event.cpp:66-113).  So a tile is taken at
// a molecule's turn if
//   * its occupant at the start of the pass does not step in it, or is behind
//     in the order, or is ahead and its step ends on that same tile, or
//   * the step of some molecule ahead in the order ends on it.
// A step therefore depends on where the steps of molecules ahead of it end,
// and on nothing else that moves.  Rounds of all steps at once solve for the
// ends: every round works each step out from the ends of the round before
// (before the first, every molecule ends where it is); the first molecule's
// is right after one round, and each round makes right every step whose
// molecules ahead were, so a round that changes no end has found the
// sequential order's.  Only then do the movers move (two launches: all
// leave their tiles, then all arrive), so that within a round nothing is
// written that another molecule's step reads.  The tiles a step's attempts
// fall on do not depend on the others: they are kept, so that a later round
// only asks which of them is the first that is free, and works attempts out
// only where it needs one more than the rounds before.
//
// Claims: per slot the smallest order key among the movers that end there in
// a round, by atomicMin of code << 33 | key.  The code falls from round to
// round, so the claims of older rounds never stand in the way and need no
// clearing; two arrays take turns.
//
// Species with time steps below one iteration step again in further passes
// of the phase (the reference's later diffuse actions of the iteration), in
// the first pass's order, each pass reading the next pass of the molecule's
// stream.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "device/schedule.h"
#include "device/surface.h"
#include "kernels_react.h"
#include "kernels_surface.h"

namespace mcg {

namespace {

inline dim3 blocks_for(uint32_t n) { return dim3(std::max(1u, n / 256 + (n % 256 != 0))); }

__global__ void k_fill_claims(unsigned long long* claim, uint32_t n) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) claim[i] = ~0ull;
}

// A molecule's place in the phase's order: delayed << 32 | id.  In the
// first pass, delayed is read from the diffusion-time offset the molecule
// starts the iteration with (cmp_eq(delay, 0) fails); later passes keep
// the first pass's order through the tile word.
__device__ __forceinline__ bool surf_delayed(const SurfPhase& P, uint32_t tw, double toff) {
  return P.pass == 0 ? !cmp_eq_d(toff, 0.0, 1e-12) : (tw & kTileDelayed) != 0;
}
__device__ __forceinline__ unsigned long long surf_key(bool delayed, uint32_t id) {
  return ((unsigned long long)delayed << 32) | id;
}

// The time a surface molecule's step covers (diffuse_surf_molecule, :1081-
// 1116) with get_max_time's limits (:164-198): the time up to the barrier,
// shortened for a young molecule of a species with a long time step (no
// unimolecular clipping on this path).
struct SurfTiming {
  double t_steps, space_factor;
  bool mature;  // the molecule becomes mature with this step
};

__device__ __forceinline__ SurfTiming surf_timing(const SurfPhase& P, const SpeciesRec& sp, uint32_t tw, double toff,
                                                  double birth) {
  SurfTiming r;
  double max_time = P.barrier - toff;
  r.mature = false;
  if (!(tw & kTileMature) && sp.time_step > 1.0) {
    const double age_dependent_max_time = 1.0 + 0.2 * (((double)P.iteration + toff) - birth);
    if (max_time > age_dependent_max_time) max_time = age_dependent_max_time;
    r.mature = age_dependent_max_time > sp.time_step;
  }
  constexpr double EPS = 1e-12;
  r.t_steps = sp.time_step > max_time ? max_time : sp.time_step;
  double steps = 1.0;
  if (sp.time_step > max_time) {
    steps = max_time / sp.time_step;
    if (steps < EPS) {
      r.t_steps = EPS * sp.time_step;
      steps = EPS;
    }
  }
  r.space_factor = steps == 1.0 ? sp.space_step : sp.space_step * sqrt(steps);
  return r;
}

// The end of a molecule's step in slot s (diffuse_single_molecule's
// rescheduling, :287-318): diffusion_time += t_steps; still before the
// iteration's end, the molecule steps again in the next pass (its offset
// kept from this iteration's start), else its offset moves past the next
// iteration's start.
__device__ __forceinline__ void surf_step_over(const SurfPhase& P, uint32_t s, uint32_t tw, double toff,
                                               const SurfTiming& tm, bool delayed) {
  const double t_new = ((double)P.iteration + toff) + tm.t_steps;
  const bool again = cmp_lt_d(t_new, (double)P.iteration + 1.0, 1e-12);
  const uint32_t tw2 = (tw & ~kTileDelayed) | (tm.mature ? kTileMature : 0u) | (delayed ? kTileDelayed : 0u);
  if (tw2 != tw) P.tiles[s] = tw2;
  P.ttoff[s] = again ? t_new - (double)P.iteration : next_toff(P.iteration, toff, tm.t_steps);
  if (again) {
    if (P.pass + 1 >= kSurfPasses) {
      atomicOr(P.err, (uint32_t)ERR_PASSES);
      P.done[s] = P.stamp_base | kDoneFinal;
      return;
    }
    P.done[s] = P.stamp_base | (P.pass + 1);
    P.clist[atomicAdd(P.ccount, 1u)] = s;
  } else {
    P.done[s] = P.stamp_base | kDoneFinal;
  }
}

constexpr unsigned long long kClaimKey = (1ull << 33) - 1;

__device__ __forceinline__ bool surf_moves(const SpeciesRec& sp) {
  return (sp.flags & SPF_SURFACE) && sp.space_step > 0;
}
__device__ __forceinline__ const SpeciesRec& surf_species(const SurfPhase& P, uint32_t rep, uint32_t tw) {
  return P.species.rec[rep * P.species.stride + tile_species(tw)];
}

// Whether a step of the round before ends on slot ts, of a molecule ahead of
// `key` in the order.
__device__ __forceinline__ bool claimed_ahead(const SurfPhase& P, uint32_t ts, unsigned long long key) {
  const unsigned long long c = P.claim_prev[ts];
  return (uint32_t)(c >> 33) == P.code_prev && (c & kClaimKey) < key;
}

// Whether the tile of slot ts is taken at the turn of the molecule with order
// key `key`, as far as the round before knows.
__device__ __forceinline__ bool tile_taken(const SurfPhase& P, uint32_t rep, uint32_t ts, unsigned long long key) {
  const uint32_t occ = P.tiles[ts];
  if (occ != kTileEmpty) {
    if (!surf_moves(surf_species(P, rep, occ))) return true;
    const double toff = P.ttoff[ts];
    const bool steps = P.pass == 0 ? ready_this_iteration(P.iteration, toff) : P.done[ts] == (P.stamp_base | P.pass);
    if (!steps || surf_key(surf_delayed(P, occ, toff), P.tile_id[ts]) > key) return true;
    if (P.round == 0 || P.dest_prev[ts] == ts) return true;
  }
  return claimed_ahead(P, ts, key);
}

// The slot the molecule in slot s, the list's entry `at`, ends on, from the
// attempts kept: kSurfUnknown if they do not say.
__device__ __forceinline__ uint32_t kept_end(const SurfPhase& P, uint32_t at, uint32_t s, unsigned long long key) {
  if (at >= P.max_tries) return kSurfUnknown;
  for (uint32_t k = 0; k < kSurfTries; ++k) {
    const uint32_t ts = P.tries[(size_t)kSurfTries * at + k];
    if (ts == kSurfUnknown || ts == s) return ts;
    if (ts == kSurfSpent) return s;
    if (!tile_taken(P, s / P.total_tiles, ts, key)) return ts;
  }
  return s;
}

// The step of the molecule in slot s: the slot it ends on, the position there
// in pu, pv, and its attempts.
__device__ __forceinline__ uint32_t surf_step(const SurfPhase& P, uint32_t at, uint32_t s, uint32_t tw, double toff,
                                              unsigned long long key) {
  const uint32_t rep = s / P.total_tiles, lt = s - rep * P.total_tiles;
  const SurfTiming tm = surf_timing(P, surf_species(P, rep, tw), tw, toff, P.birth[s]);
  PhiloxStream rng;
  rng.init(P.seed, (uint32_t)key, P.iteration, rep, P.pass);
  const uint32_t wi = P.tile_wall[lt];
  const uint32_t t0 = lt - P.grids[wi].tile_base;
  const double u = P.tu[s], v = P.tv[s];
  const bool keep = at < P.max_tries;
  uint32_t* const tries = P.tries + (size_t)kSurfTries * at;
  double* const tries_uv = P.tries_uv + 2 * (size_t)kSurfTries * at;
  uint32_t err = 0, err_from = 0, end = s, tried = 0, next = kSurfSpent;
  double eu = u, ev = v;  // no position found: the molecule stays where it is for this step
  for (int attempt = 0; attempt <= kSurfRetries; ++attempt) {
    double du, dv;
    surf_displacement(rng, tm.space_factor, du, dv);
    double nu = 0, nv = 0;
    if (!err) err_from = tried;
    const uint32_t nw = ray_trace_surf(P.walls, P.edges, wi, u, v, du, dv, nu, nv, err);
    if (nw == kInvalid) continue;  // an ambiguous edge crossing: draw again
    const WallGrid& g = P.grids[nw];
    const uint32_t nt = uv2grid(P.walls[nw], g, nu, nv);
    if (nt == kInvalid) {
      err |= ERR_GRID;
      break;
    }
    // the same tile: the molecule moves within it
    const uint32_t ts = nw == wi && nt == t0 ? s : rep * P.total_tiles + g.tile_base + nt;
    if (keep) {
      tries[tried] = ts;
      tries_uv[2 * tried] = nu;
      tries_uv[2 * tried + 1] = nv;
    }
    ++tried;
    if (ts != s && tile_taken(P, rep, ts, key)) continue;
    end = ts;
    eu = nu;
    ev = nv;
    next = kSurfUnknown;
    break;
  }
  if (keep && tried < kSurfTries) tries[tried] = next;
  P.pu[s] = eu;
  P.pv[s] = ev;
  P.flags[s] = err ? err | err_from << 16 : 0u;
  return end;
}

// A round (n_all > 0: the first pass's first, over every slot).  The first of
// a pass is bound by the latency of a step (draws, edge crossings), the later
// ones by that of the few steps that need another attempt, or of the loads
// that say which tile is free.
__global__ __launch_bounds__(256) void k_surf_round(SurfPhase P, uint32_t n_all) {
  const uint32_t n = n_all ? n_all : *P.count;
  for (uint64_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
    const uint32_t s = n_all ? (uint32_t)i : P.list[i];
    const uint32_t tw = P.tiles[s];
    uint32_t at = (uint32_t)i;
    if (n_all) {
      if (tw == kTileEmpty || !surf_moves(surf_species(P, s / P.total_tiles, tw))) continue;
      at = atomicAdd(P.hdr + kHdrSurfMovers, 1u);
      P.list[at] = s;
    }
    const uint32_t before = P.round ? P.dest_prev[s] : s;
    const double toff = P.ttoff[s];
    if (n_all ? !ready_this_iteration(P.iteration, toff) : before == kSurfNotDue) {
      P.dest[s] = kSurfNotDue;
      continue;
    }
    const unsigned long long key = surf_key(surf_delayed(P, tw, toff), P.tile_id[s]);
    uint32_t end = P.round ? kept_end(P, at, s, key) : kSurfUnknown;
    if (end == kSurfUnknown) end = surf_step(P, at, s, tw, toff, key);
    if (end != before) atomicAdd(P.hdr + kHdrSurfChanged + P.slot, 1u);
    P.dest[s] = end;
    if (end != s) atomicMin(P.claim + end, ((unsigned long long)P.code << 33) | key);
  }
}

// The movers leave: steps within a tile are booked where they are, the others
// take their molecule off its tile (offset and birthday wait in the slot's
// claim words, which this pass is done with).
__global__ __launch_bounds__(256) void k_surf_leave(SurfPhase P) {
  if (P.hdr[kHdrSurfChanged + P.slot]) return;
  const uint32_t n = *P.count;
  for (uint64_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
    const uint32_t s = P.list[i], end = P.dest[s];
    const uint32_t tw = P.tiles[s];
    const double toff = P.ttoff[s];
    if (end == kSurfNotDue) {
      P.ttoff[s] = toff_past_iteration(P.iteration, toff);
      P.done[s] = P.stamp_base | kDoneFinal;
      continue;
    }
    // the position of the attempt it takes (none: where it is), and the
    // errors of the attempts up to it
    uint32_t k = kSurfTries;
    if (i < P.max_tries) {
      const size_t t = (size_t)kSurfTries * i;
      for (k = 0; k < kSurfTries; ++k) {
        const uint32_t ts = P.tries[t + k];
        if (ts == end || ts == kSurfSpent) break;
      }
      const bool found = k < kSurfTries && P.tries[t + k] == end;
      P.pu[s] = found ? P.tries_uv[2 * (t + k)] : P.tu[s];
      P.pv[s] = found ? P.tries_uv[2 * (t + k) + 1] : P.tv[s];
    }
    const uint32_t f = P.flags[s];
    if (f && k >= f >> 16) atomicOr(P.err, f & 0xFFFFu);
    const double birth = P.birth[s];
    if (end == s) {
      P.tu[s] = P.pu[s];
      P.tv[s] = P.pv[s];
      surf_step_over(P, s, tw, toff, surf_timing(P, surf_species(P, s / P.total_tiles, tw), tw, toff, birth),
                     surf_delayed(P, tw, toff));
      continue;
    }
    P.flags[s] = tw;
    P.moved_id[s] = P.tile_id[s];
    P.claim[s] = (unsigned long long)__double_as_longlong(toff);
    P.claim_prev[s] = (unsigned long long)__double_as_longlong(birth);
    P.tiles[s] = kTileEmpty;
    P.tile_id[s] = kInvalid;
  }
}

// The movers that left arrive and end their step there.
__global__ __launch_bounds__(256) void k_surf_arrive(SurfPhase P) {
  if (P.hdr[kHdrSurfChanged + P.slot]) return;
  const uint32_t n = *P.count;
  for (uint64_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
    const uint32_t s = P.list[i], ts = P.dest[s];
    if (ts == kSurfNotDue || ts == s) continue;
    const uint32_t tw = P.flags[s];
    const double toff = __longlong_as_double((long long)P.claim[s]);
    const double birth = __longlong_as_double((long long)P.claim_prev[s]);
    P.claim[s] = P.claim_prev[s] = ~0ull;
    P.tiles[ts] = tw;
    P.tile_id[ts] = P.moved_id[s];
    P.tu[ts] = P.pu[s];
    P.tv[ts] = P.pv[s];
    P.birth[ts] = birth;
    P.tile_consumed[ts] = 0;  // the molecule reacts with the volume movers of later iterations
    surf_step_over(P, ts, tw, toff, surf_timing(P, surf_species(P, s / P.total_tiles, tw), tw, toff, birth),
                   surf_delayed(P, tw, toff));
  }
}

__global__ void k_fill_ones(uint32_t* p, uint32_t n) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = ~0u;
}

__global__ void k_clear_words(uint32_t* hdr, uint32_t a, uint32_t b) {
  if (threadIdx.x == 0) hdr[a] = hdr[b] = 0;
}

}  // namespace

// no stamp of any iteration
hipError_t launch_fill_done(hipStream_t s, uint32_t* done, uint32_t n) {
  if (n) hipLaunchKernelGGL(k_fill_ones, blocks_for(n), dim3(256), 0, s, done, n);
  return hipGetLastError();
}

hipError_t launch_clear_words(hipStream_t s, uint32_t* hdr, uint32_t a, uint32_t b) {
  hipLaunchKernelGGL(k_clear_words, dim3(1), dim3(64), 0, s, hdr, a, b);
  return hipGetLastError();
}

hipError_t launch_fill_claims(hipStream_t s, unsigned long long* claim, uint32_t n) {
  if (n) hipLaunchKernelGGL(k_fill_claims, blocks_for(n), dim3(256), 0, s, claim, n);
  return hipGetLastError();
}

// (grid-stride: any grid is right)
static inline dim3 movers_grid(uint32_t n) { return dim3(std::min<uint32_t>(blocks_for(n).x, 2048u)); }

hipError_t surf_round(hipStream_t s, const SurfPhase& P, uint32_t n_all, uint32_t max_movers) {
  hipLaunchKernelGGL(k_surf_round, n_all ? blocks_for(n_all) : movers_grid(max_movers), dim3(256), 0, s, P, n_all);
  return hipGetLastError();
}

hipError_t surf_commit(hipStream_t s, const SurfPhase& P, uint32_t max_movers) {
  hipLaunchKernelGGL(k_surf_leave, movers_grid(max_movers), dim3(256), 0, s, P);
  hipLaunchKernelGGL(k_surf_arrive, movers_grid(max_movers), dim3(256), 0, s, P);
  return hipGetLastError();
}

}  // namespace mcg
