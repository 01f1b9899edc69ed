// HIP kernels of the diffuse-react engine (gfx950).
//
// One iteration of non-reacting volume molecules is two launches:
//   k_light*  every molecule: draw the displacement; if the straight move
//             certainly touches no wall, commit it; otherwise append the
//             molecule to the hard queue (one atomic per wave).
//   k_hard*   queued molecules: the full ray trace with reflections, which
//             re-draws the same displacement from the molecule's stream.
// The light kernel holds few registers (high occupancy for the HBM stream);
// the register-heavy trace runs only for the few molecules near walls.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "device/displace.h"
#include "device/fastdraw.h"
#include "device/light.h"
#include "device/path32.h"
#include "device/path64.h"
#include "device/rng.h"
#include "device/types.h"
#include "kernels.h"

namespace mcg {

static __constant__ ZigguratTables c_zig = MCG_ZIGGURAT_TABLES_INIT;

// Stages the Ziggurat tables (2.5 KB) into LDS so that the per-lane strip
// lookups of a wave are LDS gathers rather than scattered cache reads.
__device__ __forceinline__ void stage_ziggurat(ZigguratTables& T) {
  const uint32_t* src = reinterpret_cast<const uint32_t*>(&c_zig);
  uint32_t* dst = reinterpret_cast<uint32_t*>(&T);
  constexpr int words = sizeof(ZigguratTables) / 4;
  for (int k = threadIdx.x; k < words; k += blockDim.x) dst[k] = src[k];
  __syncthreads();
}

__global__ void k_reset_counters(uint32_t* c, uint32_t n) {
  uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) c[i] = 0;
}

// The light passes run persistent: a grid of a few workgroups per CU walks
// the molecules tile by tile (256 per tile), so the strip tables are staged
// once per workgroup.  A tile's queued molecules go to shard tile % 2048.
//
// Queues: light passes append molecules whose displacement left the
// Ziggurat's fast path to the middle queue (shard = tile % 2048) and
// molecules a wall may stop to the first half of the full-step queue (shard
// = tile % 1024); the middle pass appends the molecules it does not clear to
// the second half (shard = 1024 + its tile % 1024).  Every shard holds the
// slots of all the tiles that map to it, so neither can overflow.
constexpr uint32_t kHalfShards = kQueueShards / 2;
__device__ __forceinline__ void append_light(bool mid, bool hard, uint32_t i, uint32_t tile, const SlowQueue& MQ,
                                             const SlowQueue& HQ) {
  const uint32_t ms = tile % kQueueShards, hs = tile % kHalfShards;
  wave_append(mid, i, MQ.slots + (size_t)ms * MQ.shard_cap, MQ.count + ms);
  wave_append(hard, i, HQ.slots + (size_t)hs * HQ.shard_cap, HQ.count + hs);
}
__device__ __forceinline__ void append_mid(bool hard, uint32_t i, uint32_t base, const SlowQueue& HQ) {
  const uint32_t hs = kHalfShards + (base / 256u) % kHalfShards;
  wave_append(hard, i, HQ.slots + (size_t)hs * HQ.shard_cap, HQ.count + hs);
}

// The move p -> p + m (FP32) certainly meets no wall and stays inside the
// partition, with its end point clear of every tested wall plane by `band`.
__device__ __forceinline__ bool clear_move32(const PartitionParams32& Q, const Walls32View& W, const FilterParams& F,
                                             float band, float px, float py, float pz, float mx, float my,
                                             float mz) {
  const float ex = px + mx, ey = py + my, ez = pz + mz;
  int lo[3], hi[3];
  if (!index_box32(Q, px, py, pz, ex, ey, ez, lo, hi)) return false;
  return walls_clear(Q, W.off, W.box, px, py, pz, ex, ey, ez, lo, hi, [&](uint32_t k) {
    float de;
    return certain_miss32(W.ent32[k], F, px, py, pz, mx, my, mz, &de) && fabs_f(de) >= band;
  });
}

// The FP64 move certainly meets no wall (the reference's collide_wall of
// every wall of the index box returns MISS: bit-exact) and stays inside the
// partition.  The index and entry boxes are FP32 and conservative.
__device__ __forceinline__ bool clear_move64(const PartitionParams32& Q, const WallView64& W, const D3& pos,
                                             const D3& disp, const D3& end) {
  const float px = (float)pos.x, py = (float)pos.y, pz = (float)pos.z;
  const float ex = (float)end.x, ey = (float)end.y, ez = (float)end.z;
  int lo[3], hi[3];
  if (!index_box32(Q, px, py, pz, ex, ey, ez, lo, hi)) return false;
  return walls_clear(Q, W.off, W.box, px, py, pz, ex, ey, ez, lo, hi,
                     [&](uint32_t k) { return wall_certain_miss64(W.ent[k], pos, disp); });
}

// One molecule's step on the light path: whether it commits (pos moved), or
// who takes it: its displacement is off the Ziggurat's fast path (the full
// draw decides), or a wall may stop it (the full ray trace).
enum : uint32_t { kStepDone = 0, kStepMid = 1, kStepHard = 2 };

__device__ __forceinline__ uint32_t light_step64(const FastZiggurat& T, const PartitionParams32& Q,
                                                 const WallView64& W, uint64_t seed, uint32_t id, uint32_t iteration,
                                                 uint32_t replica, double space_step, D3& pos) {
  uint32_t r0, r1, r2, r3;
  philox_block0(seed, id, iteration, replica, 0, r0, r1, r2, r3);
  D3 disp;
  if (!fast_displacement(r0, r1, r2, T, space_step, disp.x, disp.y, disp.z)) return kStepMid;
  const D3 end = {pos.x + disp.x, pos.y + disp.y, pos.z + disp.z};
  if (!clear_move64(Q, W, pos, disp, end)) return kStepHard;
  pos = end;
  return kStepDone;
}

struct F3 {
  float x, y, z;
};
__device__ __forceinline__ uint32_t light_step32(const FastZiggurat& T, const PartitionParams32& Q,
                                                 const Walls32View& W, const FilterParams& F, float band,
                                                 uint64_t seed, uint32_t id, uint32_t iteration, uint32_t replica,
                                                 double space_step, F3& pos) {
  uint32_t r0, r1, r2, r3;
  philox_block0(seed, id, iteration, replica, 0, r0, r1, r2, r3);
  float mx, my, mz;
  if (!fast_displacement32(r0, r1, r2, T, (float)(space_step * 0.70710678118654752440), mx, my, mz)) return kStepMid;
  if (!clear_move32(Q, W, F, band, pos.x, pos.y, pos.z, mx, my, mz)) return kStepHard;
  pos = {pos.x + mx, pos.y + my, pos.z + mz};
  return kStepDone;
}

// ------------------------------------------------------------------- FP64 --
// Every molecule whose three Gaussians are on the Ziggurat's fast path and
// whose straight move certainly meets no wall (FP64 collide_wall of every
// wall in the move's index box, bit-exact: wall_certain_miss64) commits here;
// the others go to k_hard64, which draws the same stream through rng_gauss.
__global__ __launch_bounds__(256) void k_light64(MolView64 m, uint32_t n, SpeciesTable species,
                                                 PartitionParams32 Q, WallView64 W, uint64_t seed,
                                                 uint32_t iteration, SlowQueue MQ, SlowQueue HQ, HitTrace trace) {
  __shared__ FastZiggurat T;
  stage_fast_ziggurat(T, c_zig);
  for (uint32_t tile = blockIdx.x; tile * 256u < n; tile += gridDim.x) {
    const uint32_t i = tile * 256u + threadIdx.x;
    bool mid = false, hard = false;
    if (i < n) {
      const uint32_t tag = m.tag[i];
      const uint32_t idv = m.id[i];
      const D3 pos = {m.x[i], m.y[i], m.z[i]};
      const SpeciesRec sp = species.of(tag);
      if (!(tag_flags(tag) & MF_DEFUNCT) && sp.space_step > 0) {
        D3 at = pos;
        const uint32_t r = light_step64(T, Q, W, seed, idv, iteration, tag_replica(tag), sp.space_step, at);
        if (r == kStepDone) {
          m.x[i] = at.x;
          m.y[i] = at.y;
          m.z[i] = at.z;
          if (trace.enabled) trace.count[i] = 0;
        }
        mid = r == kStepMid;
        hard = r == kStepHard;
      }
    }
    append_light(mid, hard, i, tile, MQ, HQ);
  }
}

__global__ __launch_bounds__(256) void k_mid64(MolView64 m, SpeciesTable species, PartitionParams32 Q,
                                               WallView64 W, uint64_t seed, uint32_t iteration, SlowQueue MQ,
                                               SlowQueue HQ, HitTrace trace) {
  __shared__ ZigguratTables T;
  __shared__ uint32_t pre[kQueueShards + 1];
  __shared__ uint32_t part[4];
  const uint32_t total = queue_prefix(MQ.count, MQ.nshards, pre, part);
  if ((uint64_t)blockIdx.x * blockDim.x >= total) return;
  stage_ziggurat(T);
  for (uint32_t base = blockIdx.x * blockDim.x; base < total; base += gridDim.x * blockDim.x) {
    const uint32_t q = base + threadIdx.x;
    uint32_t i = 0;
    bool hard = false;
    if (q < total) {
      i = queue_at(MQ.slots, MQ.shard_cap, pre, q);
      const uint32_t tag = m.tag[i];
      const SpeciesRec sp = species.of(tag);
      PhiloxStream rng;
      rng.init(seed, m.id[i], iteration, tag_replica(tag), 0);
      const D3 disp = draw_displacement(rng, T, sp.space_step);
      const D3 pos = {m.x[i], m.y[i], m.z[i]};
      const D3 end = {pos.x + disp.x, pos.y + disp.y, pos.z + disp.z};
      hard = !clear_move64(Q, W, pos, disp, end);
      if (!hard) {
        m.x[i] = end.x;
        m.y[i] = end.y;
        m.z[i] = end.z;
        if (trace.enabled) trace.count[i] = 0;
      }
    }
    append_mid(hard, i, base, HQ);
  }
}

__global__ __launch_bounds__(256) void k_hard64(MolView64 m, SpeciesTable species, SurfaceClasses SC,
                                                PartitionParams P, WallView64 W, uint64_t seed, uint32_t iteration,
                                                SlowQueue Q, uint32_t* __restrict__ err_out, HitTrace trace,
                                                unsigned long long* __restrict__ ctr) {
  __shared__ ZigguratTables T;
  __shared__ uint32_t pre[kQueueShards + 1];
  __shared__ uint32_t part[4];
  // the shards read as one list, grid-stride
  const uint32_t total = queue_prefix(Q.count, Q.nshards, pre, part);
  if ((uint64_t)blockIdx.x * blockDim.x >= total) return;
  stage_ziggurat(T);
  uint32_t n_reflect = 0, n_cross = 0;
  // every thread of the block runs the same number of rounds (the counters
  // are wave-summed after the loop)
  for (uint32_t base = blockIdx.x * blockDim.x; base < total; base += gridDim.x * blockDim.x) {
    const uint32_t q = base + threadIdx.x;
    if (q >= total) continue;
    const uint32_t i = queue_at(Q.slots, Q.shard_cap, pre, q);
    const uint32_t tag = m.tag[i];
    const SpeciesRec sp = species.of(tag);
    PhiloxStream rng;
    rng.init(seed, m.id[i], iteration, tag_replica(tag), 0);
    D3 pos = {m.x[i], m.y[i], m.z[i]};
    const D3 disp = draw_displacement(rng, T, sp.space_step);
    uint32_t err = 0, tn = 0;
    uint32_t* tw = trace.enabled ? trace.wall + (size_t)i * kTraceHits : nullptr;
    const bool alive = diffuse_reflect64(P, W.walls, W.ent, W.off, W.idx, W.box, SC, tag_species(tag), pos, disp, rng,
                                         err, tw, tn, n_reflect, n_cross);
    m.x[i] = pos.x;
    m.y[i] = pos.y;
    m.z[i] = pos.z;
    if (!alive) m.tag[i] = tag | (MF_DEFUNCT << 8);
    if (trace.enabled) trace.count[i] = tn;
    if (err) atomicOr(err_out, err);
  }
  wave_count(ctr + CTR_REFLECTIONS, n_reflect);
  wave_count(ctr + CTR_CROSSINGS, n_cross);
}

// ------------------------------------------------------------------- FP32 --
// Everything in FP32: the displacement (within kMoveUlps of the FP64 one),
// the end point, the index and entry boxes, and the wall filter (filter32.h,
// widened by the displacement's error), which certifies misses of the FP64
// move as well.  An end point within `band` of a tested wall's plane takes
// the full step, which rounds the FP64 end point onto its side.
__global__ __launch_bounds__(256) void k_light32(MolView32 m, uint32_t n, SpeciesTable species,
                                                 PartitionParams32 Q, Walls32View W, FilterParams F, float band,
                                                 uint64_t seed, uint32_t iteration, SlowQueue MQ, SlowQueue HQ,
                                                 HitTrace trace) {
  __shared__ FastZiggurat T;
  stage_fast_ziggurat(T, c_zig);
  for (uint32_t tile = blockIdx.x; tile * 256u < n; tile += gridDim.x) {
    const uint32_t i = tile * 256u + threadIdx.x;
    bool mid = false, hard = false;
    if (i < n) {
      const uint32_t tag = m.tag[i];
      const uint32_t idv = m.id[i];
      const float px = m.x[i], py = m.y[i], pz = m.z[i];
      const SpeciesRec sp = species.of(tag);
      if (!(tag_flags(tag) & MF_DEFUNCT) && sp.space_step > 0) {
        F3 at = {px, py, pz};
        const uint32_t r = light_step32(T, Q, W, F, band, seed, idv, iteration, tag_replica(tag), sp.space_step, at);
        if (r == kStepDone) {
          m.x[i] = at.x;
          m.y[i] = at.y;
          m.z[i] = at.z;
          if (trace.enabled) trace.count[i] = 0;
        }
        mid = r == kStepMid;
        hard = r == kStepHard;
      }
    }
    append_light(mid, hard, i, tile, MQ, HQ);
  }
}

// Middle pass: the molecules whose displacement left the fast path.  The
// displacement is drawn through rng_gauss from the same stream (FP64, the
// reference's), then the light checks decide as in the light passes; the
// molecules they do not clear go on to the full step.
__global__ __launch_bounds__(256) void k_mid32(MolView32 m, SpeciesTable species, PartitionParams32 Q,
                                               Walls32View W, FilterParams F, float band, uint64_t seed,
                                               uint32_t iteration, SlowQueue MQ, SlowQueue HQ, HitTrace trace) {
  __shared__ ZigguratTables T;
  __shared__ uint32_t pre[kQueueShards + 1];
  __shared__ uint32_t part[4];
  const uint32_t total = queue_prefix(MQ.count, MQ.nshards, pre, part);
  if ((uint64_t)blockIdx.x * blockDim.x >= total) return;
  stage_ziggurat(T);
  for (uint32_t base = blockIdx.x * blockDim.x; base < total; base += gridDim.x * blockDim.x) {
    const uint32_t q = base + threadIdx.x;
    uint32_t i = 0;
    bool hard = false;
    if (q < total) {
      i = queue_at(MQ.slots, MQ.shard_cap, pre, q);
      const uint32_t tag = m.tag[i];
      const SpeciesRec sp = species.of(tag);
      PhiloxStream rng;
      rng.init(seed, m.id[i], iteration, tag_replica(tag), 0);
      const D3 disp = draw_displacement(rng, T, sp.space_step);
      const float px = m.x[i], py = m.y[i], pz = m.z[i];
      const float mx = (float)disp.x, my = (float)disp.y, mz = (float)disp.z;
      hard = !clear_move32(Q, W, F, band, px, py, pz, mx, my, mz);
      if (!hard) {
        m.x[i] = px + mx;
        m.y[i] = py + my;
        m.z[i] = pz + mz;
        if (trace.enabled) trace.count[i] = 0;
      }
    }
    append_mid(hard, i, base, HQ);
  }
}

__global__ __launch_bounds__(256) void k_hard32(MolView32 m, SpeciesTable species, SurfaceClasses SC,
                                                PartitionParams P, Walls32View W,
                                                uint64_t seed, uint32_t iteration, SlowQueue Q,
                                                uint32_t* __restrict__ err_out, HitTrace trace,
                                                unsigned long long* __restrict__ ctr) {
  __shared__ ZigguratTables T;
  __shared__ uint32_t pre[kQueueShards + 1];
  __shared__ uint32_t part[4];
  // the shards read as one list, grid-stride
  const uint32_t total = queue_prefix(Q.count, Q.nshards, pre, part);
  if ((uint64_t)blockIdx.x * blockDim.x >= total) return;
  stage_ziggurat(T);
  uint32_t n_reflect = 0, n_cross = 0;
  for (uint32_t base = blockIdx.x * blockDim.x; base < total; base += gridDim.x * blockDim.x) {
    const uint32_t q = base + threadIdx.x;
    if (q >= total) continue;
    const uint32_t i = queue_at(Q.slots, Q.shard_cap, pre, q);
    const uint32_t tag = m.tag[i];
    const SpeciesRec sp = species.of(tag);
    PhiloxStream rng;
    rng.init(seed, m.id[i], iteration, tag_replica(tag), 0);
    D3 pos = {(double)m.x[i], (double)m.y[i], (double)m.z[i]};
    const D3 disp = draw_displacement(rng, T, sp.space_step);
    uint32_t err = 0, tn = 0;
    uint32_t* tw = trace.enabled ? trace.wall + (size_t)i * kTraceHits : nullptr;
    // the FP64 wall search (a queued molecule meets few walls after the
    // entry-box pre-test; the FP32 filter in front of them cost more than
    // it saved), then the end point rounded to FP32 on its side of nearby
    // wall planes
    const bool alive = diffuse_reflect64(P, W.w64, W.ent64, W.off, W.idx, W.box, SC, tag_species(tag), pos, disp,
                                         rng, err, tw, tn, n_reflect, n_cross);
    if (!alive) m.tag[i] = tag | (MF_DEFUNCT << 8);
    float fx, fy, fz;
    if (!round_to_fp32_same_side(Solo{}, P, W.w64, W.off, W.idx, W.box, pos.x, pos.y, pos.z, &fx, &fy, &fz))
      err |= ERR_ROUND32;
    m.x[i] = fx;
    m.y[i] = fy;
    m.z[i] = fz;
    if (trace.enabled) trace.count[i] = tn;
    if (err) atomicOr(err_out, err);
  }
  wave_count(ctr + CTR_REFLECTIONS, n_reflect);
  wave_count(ctr + CTR_CROSSINGS, n_cross);
}

// ------------------------------------------------- several iterations at once --
// Molecules that react with nothing do not see each other, so a wave keeps
// up to 64 molecules in registers and takes them through all iterations of
// the call: memory is read and written once per call, and no launch, queue or
// synchronisation lies between two steps.  Every lane counts its own
// iterations.  Steps off the light path wait until half of the wave's
// unfinished lanes wait for one, and are then taken together: a full step's
// chain costs the wave many light steps however many lanes take it, and
// about one step in ten needs one.  Few molecules are spread over all the
// waves the chip holds (kRunWaves; 224 registers, two waves per SIMD): a
// wave's chains are then shorter and fewer.  Same steps, same order per
// molecule: the results equal those of single iterations bit for bit.
// Bound by the chains' latency; 10,000 molecules in a box take 11 us an
// iteration in calls of 64 (the three passes: 80), 262,144 take 42 (100).
struct FreeForm64 {
  using Pos = D3;
  MolView64 m;
  WallView64 W;
  __device__ __forceinline__ Pos load(uint32_t i) const { return {m.x[i], m.y[i], m.z[i]}; }
  __device__ __forceinline__ void store(uint32_t i, const Pos& p) const {
    m.x[i] = p.x;
    m.y[i] = p.y;
    m.z[i] = p.z;
  }
  __device__ __forceinline__ uint32_t light(const FastZiggurat& T, const PartitionParams32& Q, uint64_t seed,
                                            uint32_t id, uint32_t it, uint32_t rep, double step, Pos& p) const {
    return light_step64(T, Q, W, seed, id, it, rep, step, p);
  }
  // the move of a full draw, if it certainly meets no wall
  __device__ __forceinline__ bool clear(const PartitionParams32& Q, const D3& disp, Pos& p) const {
    const D3 end = {p.x + disp.x, p.y + disp.y, p.z + disp.z};
    if (!clear_move64(Q, W, p, disp, end)) return false;
    p = end;
    return true;
  }
  __device__ __forceinline__ bool trace(const PartitionParams& P, const SurfaceClasses& SC, uint32_t species,
                                        const D3& disp, PhiloxStream& rng, Pos& p, uint32_t& err, uint32_t& n_reflect,
                                        uint32_t& n_cross) const {
    uint32_t tn = 0;
    return diffuse_reflect64(P, W.walls, W.ent, W.off, W.idx, W.box, SC, species, p, disp, rng, err, nullptr, tn,
                             n_reflect, n_cross);
  }
};

struct FreeForm32 {
  using Pos = F3;
  MolView32 m;
  Walls32View W;
  FilterParams F;
  float band;
  __device__ __forceinline__ Pos load(uint32_t i) const { return {m.x[i], m.y[i], m.z[i]}; }
  __device__ __forceinline__ void store(uint32_t i, const Pos& p) const {
    m.x[i] = p.x;
    m.y[i] = p.y;
    m.z[i] = p.z;
  }
  __device__ __forceinline__ uint32_t light(const FastZiggurat& T, const PartitionParams32& Q, uint64_t seed,
                                            uint32_t id, uint32_t it, uint32_t rep, double step, Pos& p) const {
    return light_step32(T, Q, W, F, band, seed, id, it, rep, step, p);
  }
  __device__ __forceinline__ bool clear(const PartitionParams32& Q, const D3& disp, Pos& p) const {
    const float mx = (float)disp.x, my = (float)disp.y, mz = (float)disp.z;
    if (!clear_move32(Q, W, F, band, p.x, p.y, p.z, mx, my, mz)) return false;
    p = {p.x + mx, p.y + my, p.z + mz};
    return true;
  }
  __device__ __forceinline__ bool trace(const PartitionParams& P, const SurfaceClasses& SC, uint32_t species,
                                        const D3& disp, PhiloxStream& rng, Pos& p, uint32_t& err, uint32_t& n_reflect,
                                        uint32_t& n_cross) const {
    uint32_t tn = 0;
    D3 q = {(double)p.x, (double)p.y, (double)p.z};
    const bool alive = diffuse_reflect64(P, W.w64, W.ent64, W.off, W.idx, W.box, SC, species, q, disp, rng, err,
                                         nullptr, tn, n_reflect, n_cross);
    if (!round_to_fp32_same_side(Solo{}, P, W.w64, W.off, W.idx, W.box, q.x, q.y, q.z, &p.x, &p.y, &p.z))
      err |= ERR_ROUND32;
    return alive;
  }
};

template <class Form>
__global__ __launch_bounds__(64, 2) void k_run(Form S, uint32_t n, uint32_t per_wave, SpeciesTable species,
                                               SurfaceClasses SC, PartitionParams P, PartitionParams32 Q,
                                               uint64_t seed, uint32_t first, uint32_t num,
                                               uint32_t* __restrict__ err_out,
                                               unsigned long long* __restrict__ ctr) {
  __shared__ FastZiggurat F;
  __shared__ ZigguratTables T;
  stage_fast_ziggurat(F, c_zig);
  stage_ziggurat(T);
  const uint32_t i = blockIdx.x * per_wave + threadIdx.x;
  uint32_t tag = 0, id = 0, it = num;
  typename Form::Pos pos = {0, 0, 0};
  double step = 0;
  if (threadIdx.x < per_wave && i < n) {
    tag = S.m.tag[i];
    id = S.m.id[i];
    pos = S.load(i);
    step = species.of(tag).space_step;
    if (!(tag_flags(tag) & MF_DEFUNCT) && step > 0) it = 0;
  }
  const bool moves = it == 0 && num > 0;
  const uint32_t rep = tag_replica(tag);
  uint32_t wait = kStepDone, err = 0, n_reflect = 0, n_cross = 0, n_last = 0;
  for (;;) {
    for (;;) {
      const bool go = it < num && wait == kStepDone;
      const uint32_t going = (uint32_t)__popcll(__ballot(go));
      const uint32_t waiting = (uint32_t)__popcll(__ballot(wait != kStepDone));
      if (going <= waiting) break;  // (also when none goes)
      if (go) {
        wait = S.light(F, Q, seed, id, first + it, rep, step, pos);
        if (wait == kStepDone) ++it;
      }
    }
    if (__ballot(wait != kStepDone) == 0) break;  // every lane is through
    if (wait != kStepDone) {
      PhiloxStream rng;
      rng.init(seed, id, first + it, rep, 0);
      const D3 disp = draw_displacement(rng, T, step);
      bool alive = true;
      if (!(wait == kStepMid && S.clear(Q, disp, pos))) {
        if (it + 1 == num) ++n_last;
        alive = S.trace(P, SC, tag_species(tag), disp, rng, pos, err, n_reflect, n_cross);
      }
      if (!alive) {
        S.m.tag[i] = tag | (MF_DEFUNCT << 8);
        it = num;
      } else {
        ++it;
      }
      wait = kStepDone;
    }
  }
  if (moves) S.store(i, pos);
  if (err) atomicOr(err_out, err);
  wave_count(ctr + CTR_REFLECTIONS, n_reflect);
  wave_count(ctr + CTR_CROSSINGS, n_cross);
  wave_count(ctr + CTR_LAST_TRACED, n_last);
}

// Copy kernel of known size (device-to-device bandwidth reference).
__global__ __launch_bounds__(256) void k_copy(const float4* __restrict__ src, float4* __restrict__ dst, size_t n) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  size_t stride = (size_t)gridDim.x * blockDim.x;
  for (; i < n; i += stride) dst[i] = src[i];
}

// -------------------------------------------------------------- launchers --
static_assert(kNumQueueShards == kQueueShards, "host and device shard counts differ");
static_assert(kQueueShards % 256 == 0, "counter reset grid");

// Persistent grid of a 256-thread kernel: as many workgroups as can be
// resident at once (CUs x the kernel's occupancy), never more than the tiles
// -- a workgroup beyond what fits would only start after others finish and
// then walk its share of the tiles alone.
template <typename Kernel>
static dim3 persistent_grid(Kernel kernel, uint32_t n) {
  static int resident = 0;
  if (resident == 0) {
    int dev = 0, cus = 0, per_cu = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
      cus = 256;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, 256, 0) != hipSuccess || per_cu <= 0)
      per_cu = 1;
    resident = cus * per_cu;
  }
  const uint32_t tiles = (n + 255) / 256;
  return dim3(std::max<uint32_t>(1u, std::min<uint32_t>(tiles, (uint32_t)resident)));
}

uint32_t shard_capacity(uint32_t n, uint32_t shards) {
  uint32_t blocks = (n + 255) / 256;
  return 256u * ((blocks + shards - 1) / shards);
}


constexpr uint32_t kRunWaves = 2048;  // waves of k_run the chip holds (256 CUs x 4 SIMDs x 2)
static inline uint32_t run_per_wave(uint32_t n) {
  return std::max<uint32_t>(1u, std::min<uint32_t>(64u, (n + kRunWaves - 1) / kRunWaves));
}

// Two turns of the waves the chip holds: the line up to which no call loses.
// In a box single calls of 262,144 molecules take 155 us by k_run and 170 by
// the passes, of 300,000 173 and 170 (FP32 177 and 169), of 500,000 240 and
// 180.  Longer calls would still gain above it (calls of 64, us an iteration:
// 40 and 92 at 262,144, 72 and 108 at 500,000, 135 and 134 at 1,000,000), and
// so would fine meshes, where k_run's full steps gain most (163,852 walls, a
// mean list of 233: 35 and 317 at 1,000 molecules, 254 and 1,520 at 262,144).
bool run_pays(uint32_t n) { return n <= 2u * 64u * kRunWaves; }

hipError_t launch_run64(hipStream_t s, const MolView64& m, uint32_t n, SpeciesTable species, const SurfaceClasses& SC,
                        const PartitionParams& P, const WallView64& W, uint64_t seed, uint32_t first, uint32_t num,
                        uint32_t* err, unsigned long long* ctr) {
  if (n == 0 || num == 0) return hipSuccess;
  const uint32_t per = run_per_wave(n);
  hipLaunchKernelGGL(k_run<FreeForm64>, dim3((n + per - 1) / per), dim3(64), 0, s, FreeForm64{m, W}, n, per,
                     species, SC, P, make_partition32(P), seed, first, num, err, ctr);
  return hipGetLastError();
}

hipError_t launch_run32(hipStream_t s, const MolView32& m, uint32_t n, SpeciesTable species, const SurfaceClasses& SC,
                        const PartitionParams& P, const WallView64& W, const WallRec32* w32, float max_abs_coord,
                        uint64_t seed, uint32_t first, uint32_t num, uint32_t* err, unsigned long long* ctr) {
  if (n == 0 || num == 0) return hipSuccess;
  const uint32_t per = run_per_wave(n);
  const FilterParams F = make_filter_params(max_abs_coord, kMoveUlps);
  const float band = 2.0f * F.e_dd + 8.0f * F.eps * max_abs_coord;
  const Walls32View W32{W.walls, reinterpret_cast<const FilterWall*>(w32), W.off, W.idx,
                        reinterpret_cast<const FilterWall*>(W.ent32), W.box, W.ent};
  hipLaunchKernelGGL(k_run<FreeForm32>, dim3((n + per - 1) / per), dim3(64), 0, s, FreeForm32{m, W32, F, band}, n, per,
                     species, SC, P, make_partition32(P), seed, first, num, err, ctr);
  return hipGetLastError();
}

hipError_t launch_diffuse_reflect64(hipStream_t s, const MolView64& m, uint32_t n, SpeciesTable species,
                                    const SurfaceClasses& SC,
                                    const PartitionParams& P, const WallView64& W, uint64_t seed, uint32_t iteration,
                                    SlowQueue MQ, SlowQueue Q, uint32_t* err, const HitTrace& trace,
                                    unsigned long long* ctr) {
  if (n == 0) return hipSuccess;
  const PartitionParams32 P32 = make_partition32(P);
  MQ.shard_cap = shard_capacity(n);
  MQ.nshards = kQueueShards;
  Q.shard_cap = shard_capacity(n, kHalfShards);
  Q.nshards = kQueueShards;
  hipLaunchKernelGGL(k_reset_counters, dim3(kQueueShards / 256), dim3(256), 0, s, MQ.count, kQueueShards);
  hipLaunchKernelGGL(k_reset_counters, dim3(kQueueShards / 256), dim3(256), 0, s, Q.count, kQueueShards);
  hipLaunchKernelGGL(k_light64, persistent_grid(k_light64, n), dim3(256), 0, s, m, n, species, P32, W, seed,
                     iteration, MQ, Q, trace);
  hipLaunchKernelGGL(k_mid64, persistent_grid(k_mid64, n), dim3(256), 0, s, m, species, P32, W, seed, iteration, MQ,
                     Q, trace);
  hipLaunchKernelGGL(k_hard64, dim3(std::min<uint32_t>(kQueueShards, (n + 255) / 256)), dim3(256), 0, s, m, species,
                     SC, P, W, seed, iteration, Q, err, trace, ctr);
  return hipGetLastError();
}

hipError_t launch_diffuse_reflect32(hipStream_t s, const MolView32& m, uint32_t n, SpeciesTable species,
                                    const SurfaceClasses& SC,
                                    const PartitionParams& P, const WallView64& W, const WallRec32* w32,
                                    float max_abs_coord, uint64_t seed, uint32_t iteration, SlowQueue MQ,
                                    SlowQueue Q, uint32_t* err, const HitTrace& trace, unsigned long long* ctr) {
  if (n == 0) return hipSuccess;
  FilterParams F = make_filter_params(max_abs_coord, kMoveUlps);
  float band = 2.0f * F.e_dd + 8.0f * F.eps * max_abs_coord;
  Walls32View W32{W.walls, reinterpret_cast<const FilterWall*>(w32), W.off, W.idx,
                  reinterpret_cast<const FilterWall*>(W.ent32), W.box, W.ent};
  const PartitionParams32 P32 = make_partition32(P);
  MQ.shard_cap = shard_capacity(n);
  MQ.nshards = kQueueShards;
  Q.shard_cap = shard_capacity(n, kHalfShards);
  Q.nshards = kQueueShards;
  hipLaunchKernelGGL(k_reset_counters, dim3(kQueueShards / 256), dim3(256), 0, s, MQ.count, kQueueShards);
  hipLaunchKernelGGL(k_reset_counters, dim3(kQueueShards / 256), dim3(256), 0, s, Q.count, kQueueShards);
  hipLaunchKernelGGL(k_light32, persistent_grid(k_light32, n), dim3(256), 0, s, m, n, species, P32, W32, F, band,
                     seed, iteration, MQ, Q, trace);
  hipLaunchKernelGGL(k_mid32, persistent_grid(k_mid32, n), dim3(256), 0, s, m, species, P32, W32, F, band, seed,
                     iteration, MQ, Q, trace);
  hipLaunchKernelGGL(k_hard32, dim3(std::min<uint32_t>(kQueueShards, (n + 255) / 256)), dim3(256), 0, s, m, species,
                     SC, P, W32, seed, iteration, Q, err, trace, ctr);
  return hipGetLastError();
}

hipError_t launch_copy(hipStream_t s, const void* src, void* dst, size_t bytes) {
  size_t n = bytes / sizeof(float4);
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_copy, dim3(2048), dim3(256), 0, s, static_cast<const float4*>(src), static_cast<float4*>(dst),
                     n);
  return hipGetLastError();
}

}  // namespace mcg
