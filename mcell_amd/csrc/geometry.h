// Host-side geometry set-up (wall constants, wall lists per subpartition).
#pragma once
#include <stdint.h>

#include <vector>

#include "device/types.h"

namespace mcg {

// Wall::initialize_wall_constants (src4/wall.cpp:281-342) for the triangle
// (p0, p1, p2), FP64, glm evaluation order.
WallRec64 wall_constants(const double* p0, const double* p1, const double* p2);

WallRec32 wall_to_fp32(const WallRec64& w);

// Per-subpartition wall lists in CSR form, wall indices ascending inside each
// list (Partition::walls_per_subpart holds ordered sets).
void bin_walls(const PartitionParams& P, const std::vector<WallRec64>& walls, std::vector<uint32_t>& off,
               std::vector<uint32_t>& idx);

// The sub-cell box (device/wallbox.h) of every list entry: the wall's
// bounding box within the entry's subpartition.  Returns the sum of the
// squared list lengths (over the entries: the mean list an entry sits in).
uint64_t entry_boxes(const PartitionParams& P, const std::vector<WallRec64>& walls, const std::vector<uint32_t>& off,
                 const std::vector<uint32_t>& idx, std::vector<uint32_t>& box);

// One bit per subpartition: whether a wall is listed in it or in one of its
// 26 neighbours (device/light.h, walls_around).
void cells_near_walls(const PartitionParams& P, const std::vector<uint32_t>& off, std::vector<uint32_t>& bits);

}  // namespace mcg
