// Level tiles of the launched levels (kernels/tile.hip): the host side.
#pragma once

#include "gpu_solver.hpp"

namespace apxchol_amd {

struct tile_tables {
    std::vector<lane_rec> rec;     // batches of 64 lanes, step by step and level by level
    std::vector<entry32> ent;      // kEpl planes of 64 per batch
    long long batches = 0;
    std::vector<tile_step> steps;  // ascending levels, disjoint
};

// Groups consecutive levels of [l0, l1) -- every one in the lane layout lt, its
// first lane batch level_lb[q], its batches level_first[q + 1] -
// level_first[q], its sweep positions from level_pos[q] -- into steps of up to
// max_levels levels where one launch of tiles is expected to take less time
// than the levels' own launches. m: the sweep's rows.
void append_tiles(const lane_tables& lt, bool backward, std::uint32_t m, const std::vector<int>& level_first,
                  const std::vector<int>& level_lb, const std::vector<int>& level_pos, int l0, int l1, int max_levels,
                  tile_tables& tt);

}  // namespace apxchol_amd
