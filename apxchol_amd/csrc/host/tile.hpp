// Level tiles of the launched levels (kernels/tile.hip): the host side.
#pragma once

#include <memory>

#include "gpu_solver.hpp"

namespace apxchol_amd {

struct tile_tables {
    // One piece a step, level by level in it: 64 lanes and kEpl planes of 64
    // entries a batch.
    struct piece {
        std::size_t batches = 0;
        std::unique_ptr<lane_rec[]> rec;
        std::unique_ptr<entry32[]> ent;
    };
    std::vector<piece> pieces;
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
