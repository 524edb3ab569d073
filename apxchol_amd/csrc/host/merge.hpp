// Host side of the merged levels (kernels/merge.hip): which consecutive levels
// of a sweep run as one launch, and the rows of those launches.
#pragma once
#include <cstdint>
#include <vector>

#include "../device.hpp"
#include "../kernels/launch.hpp"
#include "trsv_prep.hpp"

namespace apxchol_amd {

struct merge_tables {
    std::vector<merge_step> steps;
    std::vector<lane_rec> rec;            // 64 per batch
    std::vector<merge_batch> batch;
    // Entries, kEpl * 64 per chunk; one piece per merged step, one after another.
    struct piece {
        std::vector<std::int32_t> idx;
        std::vector<double> val;
    };
    std::vector<piece> pieces;
    std::size_t slots = 0;
    std::uint64_t entries = 0;
};

// Steps for the levels [lo, hi) of one direction. level_first: first batch of
// each level in the direction's batch table (what a launch of the level on its
// own reads). A level joins the step before it while its merged rows hold at
// most max_growth entries more than the level's own (< 0: the default).
merge_tables build_merged_levels(const trsv_factor& T, bool backward, int lo, int hi,
                                 const std::vector<int>& level_first, long long max_growth = -1);

}  // namespace apxchol_amd
