// Host side of the trailing block (kernels/trail.hip): which rows it holds
// and the layout of its coupling to the rows before it.
#pragma once
#include <cstdint>
#include <vector>

#include "../device.hpp"
#include "trsv_prep.hpp"

namespace apxchol_amd {

// First level of the trailing block (the number of levels: no block). `value
// bytes` is the width of the sweeps' vectors; fwd_first / bck_first are the
// first batches of the levels of the two directions (levels + 1 each).
// max_rows < 0: by the cost model; otherwise the longest run of whole levels
// at the end of the factor with at most max_rows rows (0: no block).
std::size_t choose_trail_level(const trsv_factor& T, int value_bytes, const std::vector<int>& fwd_first,
                               const std::vector<int>& bck_first, int max_rows = -1);

// Whether S = T^-T W T^-1 of the rows from `first` on, each entry rounded to
// the sweeps' vector type, may stand for the walk of those rows. s_diag: S's
// diagonal before the rounding.
bool trail_is_sound(const trsv_factor& T, std::uint32_t first, const std::vector<double>& s_diag);

// The entries of the rows [first, m) that lie before `first`, for
// trail_couple: rows of at most 64 * kEpl of them in lane batches, the others
// listed with their range in the forward lists.
struct trail_couple_tables {
    std::vector<lane_rec> rec;
    std::vector<entry32> ent;
    std::vector<int4> longrow;
    int batches = 0;
};
trail_couple_tables build_trail_couple(const trsv_factor& T, std::uint32_t first);

}  // namespace apxchol_amd
