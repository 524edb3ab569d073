// Level tiles: consecutive launched levels covered by one launch of independent
// tiles. A tile holds some rows of the last level and, in every level before
// it, all rows of the group of levels that they reach; a row that several tiles
// reach is computed by each of them, with the same bits, and written by the
// first. So no tile waits for another, and a launch boundary is needed once per
// group of levels only.
#include "tile.hpp"

#include <algorithm>
#include <cmath>
#include <numeric>
#include <stdexcept>

#include "threads.hpp"

namespace apxchol_amd {
namespace {

// Expected microseconds of a launch: its latency chain; a further level of a
// tile (a barrier, an LDS gather and the row sums); a batch of the tile with
// most of them (four gathers of a line a cycle each, one after the other on its
// compute unit); a batch of all (its 2.5 KB of layout). Mixed 128^3 SDDM solves
// stay within 1 % for half and twice the last two; without the last one they
// lose 4 %, at four times it as well.
constexpr double kLaunchUs = 3.6, kLevelUs = 0.8, kTileBatchUs = 0.11, kBatchUs = 0.001;
constexpr int kUnits = 256;   // compute units
// Tiles a trial looks at. A mixed 128^3 solve and the host time of its tiles
// (the trials one after another and the tables in one array): all 25.2 ms and
// 0.17 s, 32 25.4 and 0.13, 4 26.0 and 0.13.
constexpr int kSampleTiles = 32;

double launch_us(int levels, double batches, double tile_batches) {
    return kLaunchUs + kLevelUs * (levels - 1) + kTileBatchUs * std::max(tile_batches, batches / kUnits) +
           kBatchUs * batches;
}

struct tiling {
    std::vector<std::uint32_t> pos;   // positions, tile by tile and level by level
    std::vector<std::size_t> first;   // first position of (tile, level), one past the last at the end
    std::vector<long long> lanes;     // lanes of (tile, level)
    double us = 0;
};

class tiler {
public:
    tiler(const lane_tables& lt, bool backward, std::uint32_t m, const std::vector<int>& lf, const std::vector<int>& lb,
          const std::vector<int>& lp, int l0, int l1)
        : lt_(lt), backward_(backward), m_(m), p0_(static_cast<std::uint32_t>(lp[l0])), lp_(lp) {
        const std::size_t n = static_cast<std::size_t>(lp[l1]) - p0_;
        head_.assign(n, -1);
        level_.assign(n, -1);
        for (scratch& x : scratch_) x.mark.assign(n, 0);
        owner_.assign(n, 0);
        lanes_.assign(n, 0);
        for (int q = l0; q < l1; ++q)
            for (long long b = lb[q]; b < lb[q] + (lf[q + 1] - lf[q]); ++b)
                for (int l = 0; l < kWave; ++l) {
                    const lane_rec& r = lt.rec[static_cast<std::size_t>(b) * kWave + l];
                    if (r.row < 0 || ((r.info >> 3) & 63u)) continue;
                    const std::uint32_t p = position(r.row);
                    if (p < static_cast<std::uint32_t>(lp[q]) || p >= static_cast<std::uint32_t>(lp[q + 1]))
                        throw std::runtime_error("apxchol_amd: level tiles: row outside its level");
                    const std::uint32_t i = p - p0_;
                    head_[i] = b * kWave + l;
                    level_[i] = q;
                    const int G = group(i);
                    lanes_[i] = static_cast<unsigned char>(G);
                    if (l % G || l + G > kWave) throw std::runtime_error("apxchol_amd: level tiles: lane group");
                }
        // What the trials walk: a row's dependencies few enough levels back.
        dep_at_.reserve(n + 1);
        dep_at_.push_back(0);
        for (std::size_t i = 0; i < n; ++i) {
            if (head_[i] < 0) throw std::runtime_error("apxchol_amd: level tiles: row without lanes");
            const std::uint32_t from = static_cast<std::uint32_t>(lp[std::max(l0, level_[i] - kTileMaxLevels + 1)]);
            each_entry(static_cast<std::uint32_t>(i), [&](std::int32_t row) {
                const std::uint32_t p = position(row);
                if (p >= from) dep_.push_back(p - p0_);
            });
            dep_at_.push_back(dep_.size());
        }
    }

    // Tiles of the levels [a, a + J) with at most `waves` batches a level; false
    // when a row's tile would have more. limit > 0: an estimate of t.us from the
    // first tiles of the last level. Calls with another `place` (below kPlaces)
    // may run beside each other.
    static constexpr int kPlaces = 3;
    static_assert(4 << (kPlaces - 1) == kTileWaves, "a place for each number of waves");
    bool build(int a, int J, int waves, tiling& t, int limit = 0, int place = 0) {
        t = {};
        std::vector<int>& mark = scratch_[place].mark;
        std::vector<int>& undo = scratch_[place].undo;
        int& stamp = scratch_[place].stamp;
        std::vector<std::uint32_t> cur[kTileMaxLevels], add, stack;
        long long cnt[kTileMaxLevels] = {}, more[kTileMaxLevels];
        const std::uint32_t from = static_cast<std::uint32_t>(lp_[a]) - p0_;
        const int base = stamp;
        ++stamp;
        bool open = false;
        const auto close = [&] {
            for (int p = 0; p < J; ++p) {
                t.first.push_back(t.pos.size());
                t.pos.insert(t.pos.end(), cur[p].begin(), cur[p].end());
                t.lanes.push_back(cnt[p]);
                cur[p].clear();
                cnt[p] = 0;
            }
            ++stamp;
            open = false;
        };
        // Rows of the last level first; then those of the levels before it
        // that no tile has reached.
        for (int q = a + J - 1; q >= a; --q)
            for (std::uint32_t i = static_cast<std::uint32_t>(lp_[q]) - p0_; i < static_cast<std::uint32_t>(lp_[q + 1]) - p0_; ++i) {
                if (mark[i] > base) continue;
                for (;;) {
                    add.clear();
                    std::fill(more, more + J, 0);
                    const auto reach = [&](std::uint32_t j) {
                        mark[j] = stamp;
                        add.push_back(j);
                        stack.push_back(j);
                        more[level_[j] - a] += lanes_[j];
                    };
                    // Marks of the tiles before this one are kept for undoing.
                    undo.clear();
                    undo.push_back(mark[i]);
                    reach(i);
                    while (!stack.empty()) {
                        const std::uint32_t x = stack.back();
                        stack.pop_back();
                        for (std::size_t k = dep_at_[x]; k < dep_at_[x + 1]; ++k) {
                            const std::uint32_t j = dep_[k];
                            if (j < from || mark[j] == stamp) continue;
                            undo.push_back(mark[j]);
                            reach(j);
                        }
                    }
                    bool fits = true;
                    for (int p = 0; p < J; ++p) fits = fits && cnt[p] + more[p] <= waves * kWave;
                    if (fits) break;
                    for (std::size_t k = 0; k < add.size(); ++k) mark[add[k]] = undo[k];
                    if (!open) { stamp += 1; return false; }
                    close();
                    if (limit > 0 && q == a + J - 1 && static_cast<int>(t.lanes.size()) >= limit * J) {
                        const std::uint32_t q0 = static_cast<std::uint32_t>(lp_[q]) - p0_;
                        estimate(J, t, static_cast<double>(lp_[q + 1] - lp_[q]) / static_cast<double>(i - q0));
                        return true;
                    }
                }
                open = true;
                for (int p = 0; p < J; ++p) cnt[p] += more[p];
                for (const std::uint32_t j : add) cur[level_[j] - a].push_back(j);
            }
        if (open) close();
        t.first.push_back(t.pos.size());
        estimate(J, t, 1.0);
        return true;
    }

    void emit(int a, int J, const tiling& t, tile_tables& tt) {
        tile_step s;
        s.level = a;
        s.levels = J;
        s.tiles = static_cast<int>(t.lanes.size()) / J;
        for (int p = 0; p < J; ++p) {
            s.width[p] = 0;
            for (int k = 0; k < s.tiles; ++k)
                s.width[p] = std::max(s.width[p], static_cast<int>((t.lanes[static_cast<std::size_t>(k) * J + p] + kWave - 1) / kWave));
            if (tt.batches + static_cast<long long>(s.tiles) * s.width[p] > INT32_MAX)
                throw std::runtime_error("apxchol_amd: level tiles too large");
            s.base[p] = static_cast<int>(tt.batches);
            tt.batches += static_cast<long long>(s.tiles) * s.width[p];
        }
        // Written by the slices below, padding included: memory that one thread
        // has touched first, or that grows with every step, takes most of the
        // build (64^3: 97 of 128 ms).
        tile_tables::piece out;
        const long long first_batch = s.base[0];
        out.batches = static_cast<std::size_t>(tt.batches - first_batch);
        out.rec = std::make_unique_for_overwrite<lane_rec[]>(out.batches * kWave);
        out.ent = std::make_unique_for_overwrite<entry32[]>(out.batches * kWave * kEpl);
        // The first tile that computes a row writes it.
        ++step_;
        std::vector<char> own(t.pos.size());
        for (std::size_t k = 0; k < t.pos.size(); ++k) {
            own[k] = owner_[t.pos[k]] < step_;
            owner_[t.pos[k]] = step_;
        }
        const std::uint32_t p0 = static_cast<std::uint32_t>(lp_[a]), np = static_cast<std::uint32_t>(lp_[a + J]) - p0;
        // Tiles [k0, k1): their own slots in the records and entries.
        const auto write = [&](int k0, int k1, int& slots) {
            const auto slot_of = std::make_unique_for_overwrite<std::int32_t[]>(np);
            std::vector<std::size_t> rows;
            for (int k = k0; k < k1; ++k) {
                int slot = 0;
                for (int p = 0; p < J; ++p) {
                    const std::size_t f = static_cast<std::size_t>(k) * J + p;
                    rows.resize(t.first[f + 1] - t.first[f]);
                    std::iota(rows.begin(), rows.end(), t.first[f]);
                    // Wide rows first: groups then start at multiples of their size.
                    std::sort(rows.begin(), rows.end(), [&](std::size_t x, std::size_t y) {
                        const int gx = lanes_[t.pos[x]], gy = lanes_[t.pos[y]];
                        return gx != gy ? gx > gy : x < y;
                    });
                    const std::size_t b0 = static_cast<std::size_t>(s.base[p] - first_batch) +
                                           static_cast<std::size_t>(k) * static_cast<std::size_t>(s.width[p]);
                    const std::size_t b1 = b0 + static_cast<std::size_t>(s.width[p]);
                    std::fill(out.rec.get() + b0 * kWave, out.rec.get() + b1 * kWave, lane_rec{-1, 0});
                    std::fill(out.ent.get() + b0 * kWave * kEpl, out.ent.get() + b1 * kWave * kEpl, entry32{0, 0.0f});
                    long long at = static_cast<long long>(b0) * kWave;
                    for (const std::size_t x : rows) {
                        const std::uint32_t i = t.pos[x];
                        slot_of[i + p0_ - p0] = slot;
                        for (int g = 0; g < lanes_[i]; ++g, ++at) {
                            const long long from = head_[i] + g;
                            const lane_rec& r = lt_.rec[static_cast<std::size_t>(from)];
                            lane_rec& o = out.rec[static_cast<std::size_t>(at)];
                            o.row = r.row;
                            o.info = r.info | static_cast<std::uint32_t>(slot) << kTileSlotShift | (own[x] ? kTileOwn : 0u);
                            const int nv = static_cast<int>((r.info >> 9) & 7u);
                            for (int e = 0; e < nv; ++e) {
                                entry32 v = lt_.ent[entry_at(from, e)];
                                const std::uint32_t pj = position(v.idx);
                                if (pj >= p0) v.idx = ~slot_of[pj - p0];
                                out.ent[entry_at(at, e)] = v;
                            }
                        }
                        ++slot;
                    }
                }
                slots = std::max(slots, slot);
            }
        };
        constexpr int kThreads = 4;
        int slots[kThreads] = {};
        if (t.pos.size() < 4096) {
            write(0, s.tiles, slots[0]);
        } else {
            side_by_side(kThreads, [&](int q) {
                write(static_cast<int>(static_cast<long long>(s.tiles) * q / kThreads),
                      static_cast<int>(static_cast<long long>(s.tiles) * (q + 1) / kThreads), slots[q]);
            });
        }
        s.slots = *std::max_element(slots, slots + kThreads);
        tt.steps.push_back(s);
        tt.pieces.push_back(std::move(out));
    }

private:
    // t.us where t's tiles are one part in `parts` of all.
    static void estimate(int J, tiling& t, double parts) {
        long long batches = 0, most = 0, tile = 0;
        for (std::size_t k = 0; k < t.lanes.size(); ++k) {
            tile = (k % J ? tile : 0) + (t.lanes[k] + kWave - 1) / kWave;
            batches += (t.lanes[k] + kWave - 1) / kWave;
            most = std::max(most, tile);
        }
        t.us = launch_us(J, parts * static_cast<double>(batches), static_cast<double>(most));
    }
    std::uint32_t position(std::int32_t row) const {
        return backward_ ? m_ - 1 - static_cast<std::uint32_t>(row) : static_cast<std::uint32_t>(row);
    }
    int group(std::uint32_t i) const { return 1 << (lt_.rec[static_cast<std::size_t>(head_[i])].info & 7u); }
    static std::size_t entry_at(long long lane, int k) {
        return (static_cast<std::size_t>(lane / kWave) * kEpl + static_cast<std::size_t>(k)) * kWave +
               static_cast<std::size_t>(lane % kWave);
    }
    template <class F>
    void each_entry(std::uint32_t i, const F& f) const {
        const int G = group(i);
        for (int g = 0; g < G; ++g) {
            const long long at = head_[i] + g;
            const int nv = static_cast<int>((lt_.rec[static_cast<std::size_t>(at)].info >> 9) & 7u);
            for (int k = 0; k < nv; ++k) f(lt_.ent[entry_at(at, k)].idx);
        }
    }

    const lane_tables& lt_;
    const bool backward_;
    const std::uint32_t m_, p0_;
    const std::vector<int>& lp_;
    std::vector<long long> head_;   // lane of the row's first group lane, by position
    std::vector<unsigned char> lanes_;   // lanes of the row
    std::vector<std::size_t> dep_at_;
    std::vector<std::uint32_t> dep_;
    std::vector<int> level_, owner_;
    int step_ = 0;
    struct alignas(64) scratch {
        std::vector<int> mark, undo;
        int stamp = 1;
    };
    scratch scratch_[kPlaces];
};

}  // namespace

void append_tiles(const lane_tables& lt, bool backward, std::uint32_t m, const std::vector<int>& level_first,
                  const std::vector<int>& level_lb, const std::vector<int>& level_pos, int l0, int l1, int max_levels,
                  tile_tables& tt) {
    max_levels = std::min(max_levels, kTileMaxLevels);
    if (max_levels < 2 || l1 - l0 < 2) return;
    tiler T(lt, backward, m, level_first, level_lb, level_pos, l0, l1);
    const auto batches = [&](int q) { return level_first[q + 1] - level_first[q]; };
    // The best number of levels and waves is looked for again where the levels
    // have become a third smaller or larger.
    int J = 0, waves = 0, at = 0;
    for (int l = l0; l + 1 < l1;) {
        tiling keep;
        if (at == 0 || 3 * std::abs(batches(l) - at) > at || l + J > l1 || (J > 1 && !T.build(l, J, waves, keep))) {
            at = std::max(1, batches(l));
            J = 1;
            double least = launch_us(1, batches(l), 0);
            for (int j = 2; j <= std::min(max_levels, l1 - l) && j <= J + 1; ++j) {
                double us[tiler::kPlaces];
                side_by_side(tiler::kPlaces, [&](int k) {
                    tiling t;
                    us[k] = T.build(l, j, 4 << k, t, kSampleTiles, k) ? t.us : HUGE_VAL;
                });
                for (int k = 0; k < tiler::kPlaces; ++k)
                    if (us[k] / j < least) {
                        least = us[k] / j;
                        J = j;
                        waves = 4 << k;
                    }
            }
            if (J > 1 && !T.build(l, J, waves, keep)) J = 1;
        }
        if (J > 1) T.emit(l, J, keep, tt);
        l += J;
    }
}

}  // namespace apxchol_amd
