#include "merge.hpp"

#include <algorithm>
#include <atomic>
#include <barrier>
#include <exception>
#include <functional>
#include <mutex>
#include <optional>
#include <stdexcept>
#include <thread>

namespace apxchol_amd {

namespace {

// A launch of a level costs about 3.3 us beyond its bytes, which move at about
// 4 TB/s: a level joins the step before it while the bytes it adds cost less.
constexpr double kLaunchUs = 3.0;
constexpr double kBytesPerUs = 4.0e6;
// ... and while its rows grow by at most this many entries: the substitution
// is host work at setup and memory. Growths of 0 / 60,000 / 100,000 / 200,000 /
// 400,000: solve grid3d 48 fp64 6.4 / 4.4 / 3.9 / 3.8 / 4.1 ms, sddm3d 89 fp64
// 12.0 / 11.1 / 10.4 / 9.7 / 9.8, apply sddm3d 63 272 / 219 / 180 / 171 / 182 us.
// At 100,000 the setups grow from 62 to 75, 358 to 373 and 109 to 136 ms: five
// to ten solves repay them, so one-shot solves do without.
constexpr long long kMaxGrowth = 100000;
// Levels of more entries than this are launched on their own: two of them
// merged grow by a third and more.
constexpr double kLevelsOf = 2.5;   // times the growth
// Entries of a merged row.
constexpr std::size_t kMaxRow = 2048;

struct term {
    std::int32_t src;   // >= 0: output of that row; < 0: right-hand side of row ~src
    double coef;
};

// The rows of the open step in sweep order, each a sum over outputs before
// the step and right-hand sides inside it.
struct open_step {
    std::vector<std::vector<term>> part;   // one per level and thread: a thread appends to its own
                                           // while all read those of the levels before
    struct ref {
        std::uint32_t part, off, len;
    };
    std::vector<ref> rows;   // those of the first level have length 0 until a level joins it
    std::size_t used = 0;    // parts in use; the others keep their memory for later levels
    std::size_t take(unsigned n) {
        const std::size_t at = used;
        used += n;
        if (part.size() < used) part.resize(used);
        for (std::size_t k = at; k < used; ++k) part[k].clear();
        return at;
    }
    void clear() {
        used = 0;
        rows.clear();
    }
};

struct scratch {
    std::vector<double> acc;           // m outputs, then the step's right-hand sides
    std::vector<unsigned char> seen;
    std::vector<std::uint32_t> touched;
};

// A few threads that run one job after another: at most n with the calling
// one, fewer where the process may not start that many.
class team {
public:
    explicit team(unsigned n) {
        const std::lock_guard<std::mutex> hold(counting_);   // the threads wait for their number
        threads_.reserve(n);
        try {
            for (unsigned w = 1; w < n; ++w)
                threads_.emplace_back([this, w] {
                    { const std::lock_guard<std::mutex> wait(counting_); }
                    loop(w);
                });
        } catch (...) {   // no thread, or no memory for one
        }
        gate_.emplace(static_cast<std::ptrdiff_t>(size()));
    }
    ~team() {
        job_ = nullptr;
        gate_->arrive_and_wait();
        for (auto& t : threads_) t.join();
    }
    unsigned size() const { return static_cast<unsigned>(threads_.size()) + 1; }
    // job(w) on every thread; rethrows the first exception.
    void run(const std::function<void(unsigned)>& job) {
        job_ = &job;
        failed_ = nullptr;
        gate_->arrive_and_wait();
        call(0);
        gate_->arrive_and_wait();
        if (failed_) std::rethrow_exception(failed_);
    }

private:
    void call(unsigned w) {
        try {
            (*job_)(w);
        } catch (...) {
            if (!taken_.exchange(true)) failed_ = std::current_exception();
        }
    }
    void loop(unsigned w) {
        for (;;) {
            gate_->arrive_and_wait();
            if (!job_) return;
            call(w);
            gate_->arrive_and_wait();
        }
    }
    std::mutex counting_;
    std::optional<std::barrier<>> gate_;
    const std::function<void(unsigned)>* job_ = nullptr;
    std::atomic<bool> taken_{false};
    std::exception_ptr failed_;
    std::vector<std::thread> threads_;
};

int lanes_of(std::size_t len) {
    std::size_t g = 1;
    while (g < 64 && g * kEpl < len) g *= 2;
    return static_cast<int>(g);
}

}  // namespace

merge_tables build_merged_levels(const trsv_factor& T, bool backward, int lo, int hi,
                                 const std::vector<int>& level_first, long long max_growth) {
    merge_tables out;
    const std::uint32_t m = T.m;
    const int L = static_cast<int>(T.level_ptr.size()) - 1;
    if (lo < 0 || hi > L || static_cast<int>(level_first.size()) != L + 1)
        throw std::runtime_error("apxchol_amd: level range of the merged levels");
    if (max_growth < 0) max_growth = kMaxGrowth;
    const auto& ptr = backward ? T.b_ptr : T.f_ptr;
    const auto& idx = backward ? T.b_idx : T.f_idx;
    const auto& val = backward ? T.b_val : T.f_val;
    const auto& hv = backward ? T.b_h : T.f_h;
    const auto pos = [&](int l) { return backward ? m - T.level_ptr[L - l] : T.level_ptr[l]; };
    const auto row_at = [&](std::uint32_t t) { return backward ? m - 1 - t : t; };
    const auto weight = [&](std::uint32_t p) {
        return static_cast<double>(T.fp16 ? fp16_widen(hv[p]) : val[p]);
    };
    // Scale of row r's right-hand side (fp16 storage, back sweep).
    const auto rhs_scale = [&](std::uint32_t r) {
        if (!backward || T.inv_scale.empty()) return 1.0;
        const double s = static_cast<double>(T.inv_scale[r]);
        return s * s;
    };
    // Without merging no thread is needed. The threads' scratch (9 bytes a row
    // each) stays under 256 MB.
    const unsigned room = static_cast<unsigned>(std::min<std::uint64_t>(8, (256ull << 20) / (9ull * std::max(m, 1u))));
    team workers(max_growth == 0 ? 1u : std::max(1u, std::min(room, std::thread::hardware_concurrency())));
    const unsigned nthr = workers.size();
    std::vector<scratch> scr(nthr);
    open_step open;
    std::uint32_t p0 = 0;        // first position of the open step
    int first = lo;              // its first level
    std::vector<double> level_bytes;   // of its levels, merged

    // Rows [ta, tb) of the level from position `base` on by thread w, into
    // part `into`; ends early once the level's entries pass the limit.
    const auto expand = [&](std::uint32_t ta, std::uint32_t tb, unsigned w, std::uint32_t into,
                            std::vector<open_step::ref>& refs, std::uint32_t base, std::atomic<long long>& entries,
                            long long limit) {
        scratch& s = scr[w];
        const std::size_t slots = static_cast<std::size_t>(m) + (base + refs.size() - p0);
        if (s.acc.size() < slots) {
            s.acc.resize(slots, 0.0);
            s.seen.resize(slots, 0);
        }
        const auto at_pos = [&](std::uint32_t r) { return backward ? m - 1 - r : r; };
        const auto add = [&](std::int32_t src, double c) {
            const std::uint32_t k = src >= 0 ? static_cast<std::uint32_t>(src)
                                             : m + (at_pos(static_cast<std::uint32_t>(~src)) - p0);
            if (!s.seen[k]) {
                s.seen[k] = 1;
                s.touched.push_back(k);
            }
            s.acc[k] += c;
        };
        long long mine = 0;
        for (std::uint32_t t = ta; t < tb; ++t) {
            const std::uint32_t r = row_at(t);
            const double inv = 1.0 / static_cast<double>(T.diag[r]);
            s.touched.clear();
            add(~static_cast<std::int32_t>(r), rhs_scale(r) * inv);
            for (std::uint32_t p = ptr[r]; p < ptr[r + 1]; ++p) {
                const std::int32_t j = idx[p];
                const std::uint32_t pj = backward ? m - 1 - static_cast<std::uint32_t>(j) : static_cast<std::uint32_t>(j);
                const double c = -weight(p) * inv;
                if (pj < p0) {
                    add(j, c);
                } else {
                    const auto& q = open.rows[pj - p0];
                    if (q.len == 0) {   // a row of the first level: its own entries
                        const std::uint32_t rj = static_cast<std::uint32_t>(j);
                        const double cj = c / static_cast<double>(T.diag[rj]);
                        add(~j, cj * rhs_scale(rj));
                        for (std::uint32_t k = ptr[rj]; k < ptr[rj + 1]; ++k) add(idx[k], -cj * weight(k));
                        continue;
                    }
                    const term* e = open.part[q.part].data() + q.off;
                    for (std::uint32_t k = 0; k < q.len; ++k) add(e[k].src, c * e[k].coef);
                }
            }
            // In order of the rows read: neighbouring lanes then gather from
            // neighbouring lines (apply sddm3d 63: 170 us, 192 unsorted).
            std::sort(s.touched.begin(), s.touched.end());
            auto& o = open.part[into];
            refs[t - base] = {into, static_cast<std::uint32_t>(o.size()), static_cast<std::uint32_t>(s.touched.size())};
            for (const std::uint32_t k : s.touched) {
                o.push_back({k < m ? static_cast<std::int32_t>(k) : ~static_cast<std::int32_t>(row_at(p0 + (k - m))),
                             s.acc[k]});
                s.acc[k] = 0.0;
                s.seen[k] = 0;
            }
            mine += static_cast<long long>(s.touched.size());
            if (s.touched.size() > kMaxRow) mine += limit + 1;
        }
        entries.fetch_add(mine);
    };
    // Expands level l into the open step; false (nothing kept) past the limit.
    const auto expand_level = [&](int l, long long limit, long long& total) {
        const std::uint32_t a = pos(l), b = pos(l + 1), n = b - a;
        std::vector<open_step::ref> refs(n);
        const std::uint32_t into = static_cast<std::uint32_t>(open.take(nthr));
        std::atomic<long long> entries{0};
        // Slices of 64 rows, handed out in order.
        std::atomic<std::uint32_t> next{0};
        const std::function<void(unsigned)> job = [&](unsigned w) {
            for (;;) {
                const std::uint32_t k = next.fetch_add(64);
                if (k >= n || entries.load(std::memory_order_relaxed) > limit) return;
                expand(a + k, std::min(b, a + k + 64), w, into + w, refs, a, entries, limit);
            }
        };
        if (n <= 64) job(0);
        else workers.run(job);
        total = entries.load();
        if (total > limit) {
            open.used = into;
            return false;
        }
        if (l == first) std::copy(refs.begin(), refs.end(), open.rows.begin());
        else open.rows.insert(open.rows.end(), refs.begin(), refs.end());
        return true;
    };
    // Bytes of level l launched on its own, and of the rows [from, ..) of the
    // open step as merged batches.
    const auto own_bytes = [&](int l) {
        return static_cast<double>(level_first[l + 1] - level_first[l]) * kWave * (8 + kEpl * 8) +
               static_cast<double>(pos(l + 1) - pos(l)) * 24.0;
    };
    const auto merged_bytes = [&](std::size_t from) {
        double lanes = 0.0;
        for (std::size_t k = from; k < open.rows.size(); ++k) {
            const std::uint32_t r = row_at(p0 + static_cast<std::uint32_t>(k));
            const std::size_t len = open.rows[k].len > 0 ? open.rows[k].len : ptr[r + 1] - ptr[r] + 1u;
            const std::size_t g = static_cast<std::size_t>(lanes_of(len));
            lanes += static_cast<double>(g) * static_cast<double>(std::max<std::size_t>(1, (len + g * kEpl - 1) / (g * kEpl)));
        }
        return lanes * (8.0 + kEpl * (4.0 + 8.0));
    };

    // Writes the open step [first, end) out.
    const auto emit = [&](int end) {
        merge_step st;
        st.l0 = first;
        st.l1 = end;
        if (end - first > 1) {
            st.b0 = static_cast<int>(out.batch.size());
            // Rows packed in order, each at a multiple of its lanes.
            struct place {
                std::uint32_t row;
                int start;
            };
            std::vector<place> places;
            std::vector<std::uint32_t> begin;   // first place of each batch
            std::uint32_t slab = static_cast<std::uint32_t>(out.slots / (kEpl * kWave));
            int used = kWave;
            for (std::uint32_t k = 0; k < open.rows.size(); ++k) {
                const std::size_t len = open.rows[k].len;
                const int G = lanes_of(len);
                int at = (used + G - 1) / G * G;
                if (at + G > kWave) {
                    if (!out.batch.empty() && !begin.empty()) slab += out.batch.back().chunks;
                    begin.push_back(static_cast<std::uint32_t>(places.size()));
                    out.batch.push_back({slab, 1});
                    at = 0;
                }
                places.push_back({k, at});
                used = at + G;
                const std::uint32_t chunks = static_cast<std::uint32_t>((len + static_cast<std::size_t>(G) * kEpl - 1) / (static_cast<std::size_t>(G) * kEpl));
                out.batch.back().chunks = std::max(out.batch.back().chunks, chunks);
                out.entries += len;
            }
            slab += out.batch.back().chunks;
            begin.push_back(static_cast<std::uint32_t>(places.size()));
            const std::size_t base = out.slots;
            out.slots = static_cast<std::size_t>(slab) * kEpl * kWave;
            out.pieces.emplace_back();
            auto& piece = out.pieces.back();
            piece.idx.resize(out.slots - base, 0);
            piece.val.resize(out.slots - base, 0.0);
            out.rec.resize(out.batch.size() * kWave, lane_rec{-1, 0u});
            const std::uint32_t nb = static_cast<std::uint32_t>(begin.size()) - 1;
            std::atomic<std::uint32_t> next{0};
            const std::function<void(unsigned)> job = [&](unsigned) {
                for (;;) {
                    const std::uint32_t q0 = next.fetch_add(32);
                    if (q0 >= nb) return;
                    for (std::uint32_t q = q0; q < std::min(nb, q0 + 32); ++q) {
                        const std::size_t bi = static_cast<std::size_t>(st.b0) + q;
                        const std::size_t e0 = static_cast<std::size_t>(out.batch[bi].chunk) * kEpl * kWave - base;
                        lane_rec* rec = out.rec.data() + bi * kWave;
                        for (std::uint32_t k = begin[q]; k < begin[q + 1]; ++k) {
                            const auto& x = open.rows[places[k].row];
                            const term* e = open.part[x.part].data() + x.off;
                            const int G = lanes_of(x.len), start = places[k].start;
                            int lg = 0;
                            while ((1 << lg) < G) ++lg;
                            for (std::uint32_t i = 0; i < x.len; ++i) {
                                const std::size_t at = e0 + static_cast<std::size_t>(i >> lg) * kWave +
                                                       static_cast<std::size_t>(start) + (i & static_cast<std::uint32_t>(G - 1));
                                piece.idx[at] = e[i].src;
                                piece.val[at] = e[i].coef;
                            }
                            for (int s = 0; s < G; ++s) {
                                const std::uint32_t nv = x.len > static_cast<std::uint32_t>(s)
                                                             ? (x.len - static_cast<std::uint32_t>(s) + static_cast<std::uint32_t>(G) - 1) >> lg : 0u;
                                rec[start + s] = {static_cast<std::int32_t>(row_at(p0 + places[k].row)),
                                                  static_cast<std::uint32_t>(lg) | static_cast<std::uint32_t>(s) << 3 | nv << 9};
                            }
                        }
                    }
                }
            };
            if (nb <= 32) job(0);
            else workers.run(job);
            st.nb = static_cast<int>(out.batch.size()) - st.b0;
        }
        if (end > first) out.steps.push_back(st);
        open.clear();
        level_bytes.clear();
        first = end;
        if (end < L) p0 = pos(end);
    };

    if (lo < L) p0 = pos(lo);
    bool usable = false;   // a level may join the open step
    double kept = 0.5;     // entries per summed term of the last level that joined or was tried in full
    double extra = 0.0;    // bytes the open step's levels cost more merged than on their own
    for (int l = lo; l < hi; ++l) {
        const std::uint32_t a = pos(l), b = pos(l + 1);
        long long own = b - a;
        std::size_t longest = 0;
        for (std::uint32_t t = a; t < b; ++t) {
            const std::size_t len = ptr[row_at(t) + 1] - ptr[row_at(t)];
            own += static_cast<long long>(len);
            longest = std::max(longest, len);
        }
        long long total = 0;
        const bool small = static_cast<double>(own) <= kLevelsOf * static_cast<double>(max_growth);
        if (l > first && usable && small) {
            const std::size_t from = open.rows.size();
            // The terms its substitution sums; a level whose entries, at the
            // share the last one kept, pass the limit is not tried.
            long long terms = 0;
            for (std::uint32_t t = a; t < b; ++t) {
                const std::uint32_t r = row_at(t);
                ++terms;
                for (std::uint32_t p = ptr[r]; p < ptr[r + 1]; ++p) {
                    const std::uint32_t j = static_cast<std::uint32_t>(idx[p]), pj = backward ? m - 1 - j : j;
                    if (pj < p0) ++terms;
                    else terms += open.rows[pj - p0].len > 0 ? open.rows[pj - p0].len : ptr[j + 1] - ptr[j] + 1;
                }
            }
            if (kept * static_cast<double>(terms) <= 1.1 * static_cast<double>(own + max_growth) &&
                expand_level(l, own + max_growth, total)) {
                kept = static_cast<double>(total) / static_cast<double>(terms);
                const double more = extra + merged_bytes(from) - own_bytes(l);
                if (more / kBytesPerUs < kLaunchUs * (l - first)) {
                    if (l == first + 1) expand_level(first, INT64_MAX / 4, total);
                    extra = more;
                    continue;
                }
                open.rows.resize(from);
            }
        }
        emit(l);
        usable = small && longest < kMaxRow;
        if (usable) {
            open.rows.assign(b - a, {0, 0, 0});
            extra = merged_bytes(0) - own_bytes(l);
        }
    }
    emit(hi);
    return out;
}

}  // namespace apxchol_amd
