#include "trail.hpp"

#include <algorithm>
#include <cmath>
#include <stdexcept>

namespace apxchol_amd {

namespace {

// What one level costs a sweep, in microseconds (graph replay): a launched
// level 5.2 with the gap before the next launch, a level inside a one-workgroup
// tail run 0.6 plus 0.02 per batch. Levels of up to 48 batches and 2048 rows
// are walked.
double level_cost(std::uint32_t rows, int batches) {
    return batches <= 48 && rows < 2048 ? 0.6 + 0.02 * batches : 5.2;
}

// The product reads n^2 values at about 5 TB/s; the coupling and product
// launches cost 8 us; forming S takes n^3 / 2e7 us once, spread over the 250
// applications of ten solves. Solves at other block sizes (whole solve, us,
// and rows of the block): 48^3 grid fp64 8,266 at 1,467, 6,779 at 3,773,
// 8,057 at 7,650; 89^3 fp64 13,058 at 1,962, 11,864 at 3,905, 12,978 at
// 8,167; R-MAT s18 mixed 12,476 at 4,094, 9,320 at 8,176.
constexpr double kProductBytesPerUs = 5.0e6;
constexpr double kProductFixedUs = 8.0;
constexpr double kFormPerUs = 2.0e7;
constexpr double kFormShare = 250.0;

// Small factors are solved many at a time (a launch then serves all members of
// a group, but every member reads its own S): at most a sixth of the rows.
constexpr std::uint32_t kMinFactorPerBlock = 6;

// Off-diagonals a row from which the block is used, by the width of the
// sweeps' vectors. Conjugate gradients amplify the rounding of an application
// on some factors, and a solve to 1e-8 then differs between the two forms,
// which agree to 1e-15 (fp64) or 1e-7 (fp32) themselves:
// * fp64: 2-D grids (3.9 .. 4.5 a row) by up to 2e-9, or by an iteration (two
//   of eight sides from 24 to 1000); 3-D grids (5.7 .. 8.5) and R-MAT graphs
//   (11 .. 31) by less than 1e-13;
// * fp32: 2-D grids by up to 2e-9, 3-D grids by up to 3e-7 of x's rms at a
//   single vertex (128^3); R-MAT graphs by less than 1e-10.
// The factors below the line walk every level as before. They gain least: a
// 100^2 mixed solve 3.28 -> 2.45 ms, 256^2 fp64 7.2 -> 5.3, 128^3 mixed 28.9 ->
// 18.2, against R-MAT s18 mixed 42.8 -> 9.8 and 89^3 fp64 18.6 -> 11.8.
constexpr std::uint64_t kMinPerRow64 = 5, kMinPerRow32 = 10;

// Largest sqrt(n) |D T|^2 of a block (trail_is_sound). A weak link between
// clusters or a slight regularisation leaves S a large, nearly constant part,
// whose rounding hides S's small eigenvalues; the walk, which rounds each row
// once, is off by the square root of this only. The largest component of an
// R-MAT graph of scale 11 (alone, with e on the diagonal, two of it joined by
// an edge of weight w): sqrt(n) |D T|^2, the least eigenvalue of D^-1 S D^-1
// exact and rounded to fp32, and iterations of mixed solves (N(0,1) projected,
// 1e-8) walked and with S:
//   alone            127     0.374    0.374
//   e = 1e-2       9,800   5.1e-3   5.1e-3     11, 11, 11   11, 11, 11
//   w = 1          2.4e5   2.7e-4   2.7e-4     13, 12, 11   12, 12, 11
//   w = 1e-2       2.4e7  2.68e-6  2.67e-6     13, 12, 12   13, 12, 12
//   e = 1e-6       1.0e8   4.4e-7  -8.2e-8     11, 10, 11   22, 22, 18
//   w = 1e-3       2.4e8   2.7e-7  -2.5e-8     68, 13, 11   none converges
//   e = 1e-8       1.0e10  4.4e-9  -2.9e-6     13, 13, 13   none converges
// fp64 solves keep their iterations, but an application is further off: at the
// limit S may be 7e-12 off (fp32: 0.4 %). Energy-norm errors of an application
// to T times N(0,1), walked and with S: R-MAT s18 (13,000) 3e-15 / 3e-13,
// w = 1 3e-15 / 3e-12, w = 1e-4 2e-13 / 2e-8. Blocks of grids (2-D up to
// 1000, 3-D up to 112, anisotropic up to 80) have up to 3,300, of R-MAT graphs
// of scale 11 to 22 up to 14,000.
constexpr double kMaxSpread = 65536.0;
constexpr int kSpreadSteps = 8;

}  // namespace

std::size_t choose_trail_level(const trsv_factor& T, int value_bytes, const std::vector<int>& fwd_first,
                               const std::vector<int>& bck_first, int max_rows) {
    const std::size_t L = T.level_ptr.empty() ? 0 : T.level_ptr.size() - 1;
    if (fwd_first.size() != L + 1 || bck_first.size() != L + 1)
        throw std::runtime_error("apxchol_amd: level tables of the trailing block");
    const std::uint32_t cap = max_rows < 0 ? std::min(static_cast<std::uint32_t>(kTrailMaxRows), T.m / kMinFactorPerBlock)
                                           : static_cast<std::uint32_t>(std::min(max_rows, kTrailMaxRows));
    if (max_rows < 0 && T.offdiag() < (value_bytes == 8 ? kMinPerRow64 : kMinPerRow32) * T.m) return L;
    std::size_t best = L;
    double gain = 0.0, best_net = 0.0;
    for (std::size_t l = L; l-- > 0;) {
        const std::uint32_t rows = T.level_ptr[l + 1] - T.level_ptr[l];
        const std::uint32_t n = T.m - T.level_ptr[l];
        if (n > cap) break;
        if (max_rows >= 0) {
            best = l;
            continue;
        }
        const std::size_t b = L - 1 - l;   // the level's place in the back sweep
        gain += level_cost(rows, fwd_first[l + 1] - fwd_first[l]) + level_cost(rows, bck_first[b + 1] - bck_first[b]);
        const double dn = static_cast<double>(n);
        const double cost = kProductFixedUs + dn * dn * value_bytes / kProductBytesPerUs +
                            dn * dn * dn / kFormPerUs / kFormShare;
        if (gain - cost > best_net) {
            best_net = gain - cost;
            best = l;
        }
    }
    return best;
}

// With D = sqrt(diag S) every |S_ij| is at most D_i D_j, so the rounding moves
// x^T S x by at most u sqrt(n) |D x|^2 (its n^2 errors being independent), and
// x^T S x is at least |D x|^2 / |D T|^2. The product of the two, u sqrt(n)
// |D T|^2, bounds the relative change of the operator in its own norm. |D T|^2
// is at most the largest eigenvalue of B B^T with B = |D T|, hence at most
// max_i (B B^T v)_i / v_i for any v > 0: a few steps from v = 1 come within a
// tenth of it.
bool trail_is_sound(const trsv_factor& T, std::uint32_t first, const std::vector<double>& s_diag) {
    const std::uint32_t n = T.m - first;
    if (s_diag.size() < n) throw std::runtime_error("apxchol_amd: diagonal of the trailing block");
    // B's rows: the block's entries, the diagonal last (columns of T over
    // sqrt(W) where W is not 1).
    std::vector<std::size_t> at(n + 1, 0);
    std::vector<std::uint32_t> col;
    std::vector<double> val;
    for (std::uint32_t i = 0; i < n; ++i) {
        if (!(s_diag[i] > 0.0) || !std::isfinite(s_diag[i])) return false;
        const double d = std::sqrt(s_diag[i]);
        const auto add = [&](std::uint32_t j, double v) {
            col.push_back(j);
            val.push_back(d * std::fabs(v) / (T.inv_scale.empty() ? 1.0 : static_cast<double>(T.inv_scale[first + j])));
        };
        for (std::uint32_t p = T.f_ptr[first + i]; p < T.f_ptr[first + i + 1]; ++p)
            if (static_cast<std::uint32_t>(T.f_idx[p]) >= first)
                add(static_cast<std::uint32_t>(T.f_idx[p]) - first, T.fp16 ? fp16_widen(T.f_h[p]) : T.f_val[p]);
        add(i, T.diag[first + i]);
        at[i + 1] = col.size();
    }
    std::vector<double> v(n, 1.0), w(n), t(n);
    for (int step = 0; step < kSpreadSteps; ++step) {
        std::fill(w.begin(), w.end(), 0.0);
        for (std::uint32_t i = 0; i < n; ++i)
            for (std::size_t k = at[i]; k < at[i + 1]; ++k) w[col[k]] += val[k] * v[i];
        double most = 0.0, top = 0.0;
        for (std::uint32_t i = 0; i < n; ++i) {
            t[i] = 0.0;
            for (std::size_t k = at[i]; k < at[i + 1]; ++k) t[i] += val[k] * w[col[k]];
            const double q = t[i] / v[i];
            if (!std::isfinite(q)) return false;
            most = std::max(most, q);
            top = std::max(top, t[i]);
        }
        if (std::sqrt(static_cast<double>(n)) * most <= kMaxSpread) return true;
        // (Rows a step leaves far behind would divide by nothing.)
        for (std::uint32_t i = 0; i < n; ++i) v[i] = std::max(t[i] / top, 1e-30);
    }
    return false;
}

trail_couple_tables build_trail_couple(const trsv_factor& T, std::uint32_t first) {
    trail_couple_tables t;
    lane_rec rec[kWave];
    entry32 ent[kEpl][kWave];
    int used = 0;   // lanes of the open batch
    const auto close = [&] {
        if (used == 0) return;
        for (int lane = used; lane < kWave; ++lane) {
            rec[lane] = {-1, 0u};
            for (int k = 0; k < kEpl; ++k) ent[k][lane] = {0, 0.0f};
        }
        t.rec.insert(t.rec.end(), rec, rec + kWave);
        for (int k = 0; k < kEpl; ++k) t.ent.insert(t.ent.end(), ent[k], ent[k] + kWave);
        ++t.batches;
        used = 0;
    };
    for (std::uint32_t row = first; row < T.m; ++row) {
        const std::uint32_t b = T.f_ptr[row], e = T.f_ptr[row + 1];
        // Columns ascend: the entries before the block are a prefix.
        const auto end = std::partition_point(T.f_idx.begin() + b, T.f_idx.begin() + e, [&](std::int32_t j) {
            return static_cast<std::uint32_t>(j) < first;
        });
        const std::uint32_t len = static_cast<std::uint32_t>(end - (T.f_idx.begin() + b));
        if (len > static_cast<std::uint32_t>(kWave * kEpl)) {
            t.longrow.push_back(int4{static_cast<int>(row - first), static_cast<int>(b), static_cast<int>(len), 0});
            continue;
        }
        int lg = 0;
        while (static_cast<std::uint32_t>(kEpl << lg) < len) ++lg;
        const int G = 1 << lg;
        const int at = (used + G - 1) / G * G;   // groups are aligned to their size
        if (at + G > kWave) close();
        const int start = (used + G - 1) / G * G;
        for (int lane = used; lane < start; ++lane) {
            rec[lane] = {-1, 0u};
            for (int k = 0; k < kEpl; ++k) ent[k][lane] = {0, 0.0f};
        }
        for (int s = 0; s < G; ++s) {
            std::uint32_t nv = 0;
            for (int k = 0; k < kEpl; ++k) {
                const std::uint32_t q = static_cast<std::uint32_t>(s + k * G);
                ent[k][start + s] = {0, 0.0f};
                if (q >= len) continue;
                ent[k][start + s] = {T.f_idx[b + q], T.fp16 ? fp16_widen(T.f_h[b + q]) : T.f_val[b + q]};
                ++nv;
            }
            rec[start + s] = {static_cast<std::int32_t>(row - first),
                              static_cast<std::uint32_t>(lg) | static_cast<std::uint32_t>(s) << 3 | nv << 9};
        }
        used = start + G;
    }
    close();
    return t;
}

}  // namespace apxchol_amd
