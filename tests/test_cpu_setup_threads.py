"""Solver setup where the process may start few threads or none: the merged
levels' team and the level tiles do the same work on those there are. A driver
built against the library replaces pthread_create by one that fails after a
given number of threads; the tables must equal those made with all threads, and
no failure may end the process."""
import subprocess
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
sys.path.insert(0, str(ROOT))

DRIVER = r"""
#include <cerrno>
#include <cstdio>
#include <cstring>
#include <dlfcn.h>
#include <pthread.h>
#include "apxchol_amd/csrc/host/gpu_solver.hpp"
#include "apxchol_amd/csrc/host/merge.hpp"
#include "apxchol_amd/csrc/host/threads.hpp"
#include "apxchol_amd/csrc/host/tile.hpp"
using namespace apxchol_amd;

static int allowed = 1 << 30;
extern "C" int pthread_create(pthread_t* t, const pthread_attr_t* a, void* (*f)(void*), void* arg) {
    static const auto real = reinterpret_cast<decltype(&pthread_create)>(dlsym(RTLD_NEXT, "pthread_create"));
    if (allowed <= 0) return EAGAIN;
    --allowed;
    return real(t, a, f, arg);
}

template <class T>
static bool same(const std::vector<T>& a, const std::vector<T>& b) {
    return a.size() == b.size() && (a.empty() || std::memcmp(a.data(), b.data(), a.size() * sizeof(T)) == 0);
}

int main() {
    // A 40 x 40 x 20 grid with a diagonal excess.
    const int X = 40, Y = 40, Z = 20, n = X * Y * Z;
    std::vector<std::int64_t> cp(n + 1, 0);
    std::vector<std::int32_t> ri;
    std::vector<double> v;
    for (int c = 0; c < n; ++c) {
        const int x = c % X, y = c / X % Y, z = c / X / Y;
        const int at[7] = {z > 0 ? c - X * Y : -1, y > 0 ? c - X : -1, x > 0 ? c - 1 : -1, c,
                           x + 1 < X ? c + 1 : -1, y + 1 < Y ? c + X : -1, z + 1 < Z ? c + X * Y : -1};
        double deg = 1e-3;
        for (int k = 0; k < 7; ++k) deg += k != 3 && at[k] >= 0;
        for (int k = 0; k < 7; ++k)
            if (at[k] >= 0) { ri.push_back(at[k]); v.push_back(k == 3 ? deg : -1.0); }
        cp[c + 1] = static_cast<std::int64_t>(ri.size());
    }
    csc_view A;
    A.n = n; A.colptr = cp.data(); A.rowidx = ri.data(); A.vals = v.data();
    const factorization F = factorize(A, factor_options{});
    trsv_factor T = prepare_trsv(F, false, -1.0);
    relabel_within_levels(T, F.perm, true);
    const batch_table bt = build_batches(T, false);
    const int L = static_cast<int>(T.level_ptr.size()) - 1;
    // Lane layout of the levels that fit it, and the first run of them.
    lane_tables lt;
    std::vector<int> lb(L, -1), pos(L + 1);
    for (int l = 0; l <= L; ++l) pos[l] = static_cast<int>(T.level_ptr[l]);
    int end = 0;
    for (int l = 0; l < L; ++l) {
        bool fits = true;
        for (std::uint32_t r = T.level_ptr[l]; r < T.level_ptr[l + 1]; ++r) fits = fits && T.f_ptr[r + 1] - T.f_ptr[r] <= 256;
        if (!fits) break;
        lb[l] = static_cast<int>(append_lane_level(T, bt, false, bt.level_first[l], bt.level_first[l + 1], lt));
        end = l + 1;
    }
    merge_tables m0;
    tile_tables t0;
    for (int few : {1 << 30, 0, 1, 2, 5}) {
        allowed = few;
        merge_tables m = build_merged_levels(T, false, 0, L * 2 / 3, bt.level_first, 100000);
        allowed = few;
        tile_tables t;
        append_tiles(lt, false, T.m, bt.level_first, lb, pos, 0, end, 4, t);
        allowed = few;
        int done[6] = {};
        side_by_side(6, [&](int k) { ++done[k]; });
        for (int k : done) if (k != 1) { std::printf("side_by_side: a job ran %d times\n", k); return 1; }
        try {
            side_by_side(6, [&](int k) { if (k == 3) throw std::runtime_error("x"); });
            std::printf("side_by_side: lost an exception\n");
            return 1;
        } catch (const std::runtime_error&) {
        }
        if (few == 1 << 30) {
            if (m.slots == 0 || t.batches < 4096) { std::printf("nothing to compare\n"); return 1; }
            m0 = std::move(m);
            t0 = std::move(t);
            continue;
        }
        bool ok = same(m.rec, m0.rec) && same(m.batch, m0.batch) && same(m.steps, m0.steps) && m.slots == m0.slots &&
                  m.pieces.size() == m0.pieces.size() && t.batches == t0.batches &&
                  t.steps.size() == t0.steps.size() && t.pieces.size() == t0.pieces.size();
        for (std::size_t k = 0; ok && k < m.pieces.size(); ++k)
            ok = same(m.pieces[k].idx, m0.pieces[k].idx) && same(m.pieces[k].val, m0.pieces[k].val);
        for (std::size_t k = 0; ok && k < t.pieces.size(); ++k) {
            const std::size_t nb = t.pieces[k].batches;
            ok = nb == t0.pieces[k].batches &&
                 std::memcmp(t.pieces[k].rec.get(), t0.pieces[k].rec.get(), nb * kWave * sizeof(lane_rec)) == 0 &&
                 std::memcmp(t.pieces[k].ent.get(), t0.pieces[k].ent.get(), nb * kWave * kEpl * sizeof(entry32)) == 0;
        }
        for (std::size_t k = 0; ok && k < t.steps.size(); ++k)
            ok = t.steps[k].level == t0.steps[k].level && t.steps[k].levels == t0.steps[k].levels &&
                 t.steps[k].tiles == t0.steps[k].tiles && t.steps[k].slots == t0.steps[k].slots;
        std::printf("%d threads: %s\n", few, ok ? "same" : "DIFFERENT");
        if (!ok) return 1;
    }
    std::printf("OK\n");
    return 0;
}
"""


def test_tables_do_not_need_the_threads(tmp_path):
    from apxchol_amd import build as b
    if not b.LIB.exists():
        pytest.fail(f"{b.LIB} is missing: build it first")
    src, exe = tmp_path / "threads.cpp", tmp_path / "threads"
    src.write_text(DRIVER)
    r = subprocess.run([str(b.ROCM / "llvm" / "bin" / "clang++"), *b.HOST_FLAGS, f"-I{ROOT}", str(src), "-o", str(exe),
                        "-rdynamic", f"-L{b.LIB.parent}", "-lapxchol_amd", f"-Wl,-rpath,{b.LIB.parent}",
                        f"-L{b.ROCM}/lib", "-lamdhip64", f"-Wl,-rpath,{b.ROCM}/lib", "-lpthread", "-ldl"],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-3000:]
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout.strip().endswith("OK"), (out.returncode, out.stdout[-2000:], out.stderr[-2000:])
