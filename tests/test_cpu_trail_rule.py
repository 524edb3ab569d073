"""When the trailing block may be applied through its explicit inverse
(host/trail.cpp, trail_is_sound), on the CPU, against the dense block.

The host function is called on the library's own factors: well-conditioned
graphs, two R-MAT graphs joined by one edge of weight 1 to 1e-6, and slightly
regularised Laplacians. With S = (T T^t)^-1 and D = sqrt(diag S) from dense
fp64 arithmetic, an accepted block satisfies the bound the rule promises,
sqrt(n) |D T|^2 <= 65536, and its fp32 rounding keeps the least eigenvalue of
D^-1 S D^-1 (to the 65536 / 2^24 of it that the bound allows); a block a
factor four inside the bound is accepted; where the rounded S is indefinite
it is refused."""
import ctypes
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest
import scipy.linalg as sl
import scipy.sparse as sp
import scipy.sparse.csgraph as csg

ROOT = Path(__file__).resolve().parents[1]
sys.path.insert(0, str(ROOT))

from apxchol_amd import matgen as mg  # noqa: E402

LIMIT = 65536.0

SHIM = r"""
#include <cstring>
#include "apxchol_amd/csrc/host/trail.hpp"
using namespace apxchol_amd;
static trsv_factor T;
static std::uint32_t first;
// The trailing levels of at most `rows` rows, relabelled as the solver does.
extern "C" int prepare(long n, const std::int64_t* cp, const std::int32_t* ri, const double* v, int fp16, int rows) {
    csc_view A;
    A.n = n; A.colptr = cp; A.rowidx = ri; A.vals = v;
    const factorization F = factorize(A, factor_options{});
    T = prepare_trsv(F, fp16 != 0, -1.0);
    relabel_within_levels(T, F.perm, true);
    first = T.m;
    for (std::size_t l = T.level_ptr.size() - 1; l-- > 0 && T.m - T.level_ptr[l] <= static_cast<std::uint32_t>(rows);)
        first = T.level_ptr[l];
    return static_cast<int>(T.m - first);
}
// The block, row by row, its columns times sqrt of the storage's scales.
extern "C" void dense(double* t) {
    const std::size_t n = T.m - first;
    std::memset(t, 0, n * n * sizeof(double));
    const auto scale = [&](std::uint32_t j) { return T.fp16 ? 1.0 / static_cast<double>(T.inv_scale[first + j]) : 1.0; };
    for (std::uint32_t i = 0; i < n; ++i) {
        for (std::uint32_t p = T.f_ptr[first + i]; p < T.f_ptr[first + i + 1]; ++p)
            if (static_cast<std::uint32_t>(T.f_idx[p]) >= first)
                t[i * n + T.f_idx[p] - first] = scale(T.f_idx[p] - first) * (T.fp16 ? fp16_widen(T.f_h[p]) : T.f_val[p]);
        t[i * n + i] = scale(i) * T.diag[first + i];
    }
}
extern "C" int sound(const double* s_diag) {
    return trail_is_sound(T, first, std::vector<double>(s_diag, s_diag + (T.m - first)));
}
"""


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    from apxchol_amd import build as b
    if not b.LIB.exists():
        pytest.fail(f"{b.LIB} is missing: build it first")
    tmp = tmp_path_factory.mktemp("trail_rule")
    src, so = tmp / "shim.cpp", tmp / "shim.so"
    src.write_text(SHIM)
    r = subprocess.run([str(b.ROCM / "llvm" / "bin" / "clang++"), *b.HOST_FLAGS, "-shared", f"-I{ROOT}", str(src),
                        "-o", str(so), f"-L{b.LIB.parent}", "-lapxchol_amd", f"-Wl,-rpath,{b.LIB.parent}"],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-3000:]
    return ctypes.CDLL(str(so))


def joined(A, w):
    """Two copies of A joined at their largest vertices by an edge of weight w."""
    n = A.shape[0]
    k = int(np.argmax(np.diff(A.indptr)))
    B = sp.block_diag([A, A]).tolil()
    for i, j in ((k, n + k), (n + k, k)):
        B[i, j] -= w
        B[i, i] += w
    return B.tocsc()


def giant(A):
    lab = csg.connected_components(A, directed=False)[1]
    i = np.flatnonzero(lab == np.argmax(np.bincount(lab)))
    return A[i][:, i].tocsc()


def rmat():
    return giant(mg.rmat_laplacian(11))


def one_entry():
    A = rmat().tolil()
    A[5, 5] += 1e-4
    return A.tocsc()


GOOD = {
    "rmat_11": rmat,
    "grid3d_16": lambda: mg.grid_laplacian((16, 16, 16)),
    "sddm3d_16": lambda: mg.add_excess(mg.grid_laplacian((16, 16, 16), "lognormal")),
    "aniso3d_14": lambda: mg.workload("aniso3d_14")[0],
    "grid2d_61": lambda: mg.grid_laplacian((61, 61)),
}
SOFT = {f"pair_{w:g}": (lambda w=w: joined(rmat(), w)) for w in (1.0, 1e-1, 1e-2, 1e-3, 1e-4, 1e-6)}
SOFT |= {f"plus_{e:g}": (lambda e=e: (rmat() + e * sp.eye(rmat().shape[0])).tocsc()) for e in (1e-1, 1e-3, 1e-6, 1e-8)}
SOFT |= {"excess_1e-9": lambda: mg.add_excess(rmat(), 1e-9), "one_entry_1e-4": one_entry}


_cache = {}


def block(host, name, fp16):
    """(T, S, accepted) of a graph's trailing block."""
    if (name, fp16) not in _cache:
        _cache[name, fp16] = _block(host, (GOOD | SOFT)[name](), fp16)
    return _cache[name, fp16]


def _block(host, A, fp16):
    A = sp.csc_matrix(A)
    A.sort_indices()
    cp, ri, v = A.indptr.astype(np.int64), A.indices.astype(np.int32), A.data.astype(np.float64)
    p = lambda a: a.ctypes.data_as(ctypes.c_void_p)
    n = host.prepare(ctypes.c_long(A.shape[0]), p(cp), p(ri), p(v), int(fp16), A.shape[0] // 6)
    T = np.zeros((n, n))
    host.dense(p(T))
    X = sl.solve_triangular(T, np.eye(n), lower=True)
    S = X.T @ X
    accepted = bool(host.sound(p(np.ascontiguousarray(np.diag(S)))))
    return T, S, accepted


@pytest.mark.parametrize("fp16", [False, True])
@pytest.mark.parametrize("name", [*GOOD, *SOFT])
def test_accepted_blocks_survive_their_rounding(host, name, fp16):
    T, S, accepted = block(host, name, fp16)
    n = len(T)
    assert n > 50
    d = np.sqrt(np.diag(S))
    spread = np.sqrt(n) * np.linalg.norm(d[:, None] * T, 2) ** 2
    least = 1.0 / np.linalg.norm(d[:, None] * T, 2) ** 2      # of D^-1 S D^-1
    rounded = np.linalg.eigvalsh(S.astype(np.float32).astype(np.float64) / d[:, None] / d[None, :])[0]
    assert accepted or name in SOFT
    if accepted:
        assert spread <= LIMIT
        assert abs(rounded - least) <= LIMIT / 2**24 * least + 1e-12
    if spread <= LIMIT / 4:
        assert accepted
    if rounded < 0.5 * least:
        assert not accepted


def test_weak_links_and_slight_regularisations_are_refused(host):
    refused = [name for name in SOFT if not block(host, name, False)[2]]
    assert {"pair_0.001", "pair_0.0001", "pair_1e-06", "plus_1e-06", "plus_1e-08", "excess_1e-9",
            "one_entry_1e-4"} <= set(refused)


def test_a_diagonal_out_of_range_is_refused(host):
    T, S, accepted = _block(host, GOOD["rmat_11"](), False)
    assert accepted
    for bad in (np.inf, np.nan, 0.0, -1.0):
        d = np.diag(S).copy()
        d[len(d) // 2] = bad
        assert host.sound(d.ctypes.data_as(ctypes.c_void_p)) == 0
