"""The trailing block of an application (the last rows of the factor through
their explicit inverse) at the sizes where it can go wrong: none, one row,
around the 16 / 32 rows of a product workgroup, around the 64-row tiles of its
setup (a last doubling step of one tile), the whole factor, and hub rows whose
coupling a workgroup sums (R-MAT).

Bars, those of the sweeps it replaces: fp64 applications within 1e-12 of the
oracle, fp32 within 1e-6 (max norm; 1e-5 against the same fp16 storage), all
schedules, every column of a blocked application and every member of a group
the bits of the single application."""
import numpy as np
import pytest

import apxchol_amd as ax
import oracle
from apxchol_amd import matgen as mg

pytestmark = pytest.mark.gpu

CASES = {
    "sddm3d_16": lambda: mg.add_excess(mg.grid_laplacian((16, 16, 16), "lognormal")),
    "grid2d_61": lambda: mg.grid_laplacian((61, 61)),
    "rmat_13": lambda: mg.rmat_laplacian(13),
}
ROWS = [0, 1, 15, 16, 17, 33, 64, 65, 129, 200, 449, 1025, 8192]
_cache = {}


def case(name):
    if name not in _cache:
        A = CASES[name]()
        F = ax.factorize(A, seed=0)
        _cache[name] = (A, F, F.export())
    return _cache[name]


def bits(a):
    return np.ascontiguousarray(a).view(np.int64)


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("rows", ROWS)
def test_block_rows_match_oracle_and_all_paths_agree(gpu, name, rows, monkeypatch):
    import torch
    print(f"[case] trailing block {name} rows={rows}", flush=True)
    A, F, fac = case(name)
    n = A.shape[0]
    monkeypatch.setenv("APXCHOL_AMD_TRAIL_ROWS", str(rows))
    R = np.random.default_rng(rows).standard_normal((3, n))
    Rd = torch.tensor(R, device=gpu)
    for precision, fp16 in (("fp64", False), ("fp32", False), ("fp64", True), ("fp32", True)):
        ref = [oracle.Oracle(A, fac, F.sddm, fp16=fp16).apply(r) for r in R]
        s = ax.Solver(A, factor=F, precision=precision, fp16_storage=fp16)
        assert s.info["block"]["rows"] <= rows
        if rows >= 15:
            assert s.info["block"]["rows"] > 0
        s.reset_apply_count()
        Z = s.apply_batch(Rd).cpu().numpy()
        one = []
        for c in range(3):
            s.reset_apply_count()
            z = s.apply(Rd[c].clone()).cpu().numpy()
            assert np.array_equal(bits(z), bits(Z[c])), (precision, fp16, c)
            tol = 1e-12 if precision == "fp64" else 1e-5 if fp16 else 1e-6
            err = np.max(np.abs(z - ref[c])) / np.max(np.abs(ref[c]))
            assert err < tol, (precision, fp16, c, err)
            one.append(z)
        for schedule in ("levels", "dataflow"):
            o = ax.Solver(A, factor=F, precision=precision, fp16_storage=fp16, schedule=schedule)
            assert o.info["block"]["rows"] == s.info["block"]["rows"]
            z = o.apply(Rd[0].clone()).cpu().numpy()
            assert np.array_equal(bits(z), bits(one[0])), (precision, fp16, schedule)
            o.close()
        s.close()


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("growth", [0, 1, 300, 4000, 10_000_000])
def test_merged_levels_match_oracle_and_all_paths_agree(gpu, name, growth, monkeypatch):
    """The levels outside the block, merged from not at all to all into one
    launch (rows of several chunks of 256 entries)."""
    import torch
    print(f"[case] merged levels {name} growth={growth}", flush=True)
    A, F, fac = case(name)
    monkeypatch.setenv("APXCHOL_AMD_TRAIL_ROWS", "64")
    monkeypatch.setenv("APXCHOL_AMD_MERGE_GROWTH", str(growth))
    R = np.random.default_rng(growth % 97).standard_normal((6, A.shape[0]))
    Rd = torch.tensor(R, device=gpu)
    solvers = []
    for precision, fp16 in (("fp64", False), ("fp32", False), ("fp64", True), ("fp32", True)):
        s = ax.Solver(A, factor=F, precision=precision, fp16_storage=fp16)
        blk = s.info["block"]
        assert 0 < blk["rows"] <= 64
        if growth > 0 and precision == "fp64":
            assert blk["tail_runs"] == [0, 0]
        if growth == 10_000_000 and precision == "fp64":
            assert max(blk["level_launches"]) < 0.5 * s.info["levels"]
        s.reset_apply_count()
        Z = s.apply_batch(Rd).cpu().numpy()
        tol = 1e-12 if precision == "fp64" else 1e-5 if fp16 else 1e-6
        for c in range(6):
            s.reset_apply_count()
            z = s.apply(Rd[c].clone()).cpu().numpy()
            assert np.array_equal(bits(z), bits(Z[c])), (precision, fp16, c)
            if c < 2:
                ref = oracle.Oracle(A, fac, F.sddm, fp16=fp16).apply(R[c])
                err = np.max(np.abs(z - ref)) / np.max(np.abs(ref))
                assert err < tol, (precision, fp16, c, err)
        for schedule in ("levels", "dataflow"):
            o = ax.Solver(A, factor=F, precision=precision, fp16_storage=fp16, schedule=schedule)
            z = o.apply(Rd[0].clone()).cpu().numpy()
            assert np.array_equal(bits(z), bits(Z[0])), (precision, fp16, schedule)
            o.close()
        if not fp16:
            solvers.append((precision, s))
        else:
            s.close()
    b = torch.tensor(mg.request_rhs(A, F.sddm, 5), device=gpu)
    for precision, s in solvers:
        one = ax.Group([s])
        xs, rs = one.solve([b], tol=1e-8, maxiter=200)
        own = s.solve(b, tol=1e-8, maxiter=200)
        torch.cuda.synchronize()
        assert rs[0].status == 1 and torch.equal(xs[0].view(torch.int64), own.x.view(torch.int64)), precision
        one.close()
        s.close()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("k", [1, 2, 8, 17, 33, 64])
def test_block_columns_have_the_single_bits(gpu, precision, k):
    """Every width of the blocked product (1 to 8 columns a workgroup, several
    column tiles)."""
    import torch
    print(f"[case] trailing block columns {precision} k={k}", flush=True)
    A, F, _ = case("rmat_13")
    s = ax.Solver(A, factor=F, precision=precision)
    assert s.info["block"]["rows"] > 0
    R = torch.tensor(np.random.default_rng(k).standard_normal((k, A.shape[0])), device=gpu)
    s.reset_apply_count()
    Z = s.apply_batch(R).cpu().numpy()          # application 1: no centring
    for c in range(k):
        s.reset_apply_count()
        assert np.array_equal(bits(s.apply(R[c].clone()).cpu().numpy()), bits(Z[c])), c
    s.close()


def test_group_mixes_members_with_and_without_a_block(gpu, monkeypatch):
    import torch
    print("[case] trailing block in a group", flush=True)
    solvers, bs = [], []
    for i, (name, rows) in enumerate((("sddm3d_16", "0"), ("grid2d_61", "300"), ("rmat_13", "1500"),
                                      ("sddm3d_16", "8192"))):
        A, F, _ = case(name)
        monkeypatch.setenv("APXCHOL_AMD_TRAIL_ROWS", rows)
        solvers.append(ax.Solver(A, factor=F, precision="fp32"))
        bs.append(torch.tensor(mg.request_rhs(A, F.sddm, 70 + i), device=gpu))
    g = ax.Group(solvers)
    xs, rs = g.solve(bs, tol=1e-8, maxiter=200)
    torch.cuda.synchronize()
    for i, s in enumerate(solvers):
        own = s.solve(bs[i], tol=1e-8, maxiter=200)
        torch.cuda.synchronize()
        assert (rs[i].status, rs[i].iterations) == (1, own.iterations), i
        assert torch.equal(xs[i].view(torch.int64), own.x.view(torch.int64)), i
    g.close()
    for s in solvers:
        s.close()
