"""Level tiles: consecutive launched levels in one launch, whose workgroups
recompute the rows they share.

Bar: the bits of the levels' own launches (APXCHOL_AMD_TILE_LEVELS=1), for
outputs of an application and of a solve, with 2, 3 and 4 levels a launch, on
factors whose levels have one row, part of a batch, several batches of mixed
row widths, and rows too long for the lane layout (which end a group), with
every level launched (tail levels of no batch) and with the default tail."""
import numpy as np
import pytest

import apxchol_amd as ax
from apxchol_amd import matgen as mg

pytestmark = pytest.mark.gpu

CASES = {
    "grid2d_7x5": lambda: mg.grid_laplacian((7, 5)),
    "grid2d_83x61": lambda: mg.grid_laplacian((83, 61), "lognormal"),
    "grid2d_150": lambda: mg.grid_laplacian((150, 150)),
    "sddm3d_19": lambda: mg.add_excess(mg.grid_laplacian((19, 19, 19), "lognormal")),
    "rmat_12": lambda: mg.rmat_laplacian(12),
}
_cache = {}


def case(name):
    if name not in _cache:
        A = CASES[name]()
        _cache[name] = (A, ax.factorize(A, seed=0))
    return _cache[name]


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("precision,fp16", [("fp64", False), ("fp32", False), ("fp32", True)])
@pytest.mark.parametrize("tail_batches", [1, 0])
def test_bits_of_the_levels_own_launches(gpu, name, precision, fp16, tail_batches, monkeypatch):
    import torch
    print(f"[case] level tiles {name} {precision} fp16={fp16} tail_batches={tail_batches}", flush=True)
    A, F = case(name)
    b = torch.tensor(mg.request_rhs(A, F.sddm, 3), device=gpu)
    monkeypatch.setenv("APXCHOL_AMD_TRAIL_ROWS", "0")   # every level is walked
    got, launches = [], []
    for levels in ("1", "2", "3", "4"):
        monkeypatch.setenv("APXCHOL_AMD_TILE_LEVELS", levels)
        s = ax.Solver(A, factor=F, precision=precision, fp16_storage=fp16, tail_batches=tail_batches)
        s.reset_apply_count()
        z = s.apply(b)
        r = s.solve(b, tol=1e-8, maxiter=60)
        torch.cuda.synchronize()
        got.append((z.clone(), r.x.clone(), r.iterations))
        launches.append(sum(s.info["level_launches"]))
        s.close()
    for z, x, it in got[1:]:
        assert it == got[0][2]
        assert torch.equal(z.view(torch.int64), got[0][0].view(torch.int64))
        assert torch.equal(x.view(torch.int64), got[0][1].view(torch.int64))
    if tail_batches == 1 and launches[0] > 40:
        assert launches[3] < launches[0]
