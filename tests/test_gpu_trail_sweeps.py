"""Whole sweeps (Solver.sweep) of a factor whose applications use a trailing
block and merged levels run as those of a factor without: as many launches and
tail runs, the same bits."""
import numpy as np
import pytest

import apxchol_amd as ax
from apxchol_amd import matgen as mg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["sddm3d_20", "grid3d_25", "rmat_13"])
def test_whole_sweeps_are_those_without_a_block(gpu, name, monkeypatch):
    import torch
    print(f"[case] whole sweeps {name}", flush=True)
    A, _ = mg.workload(name)
    F = ax.factorize(A, seed=0)
    monkeypatch.setenv("APXCHOL_AMD_TILE_LEVELS", "1")
    s = ax.Solver(A, factor=F)
    monkeypatch.setenv("APXCHOL_AMD_TRAIL_ROWS", "0")
    plain = ax.Solver(A, factor=F)
    assert s.info["block"]["rows"] > 0 and s.info["block"]["tail_runs"] == [0, 0]
    assert s.info["tail_runs"] == plain.info["tail_runs"]
    assert s.info["level_launches"] == plain.info["level_launches"]
    r = torch.tensor(np.random.default_rng(4).standard_normal(s.m), device=gpu)
    for backward in (False, True):
        out = [torch.empty_like(r), torch.empty_like(r)]
        s.sweep(r, out[0], backward)
        plain.sweep(r, out[1], backward)
        torch.cuda.synchronize()
        assert torch.equal(out[0].view(torch.int64), out[1].view(torch.int64))
    s.close()
    plain.close()
