"""Device memory that a solver and a serving lane report: what the budget of a
server is compared with."""
import numpy as np
import pytest

import apxchol_amd as ax
from apxchol_amd import matgen as mg

pytestmark = pytest.mark.gpu


def test_device_bytes_hold_the_level_tiles(gpu, monkeypatch):
    """The tiles' layout is 2,560 bytes a batch (64 records of 8 bytes, 4 x 64
    entries of 8 bytes): at least that for every batch they cover."""
    import torch
    print("[case] device bytes with level tiles", flush=True)
    A = mg.grid_laplacian((150, 150))
    F = ax.factorize(A, seed=0)
    b = torch.tensor(mg.request_rhs(A, F.sddm, 0), device=gpu)
    bytes_, launches = [], []
    for levels in ("1", "4"):
        monkeypatch.setenv("APXCHOL_AMD_TILE_LEVELS", levels)
        s = ax.Solver(A, factor=F)
        s.solve(b, tol=1e-8)
        torch.cuda.synchronize()
        bytes_.append(s.info["device_bytes"])
        launches.append(sum(s.info["level_launches"]))
        s.close()
    assert launches[1] < launches[0]
    assert bytes_[1] - bytes_[0] >= 2560 * 2 * (launches[0] - launches[1])


def test_server_charges_every_block_buffer(gpu):
    """n-vectors: r, x, p, Ap, y, z, b, x of each block, b, x of the single
    lane; the trailing block's input and 2 x 2304 partials a column."""
    print("[case] server memory", flush=True)
    A = mg.rmat_laplacian(13)
    n = A.shape[0]
    s = ax.Solver(A, seed=0)
    assert s.info["block"]["rows"] > 0
    for slots, narrow in ((32, 4), (8, 0)):
        o = ax.Solver(A, seed=0)
        srv = ax.Server(slots=slots, narrow_slots=narrow)
        srv.add(o)
        columns = slots + narrow
        used = srv.stats()["memory_used"]
        assert used == o.info["device_bytes"] + 8 * (columns * (8 * n + s.info["block"]["rows"] + 2 * 2304) + 2 * n)
        srv.close()
        small = ax.Server(slots=slots, narrow_slots=narrow, memory_budget=used - 1)
        with pytest.raises(RuntimeError, match="memory budget"):
            small.add(ax.Solver(A, seed=0))
        small.close()
        o.close()
    s.close()


def _bits(t):
    import torch
    return t.view(torch.int64)


@pytest.mark.parametrize("graph", ["rmat", "grid3d", "grid2d"])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_without_memory_for_the_extra_forms_levels_are_walked(gpu, graph, precision, monkeypatch):
    """No room for the trailing block, the merged levels and the tiles (as a
    full device would leave): the solver is made all the same and gives the bits
    of one that is told to do without them."""
    import torch
    print(f"[case] no extra memory {graph} {precision}", flush=True)
    A = {"rmat": lambda: mg.rmat_laplacian(12), "grid3d": lambda: mg.grid_laplacian((14, 13, 12)),
         "grid2d": lambda: mg.grid_laplacian((70, 60))}[graph]()
    F = ax.factorize(A, seed=0)
    b = torch.tensor(mg.request_rhs(A, F.sddm, 1), device=gpu)
    monkeypatch.setenv("APXCHOL_AMD_EXTRA_BYTES", "0")
    s = ax.Solver(A, factor=F, precision=precision)
    monkeypatch.delenv("APXCHOL_AMD_EXTRA_BYTES")
    for name, value in (("TRAIL_ROWS", "0"), ("MERGE_GROWTH", "0"), ("TILE_LEVELS", "1")):
        monkeypatch.setenv(f"APXCHOL_AMD_{name}", value)
    plain = ax.Solver(A, factor=F, precision=precision)
    z, zp = s.apply(b).clone(), plain.apply(b).clone()
    r, rp = s.solve(b, tol=1e-8), plain.solve(b, tol=1e-8)
    torch.cuda.synchronize()
    assert s.info["block"] == plain.info["block"] and s.info["block"]["rows"] == 0
    assert s.info["device_bytes"] == plain.info["device_bytes"]
    assert r.iterations == rp.iterations and r.status == 1
    assert torch.equal(_bits(z), _bits(zp)) and torch.equal(_bits(r.x), _bits(rp.x))


def test_without_memory_for_merged_levels_the_block_stays(gpu, monkeypatch):
    """Room for a block of up to 64 rows (100 KB with its setup), not for the
    merged levels (more than 1 MB)."""
    import torch
    print("[case] no memory for merged levels", flush=True)
    A = mg.add_excess(mg.grid_laplacian((16, 16, 16), "lognormal"))
    F = ax.factorize(A, seed=0)
    b = torch.tensor(mg.rhs(A.shape[0], 2), device=gpu)
    monkeypatch.setenv("APXCHOL_AMD_TRAIL_ROWS", "64")
    monkeypatch.setenv("APXCHOL_AMD_MERGE_GROWTH", "4000")
    monkeypatch.setenv("APXCHOL_AMD_TILE_LEVELS", "1")
    full = ax.Solver(A, factor=F)
    monkeypatch.setenv("APXCHOL_AMD_EXTRA_BYTES", "1000000")
    s = ax.Solver(A, factor=F)
    monkeypatch.delenv("APXCHOL_AMD_EXTRA_BYTES")
    monkeypatch.setenv("APXCHOL_AMD_MERGE_GROWTH", "0")
    plain = ax.Solver(A, factor=F)
    assert full.info["block"]["rows"] == s.info["block"]["rows"] > 0
    assert s.info["block"] == plain.info["block"] != full.info["block"]
    assert torch.equal(_bits(s.apply(b).clone()), _bits(plain.apply(b).clone()))
