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
