"""Factors whose trailing block has directions far softer than the rest: two
R-MAT graphs joined by one weak edge, slightly regularised Laplacians, one tiny
diagonal excess. The rounding of the block's explicit inverse would hide those
directions (mixed solves then lose positive definiteness), so such factors walk
their levels.

Bar: status and iterations (+- 1) of the solver without a block, in both
precisions, for single solves and blocked columns; its bits wherever the
default solver has no block either."""
import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.csgraph as csg

import apxchol_amd as ax
from apxchol_amd import matgen as mg

pytestmark = pytest.mark.gpu


def giant():
    A = mg.rmat_laplacian(11)
    lab = csg.connected_components(A, directed=False)[1]
    i = np.flatnonzero(lab == np.argmax(np.bincount(lab)))
    return A[i][:, i].tocsc()


def pair(w):
    A = giant()
    n, k = A.shape[0], int(np.argmax(np.diff(A.indptr)))
    B = sp.block_diag([A, A]).tolil()
    for i, j in ((k, n + k), (n + k, k)):
        B[i, j] -= w
        B[i, i] += w
    return B.tocsc()


def one_entry():
    A = giant().tolil()
    A[5, 5] += 1e-4
    return A.tocsc()


CASES = {f"pair_{w:g}": (lambda w=w: pair(w)) for w in (1.0, 1e-1, 1e-2, 1e-3, 1e-4, 1e-6)}
CASES |= {f"plus_{e:g}": (lambda e=e: (giant() + e * sp.eye(giant().shape[0])).tocsc()) for e in (1e-2, 1e-6, 1e-8)}
CASES |= {"excess_1e-9": lambda: mg.add_excess(giant(), 1e-9), "one_entry_1e-4": one_entry,
          "grids_1e-8": lambda: sp.csc_matrix(grids(1e-8))}


def grids(w):
    A = mg.grid_laplacian((12, 12, 12))
    n = A.shape[0]
    B = sp.block_diag([A, A]).tolil()
    for i, j in ((0, n), (n, 0)):
        B[i, j] -= w
        B[i, i] += w
    return B


@pytest.mark.parametrize("name", list(CASES))
def test_iterations_of_the_walked_levels(gpu, name, monkeypatch):
    import torch
    A = CASES[name]()
    F = ax.factorize(A, seed=0)
    bs = torch.tensor(np.stack([mg.request_rhs(A, F.sddm, q) for q in (3, 4, 5)]), device=gpu)
    for precision in ("fp32", "fp64"):
        print(f"[case] soft trailing block {name} {precision}", flush=True)
        monkeypatch.setenv("APXCHOL_AMD_TRAIL_ROWS", "0")
        walked = ax.Solver(A, factor=F, precision=precision)
        monkeypatch.delenv("APXCHOL_AMD_TRAIL_ROWS")
        s = ax.Solver(A, factor=F, precision=precision)
        for b in bs:
            w, r = walked.solve(b, tol=1e-8, maxiter=100), s.solve(b, tol=1e-8, maxiter=100)
            torch.cuda.synchronize()
            print(f"  block {s.info['block']['rows']} walked {w.iterations} ({w.status}, {w.residual:.1e}) "
                  f"now {r.iterations} ({r.status}, {r.residual:.1e})", flush=True)
            assert r.status == w.status
            assert abs(r.iterations - w.iterations) <= 1
            if s.info["block"]["rows"] == 0:
                assert torch.equal(r.x.view(torch.int64), w.x.view(torch.int64))
        _, ws = walked.solve_batch(bs, tol=1e-8, maxiter=100)
        _, rs = s.solve_batch(bs, tol=1e-8, maxiter=100)
        torch.cuda.synchronize()
        for w, r in zip(ws, rs):
            assert r.status == w.status and abs(r.iterations - w.iterations) <= 1
        walked.close()
        s.close()
