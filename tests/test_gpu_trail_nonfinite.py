"""An infinity or NaN in one component's right-hand side stays in that
component: the trailing block's dense inverse holds the rows of all components,
with zeros between them.

Bar: in applications, blocked applications (the other columns too) and
(L L^T)^-1 products, the bits of the finite right-hand side in every row of the
other component, and no finite value lost there; walked levels alike."""
import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.csgraph as csg

import apxchol_amd as ax
from apxchol_amd import matgen as mg

pytestmark = pytest.mark.gpu


def grids():
    A = mg.add_excess(mg.grid_laplacian((14, 14, 14), "lognormal"))
    return sp.block_diag([A, A]).tocsc()


def rmats():
    A = mg.rmat_laplacian(11)
    lab = csg.connected_components(A, directed=False)[1]
    i = np.flatnonzero(lab == np.argmax(np.bincount(lab)))
    A = mg.add_excess(A[i][:, i].tocsc(), 1e-1)
    return sp.block_diag([A, A]).tocsc()


def bits(a):
    return np.ascontiguousarray(a).view(np.int64)


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("graph,precision", [(grids, "fp64"), (rmats, "fp64"), (rmats, "fp32")])
@pytest.mark.parametrize("rows", ["0", ""])
def test_other_components_keep_their_bits(gpu, graph, precision, bad, rows, monkeypatch):
    import torch
    print(f"[case] non-finite right-hand side {graph.__name__} {precision} {bad} rows={rows}", flush=True)
    A = graph()
    n = A.shape[0]
    other = np.arange(n) >= n // 2
    F = ax.factorize(A, seed=0)
    monkeypatch.setenv("APXCHOL_AMD_TRAIL_ROWS", rows)
    s = ax.Solver(A, factor=F, precision=precision)
    assert (s.info["block"]["rows"] > 0) == (rows == "")
    rng = np.random.default_rng(1)
    b = rng.standard_normal(n)
    hit = b.copy()
    hit[rng.integers(n // 2)] = bad

    def apply(r):
        return s.apply(torch.tensor(r, device=gpu)).cpu().numpy()

    z, zh = apply(b), apply(hit)
    assert np.isfinite(z).all() and not np.isfinite(zh).all()
    assert np.array_equal(bits(z[other]), bits(zh[other]))
    for k in (1, 2, 3, 8, 17):
        R = np.repeat(b[None], k, axis=0)
        R[k // 2] = hit
        Z = s.apply_batch(torch.tensor(R, device=gpu)).cpu().numpy()
        for c in range(k):
            part = other if c == k // 2 else slice(None)
            assert np.array_equal(bits(Z[c][part]), bits(z[part])), (k, c)
    # The same through (L L^T)^-1, in factor order.
    perm = F.export()[3].astype(np.int64)
    x, xh = np.empty(n), np.empty(n)
    x[perm], xh[perm] = b, hit
    y, yh = (s.solve_LLt(torch.tensor(v, device=gpu)).cpu().numpy()[perm] for v in (x, xh))
    assert np.array_equal(bits(y[other]), bits(yh[other])) and np.isfinite(y).all()
    s.close()
