"""Reductions of at most 1024 partials, which their consumer sums in every
workgroup instead of a launch in between, at the edge of that rule: 262,144
rows (1024 partials of p.Ap and of r.z), 262,145 (1025 of r.z) and 264,200 (1032
of p.Ap, 1033 of r.z).

Bars: a group sums them in launches of their own as soon as one member has too
many, so every member of a group of all sizes has the bits of its own solve;
and an operator with p.Ap < 0 still stops as a breakdown before it touches x."""
import numpy as np
import pytest

import apxchol_amd as ax
from apxchol_amd import matgen as mg

pytestmark = pytest.mark.gpu

SIZES = {3600: (60, 60), 262144: (512, 512), 262145: (5, 52429), 264200: (8, 33025)}


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("names", [(3600, 262144), (3600, 262144, 262145), tuple(SIZES)])
def test_group_members_at_the_edge_are_their_own_solves(gpu, names, precision):
    import torch
    print(f"[case] fused reductions {names} {precision}", flush=True)
    solvers, bs = [], []
    for n in names:
        A = mg.grid_laplacian(SIZES[n], "lognormal")
        assert A.shape[0] == n
        solvers.append(ax.Solver(A, seed=0, precision=precision))
        bs.append(torch.tensor(mg.request_rhs(A, False, n % 97), device=gpu))
    g = ax.Group(solvers)
    xs, rs = g.solve(bs, tol=1e-8, maxiter=25)
    for i, s in enumerate(solvers):
        own = s.solve(bs[i], tol=1e-8, maxiter=25)
        torch.cuda.synchronize()
        assert (rs[i].status, rs[i].iterations) == (own.status, own.iterations), i
        assert np.float64(rs[i].residual).view(np.int64) == np.float64(own.residual).view(np.int64), i
        assert torch.equal(xs[i].view(torch.int64), own.x.view(torch.int64)), i
    g.close()
    for s in solvers:
        s.close()


@pytest.mark.parametrize("n", [3600, 264200])
def test_breakdown_leaves_x(gpu, n):
    """The operator -A with the factor of A: p.Ap < 0 at once."""
    import torch
    print(f"[case] breakdown n={n}", flush=True)
    A = mg.add_excess(mg.grid_laplacian(SIZES[n], "lognormal"))
    s = ax.Solver((-A).tocsc(), factor=ax.factorize(A, seed=0))
    b = torch.tensor(np.random.default_rng(0).standard_normal(n), device=gpu)
    r = s.solve(b, tol=1e-8, maxiter=25)
    assert (r.status, r.iterations) == (2, 0)
    assert torch.equal(r.x, torch.zeros_like(r.x))
    s.close()
