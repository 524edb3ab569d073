"""Long operator rows of the sliced-ELL SpMV (walked by a wave, 16 entries of a
lane in flight) around the edges of its rounds: 33 entries (the first long
row), one round of 4, 12 and 16 x 64 entries and one more, several rounds.

Bars, as for every SpMV: each row within 1e-13 of (|A| |x|)_i against scipy's
fp64 product, and every column of the blocked SpMM the single product's bits."""
import numpy as np
import pytest
import scipy.sparse as sp

import apxchol_amd as ax

pytestmark = pytest.mark.gpu


def hub_graph(degree: int, n: int) -> sp.csc_matrix:
    """A ring of n vertices whose vertices 0 and 5 have `degree` entries in
    their row (the diagonal included)."""
    rng = np.random.default_rng(degree)
    i = np.arange(n)
    u, v = [i], [(i + 1) % n]
    for hub in (0, 5):
        others = np.setdiff1d(i, [hub, (hub + 1) % n, (hub - 1) % n, 0, 5])
        pick = rng.choice(others, degree - 3, replace=False)
        u.append(np.full(pick.size, hub))
        v.append(pick)
    u, v = np.concatenate(u), np.concatenate(v)
    w = rng.uniform(0.5, 2.0, u.size)
    W = sp.coo_matrix((np.r_[w, w], (np.r_[u, v], np.r_[v, u])), shape=(n, n)).tocsc()
    return (sp.diags(np.asarray(W.sum(axis=0)).ravel() * 1.01) - W).tocsc()


@pytest.mark.parametrize("degree", [32, 33, 64, 65, 256, 257, 768, 769, 832, 833, 1024, 1025, 1792, 1793, 2049, 5000])
def test_rows_at_round_edges(gpu, degree, monkeypatch):
    import torch
    print(f"[case] long rows degree={degree}", flush=True)
    A = hub_graph(degree, max(600, degree + 40))
    monkeypatch.setenv("APXCHOL_AMD_SPMV", "sell")
    s = ax.Solver(A, seed=0, precision="fp32")
    assert s.info["spmv_format"] == 1
    X = np.random.default_rng(1).standard_normal((5, A.shape[0]))
    Xd = torch.tensor(X, device=gpu)
    Y = s.spmv_batch(Xd).cpu().numpy()
    for c in range(5):
        y = s.spmv(Xd[c].clone()).cpu().numpy()
        bound = abs(A) @ abs(X[c])
        assert np.all(np.abs(y - A @ X[c]) <= 1e-13 * bound)
        assert np.array_equal(y.view(np.int64), Y[c].view(np.int64)), c
    s.close()


@pytest.mark.parametrize("k", [1, 2, 4, 7, 16, 32, 33])
@pytest.mark.parametrize("degree", [65, 1024, 1025, 1500])
def test_block_widths_on_both_sides_of_the_huge_rows(gpu, degree, k, monkeypatch):
    """A long row of up to 1024 entries (of these few) is summed by one wave for
    all columns, a longer one by a wave per column: each column the single
    product's bits at every block width, and a blocked solve converges."""
    import torch
    print(f"[case] huge rows degree={degree} k={k}", flush=True)
    A = hub_graph(degree, max(600, degree + 40))
    monkeypatch.setenv("APXCHOL_AMD_SPMV", "sell")
    s = ax.Solver(A, seed=0, precision="fp64")
    X = np.random.default_rng(2).standard_normal((k, A.shape[0]))
    Xd = torch.tensor(X, device=gpu)
    Y = s.spmv_batch(Xd).cpu().numpy()
    for c in range(k):
        y = s.spmv(Xd[c].clone()).cpu().numpy()
        assert np.array_equal(y.view(np.int64), Y[c].view(np.int64)), c
    Z, infos = s.solve_batch(Xd, tol=1e-8)
    for c in range(k):
        z = Z[c].cpu().numpy()
        assert np.linalg.norm(X[c] - A @ z) <= 2e-8 * np.linalg.norm(X[c])
    s.close()
