"""Which form the operator takes: the rows of a graph without hubs stay in the
slices of the sliced-ELL form however dense they are, the rows past the mean of
a power-law graph leave them, and a small graph whose slices pad too much with
its hubs alone left out keeps CSR lanes.

Bars: the padded entries reported, each row of a product within 1e-13 of
(|A| |x|)_i, every column of a blocked product the single product's bits."""
import numpy as np
import pytest
import scipy.sparse as sp

import apxchol_amd as ax
from apxchol_amd import matgen as mg

pytestmark = pytest.mark.gpu


def random_graph(n, degree, hub=0):
    rng = np.random.default_rng(degree)
    i = np.repeat(np.arange(n), degree)
    j = rng.integers(n, size=i.size)
    if hub:   # one row of a few hundred entries
        i, j = np.r_[i, np.zeros(hub, int)], np.r_[j, rng.choice(np.arange(1, n), hub, replace=False)]
    keep = i != j
    W = sp.coo_matrix((np.ones(keep.sum()), (i[keep], j[keep])), shape=(n, n)).tocsr()
    W = W + W.T
    return mg.add_excess((sp.diags(np.asarray(W.sum(axis=1)).ravel()) - W).tocsc())


CASES = {
    "random_2000_20": (lambda: random_graph(2000, 20), "slices"),
    "random_2000_40": (lambda: random_graph(2000, 40), "slices"),
    "random_2000_20_hub": (lambda: random_graph(2000, 20, 700), "one row out"),
    "rmat_13": (lambda: mg.rmat_laplacian(13), "rows out"),
    "rmat_9": (lambda: mg.rmat_laplacian(9), "csr"),
}


@pytest.mark.parametrize("name", list(CASES))
def test_form_and_products(gpu, name):
    import torch
    print(f"[case] SpMV form {name}", flush=True)
    make, form = CASES[name]
    A = make()
    s = ax.Solver(A, seed=0, precision="fp32")
    slots = s.info["spmv_sell_slots"]
    longest = int(np.diff(A.indptr).max())
    if form == "csr":
        assert s.info["spmv_format"] == 0 and slots == 0
    else:
        assert s.info["spmv_format"] == 1
        assert {"slices": slots >= A.nnz, "one row out": A.nnz - longest <= slots < 1.2 * A.nnz,
                "rows out": slots < 0.9 * A.nnz}[form]
    X = np.random.default_rng(3).standard_normal((5, A.shape[0]))
    Xd = torch.tensor(X, device=gpu)
    Y = s.spmv_batch(Xd).cpu().numpy()
    for c in range(5):
        y = s.spmv(Xd[c].clone()).cpu().numpy()
        assert np.all(np.abs(y - A @ X[c]) <= 1e-13 * (abs(A) @ abs(X[c])))
        if form != "csr":
            assert np.array_equal(y.view(np.int64), Y[c].view(np.int64)), c
        else:
            assert np.all(np.abs(Y[c] - A @ X[c]) <= 1e-13 * (abs(A) @ abs(X[c])))
    s.close()
