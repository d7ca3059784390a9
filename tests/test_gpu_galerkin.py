"""The numeric Galerkin product against scipy's, entry by entry: few and many entries
(64 or 256 of them to a workgroup), sums of a few terms and of more than one LDS chunk,
at setup and after an update with new values.

Bound: both sides sum k products of three factors, so they differ by at most
2 (k + 4) eps (|R| |A| |P|) with k the largest number of terms of an entry."""
import numpy as np
import pytest
import scipy.sparse as sp

from matrices import impes_like
from test_gpu_solver import csr_from_export, to_dev

pytestmark = pytest.mark.gpu


def hub(n, leaves):
    """A grid operator and one row to which `leaves` others are coupled the strongest:
    they interpolate from it, and its column of P has an entry for each."""
    A = impes_like(*n, seed=1)[0].tolil()
    N = A.shape[0]
    at = np.random.default_rng(0).choice(N - 1, size=leaves, replace=False)
    w = 3.0 * abs(A.diagonal()).max()
    H = sp.coo_matrix((np.full(leaves, -w), (np.full(leaves, N - 1), at)), shape=(N, N))
    H = (H + H.T).tocsr()
    return (A.tocsr() + H + sp.diags(-np.asarray(H.sum(1)).ravel())).tocsr()


def dense(n, per):
    """A random M-matrix of about `per` entries in a row."""
    rng = np.random.default_rng(0)
    B = sp.random(n, n, per / (2.0 * n), random_state=rng, format="csr", data_rvs=lambda k: np.exp(rng.standard_normal(k)))
    B = B + B.T
    B.setdiag(0.0)
    B.eliminate_zeros()
    A = sp.csr_matrix(sp.diags(np.asarray(B.sum(1)).ravel() + 0.01) - B)
    A.sort_indices()
    return A


CASES = {
    "tiny": (lambda: impes_like(5, 4, 3)[0], dict(coarsest_size=4, max_levels=25), 1),
    "odd": (lambda: impes_like(17, 13, 3, seed=2)[0], dict(coarsest_size=10, max_levels=25), 1),
    "wide": (lambda: impes_like(40, 40, 20, seed=3)[0], {}, 1),
    "hub": (lambda: hub((24, 24, 24), 9000), dict(coarsest_size=100), 2049),
    # few rows with product lists beyond a workgroup's LDS (the sort's long segments)
    "hub_few_rows": (lambda: hub((15, 15, 15), 3000), dict(coarsest_size=100), 2049),
    "dense_few_rows": (lambda: dense(700, 300), dict(coarsest_size=20, max_levels=25), 1),
}


@pytest.mark.parametrize("name", list(CASES))
def test_coarse_operators_are_the_product(dev, name):
    import impes_hip as H

    make, kw, terms = CASES[name]
    A = make()
    hg = H.AmgHierarchy(**kw)
    hg.setup_csr(*to_dev(A, dev))
    most = 0
    for values in ("setup", "update"):
        if values == "update":
            d = sp.diags(1.0 + 0.5 * np.random.default_rng(5).random(A.shape[0]))
            hg.update_csr(to_dev((d @ A @ d).tocsr(), dev)[2])
        for l in range(hg.num_levels - 1):
            e, nxt = hg.export_level(l), csr_from_export(hg.export_level(l + 1))
            Al = csr_from_export(e)
            P = sp.csr_matrix((e["p_val"].cpu().numpy(), e["p_col"].cpu().numpy(), e["p_rowptr"].cpu().numpy()),
                              shape=(e["n"], nxt.shape[0]))
            one = lambda M: sp.csr_matrix((np.ones(M.nnz), M.indices, M.indptr), shape=M.shape)  # noqa: E731
            Ap = one(Al) @ one(P)
            most = max(most, Ap.max(), (one(P.T.tocsr()) @ one(Ap)).max())
            k = (one(P.T.tocsr()) @ Ap).max()
            bound = 2 * (k + 4) * np.finfo(float).eps * (abs(P).T @ (abs(Al) @ abs(P)))
            diff = abs(P.T.tocsr() @ (Al @ P) - nxt)
            assert (diff - bound).max() <= 0, (values, l)
    assert most >= terms
