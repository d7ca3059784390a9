"""FGMRES of small systems in one workgroup per step against a direct solve and
against the solver's separate kernels (the three-pass form, which it does not take):
the edges of its rows per thread and of its size limit, stencil and CSR operators,
both hierarchy precisions, restarts of 1 to 32 vectors, a stop by the error check,
an exact starting guess and a zero right-hand side.

Bars: the asked relative residual times a condition allowance for the solution; the
same number of steps up to one (the stopping test sees another rounding)."""
import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spl
import torch

from matrices import impes_like

pytestmark = pytest.mark.gpu


def _solve(dev, dims, kind, precision, restart, rtol=1e-10, etol=0.0, x0=None, b=None, seed=3):
    import impes_hip as H

    A, *st = impes_like(*dims, seed=seed, wells=1)
    n = A.shape[0]
    if b is None:
        b = A @ (2e7 + 1e6 * np.random.default_rng(1).standard_normal(n))
    st = [torch.tensor(a, dtype=torch.float64, device=dev) for a in st]
    h = H.AmgHierarchy(coarsest_size=60)
    bt = torch.tensor(b, device=dev)
    x = torch.zeros(n, dtype=torch.float64, device=dev) if x0 is None else torch.tensor(x0, device=dev)
    kw = dict(precision=precision, use_x0=x0 is not None, rtol=rtol, restart=restart, maxit=300, etol=etol)
    s = H.FgmresSolver()
    if kind == "stencil":
        h.setup_st7(dims, *st)
        out = s.solve_st7(h, dims, *st, 1.0 / st[0], bt, x, **kw)
    else:
        csr = [torch.tensor(a, dtype=torch.int32, device=dev) for a in (A.indptr, A.indices)]
        csr.append(torch.tensor(A.data, dtype=torch.float64, device=dev))
        h.setup_csr(*csr)
        out = s.solve_csr(h, *csr, 1.0 / st[0], bt, x, **kw)
    return A, b, x.cpu().numpy(), out


@pytest.mark.parametrize("kind", ["stencil", "csr"])
@pytest.mark.parametrize("dims", [(1, 1, 1), (3, 1, 1), (9, 7, 1), (31, 33, 1), (16, 16, 4), (41, 25, 1), (32, 32, 2),
                                  (683, 3, 1), (16, 16, 16), (17, 241, 1)])
def test_small_matches_direct_and_separate_kernels(dev, dims, kind, monkeypatch):
    for precision, restart in ((32, 30), (64, 7)):
        monkeypatch.delenv("IMPES_FGMRES_CGS2", raising=False)
        A, b, x, st = _solve(dev, dims, kind, precision, restart)
        assert st["converged"] and st["rel_residual"] <= 1e-10
        d = A.diagonal()
        r = (b - A @ x) / d
        assert np.linalg.norm(r) <= 1.01e-10 * np.linalg.norm(b / d)
        y = spl.spsolve(A.tocsc(), b)
        assert np.linalg.norm(x - y) <= 1e-6 * np.linalg.norm(y)
        monkeypatch.setenv("IMPES_FGMRES_CGS2", "1")
        *_, x2, st2 = _solve(dev, dims, kind, precision, restart)
        assert abs(st["iterations"] - st2["iterations"]) <= 1
        assert np.linalg.norm(x - x2) <= 1e-6 * np.linalg.norm(y)


@pytest.mark.parametrize("restart", [1, 2, 31, 32])
def test_small_restarts(dev, restart):
    A, b, x, st = _solve(dev, (20, 20, 3), "stencil", 32, restart, rtol=1e-9)
    assert st["converged"]
    assert np.linalg.norm((b - A @ x) / A.diagonal()) <= 1.01e-9 * np.linalg.norm(b / A.diagonal())


@pytest.mark.parametrize("kind", ["stencil", "csr"])
def test_small_error_check_start_and_zero_rhs(dev, kind):
    A, b, x, st = _solve(dev, (20, 20, 3), kind, 32, 30, rtol=1e-8, etol=1e-9)
    y = spl.spsolve(A.tocsc(), b)
    assert st["converged"] and st["checks"] >= 1 and st["err_estimate"] <= 0.5e-9
    assert np.max(np.abs(x - y)) <= 4e-9 * np.max(np.abs(y))
    # the exact solution as start: no step, but the check
    *_, x1, st1 = _solve(dev, (20, 20, 3), kind, 64, 30, rtol=1e-6, etol=1e-6, x0=y)
    assert st1["iterations"] == 0 and st1["checks"] == 1 and st1["converged"]
    assert np.max(np.abs(x1 - y)) <= 1e-8 * np.max(np.abs(y))
    *_, x2, st2 = _solve(dev, (20, 20, 3), kind, 32, 30, b=np.zeros(A.shape[0]), x0=y)
    assert st2["converged"] and not x2.any()


@pytest.mark.parametrize("leaves", [200, 1500])
def test_one_long_row(dev, leaves):
    """A small system with one row of some hundred or thousand entries: on both sides of
    the length from which the separate kernels take it."""
    import impes_hip as H
    from test_gpu_solver import to_dev

    A = impes_like(40, 40, 1, wells=0)[0]
    n = A.shape[0]
    at = np.random.default_rng(0).choice(n - 1, size=leaves, replace=False)
    E = sp.coo_matrix((np.full(leaves, -1e-13), (np.full(leaves, n - 1), at)), shape=(n, n))
    E = (E + E.T).tocsr()
    A = (A + E + sp.diags(-np.asarray(E.sum(1)).ravel())).tocsr()
    A.sort_indices()
    csr = to_dev(A, dev)
    b = A @ np.random.default_rng(1).standard_normal(A.shape[0])
    for precision in (32, 64):
        h = H.AmgHierarchy(coarsest_size=60)
        h.setup_csr(*csr)
        x = torch.zeros(A.shape[0], dtype=torch.float64, device=dev)
        d = A.diagonal()
        st = H.FgmresSolver().solve_csr(h, *csr, torch.tensor(1.0 / d, device=dev), torch.tensor(b, device=dev), x,
                                        precision=precision, rtol=1e-10)
        assert st["converged"]
        assert np.linalg.norm((b - A @ x.cpu().numpy()) / d) <= 1.01e-10 * np.linalg.norm(b / d)
