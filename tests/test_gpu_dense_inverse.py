"""Inverse of a dense coarsest level (one-level hierarchies, whose V-cycle is one
application of it) against numpy at the edges of its 64-row blocks and of its
dispatch: one block, the sizes with the symmetry and pivot-size checks (up to 160
rows), the sizes with the pivoted fallback (up to 512) and above.

Tolerance: the elimination's forward error is a small multiple of n eps cond."""
import numpy as np
import pytest
import scipy.sparse as sp
import torch

pytestmark = pytest.mark.gpu


def _spd(n, seed):
    rng = np.random.default_rng(seed)
    B = rng.standard_normal((n, n))
    A = B @ B.T / n + np.eye(n)
    s = np.exp(rng.uniform(-3.0, 3.0, n))  # rows of different magnitude
    return A * s[:, None] * s[None, :], s


def _csr(A, dev):
    A = sp.csr_matrix(A)
    A.sort_indices()
    return (torch.tensor(A.indptr, dtype=torch.int32, device=dev), torch.tensor(A.indices, dtype=torch.int32, device=dev),
            torch.tensor(A.data, dtype=torch.float64, device=dev))


def _check(h, A, scale, dev):
    b = np.random.default_rng(1).standard_normal(A.shape[0]) * scale
    x = h.vcycle(torch.tensor(b, device=dev), precision=64).cpu().numpy()
    y = np.linalg.solve(A, b)
    S = A / scale[:, None] / scale[None, :]
    e, w = (x - y) * scale, y * scale
    assert np.linalg.norm(e) <= 4 * A.shape[0] * 2.2e-16 * np.linalg.cond(S) * np.linalg.norm(w)


@pytest.mark.parametrize("n", [1, 2, 5, 63, 64, 65, 127, 128, 159, 160, 161, 192, 511, 513, 577])
def test_spd_inverse(dev, n):
    import impes_hip as H

    A, s = _spd(n, n)
    h = H.AmgHierarchy(coarsest_size=2000, dense_max=2000, coarse_pin=0)
    h.setup_csr(*_csr(A, dev))
    _check(h, A, s, dev)
    A2, s2 = _spd(n, n + 1)
    h.update_csr(_csr(A2, dev)[2])
    _check(h, A2, s2, dev)


@pytest.mark.parametrize("n,kind", [(65, "zero_pivot"), (100, "nonsymmetric"), (160, "negative"), (200, "negative"),
                                    (512, "negative")])
def test_not_spd_falls_back_to_pivoting(dev, n, kind):
    """At setup, and at an update of an SPD hierarchy; back to SPD after it."""
    import impes_hip as H

    A, s = _spd(n, n)
    if kind == "zero_pivot":
        C = A.copy()
        C[0, 0] = 0.0
    elif kind == "nonsymmetric":
        C = A + np.triu(np.random.default_rng(3).standard_normal((n, n)) * s[:, None] * s[None, :], 1) / n
    else:
        C = -A
    h = H.AmgHierarchy(coarsest_size=2000, dense_max=2000, coarse_pin=0)
    h.setup_csr(*_csr(C, dev))
    _check(h, C, s, dev)
    if kind == "zero_pivot":  # the zero is no entry of the pattern
        return
    for M in (A, C):
        h.update_csr(_csr(M, dev)[2])
        _check(h, M, s, dev)


@pytest.mark.parametrize("scale", [1e-300, 1e-160, 1e160, 1e300])
@pytest.mark.parametrize("n", [40, 100, 300, 577])
def test_operators_far_from_one(dev, n, scale):
    """Products of two entries leave the range of doubles, the entries do not."""
    import impes_hip as H

    B = np.random.default_rng(n).standard_normal((n, n))
    A = B @ B.T / n + np.eye(n)
    h = H.AmgHierarchy(coarsest_size=2000, dense_max=2000, coarse_pin=0, equil_threshold=0.0)
    h.setup_csr(*_csr(A * scale, dev))
    b = np.random.default_rng(1).standard_normal(n)
    x = h.vcycle(torch.tensor(b * scale, device=dev), precision=64).cpu().numpy()
    y = np.linalg.solve(A, b)
    assert np.linalg.norm(x - y) <= 4 * n * 2.2e-16 * np.linalg.cond(A) * np.linalg.norm(y)


@pytest.mark.parametrize("n", [50, 64, 130, 300, 600])
def test_repeated_columns_in_any_order(dev, n):
    """Every entry given as two, in two sweeps over the columns: they add up. Each half
    is positive definite, so that a lost one would not show as a failed elimination."""
    import impes_hip as H

    halves = [_spd(n, n + k)[0] for k in range(2)]
    A = halves[0] + halves[1]
    h = H.AmgHierarchy(coarsest_size=2000, dense_max=2000, coarse_pin=0)
    rp = torch.arange(0, 2 * n * n + 1, 2 * n, dtype=torch.int32, device=dev)
    ci = torch.arange(n, dtype=torch.int32, device=dev).repeat(2 * n)
    h.setup_csr(rp, ci, torch.tensor(np.hstack(halves).ravel(), device=dev))
    _check(h, A, np.sqrt(np.diag(A)), dev)
