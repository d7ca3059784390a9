"""Prolongation and first post-sweep as one pass and the FP64 preconditioner's tiled
passes against the FP64 cycle, which has neither: every smoothing count that reaches it, odd and even, stencil and CSR finest
levels, levels above and inside the tail, at setup and after an update, replayed from the
captured graph; and the operators that keep the two passes: a row too long for a tile, a
row without a diagonal entry.

FP64: rounding of sums of up to some hundred terms. FP32: the cycle's own rounding, a few
hundred operations deep."""
import numpy as np
import pytest
import scipy.sparse as sp
import torch

from matrices import impes_like
from test_gpu_galerkin import hub
from test_gpu_solver import rel, to_dev

pytestmark = pytest.mark.gpu


def no_diagonal(n):
    A = impes_like(*n, seed=6)[0].tocoo()
    keep = ~((A.row == 777) & (A.col == 777))
    return sp.csr_matrix((A.data[keep], (A.row[keep], A.col[keep])), shape=A.shape)


DEEP = dict(coarsest_size=20, max_levels=25)
CASES = {
    "csr": ("csr", (20, 18, 16), {}),
    "csr_two_levels": ("csr", (16, 15, 14), dict(max_levels=1, dense_max=3000, coarsest_size=400)),
    "stencil": ("st7", (20, 18, 16), DEEP),
    "stencil_odd": ("st7", (37, 29, 3), DEEP),
    "stencil_above_the_limit": ("st7", (90, 60, 50), {}),
    "v11": ("csr", (20, 18, 16), dict(DEEP, pre_smooth=1, post_smooth=1)),
    "v13": ("st7", (20, 18, 16), dict(DEEP, pre_smooth=1, post_smooth=3)),
    "v32": ("csr", (20, 18, 16), dict(DEEP, pre_smooth=3, post_smooth=2, omega=0.7)),
    "v31": ("st7", (20, 18, 16), dict(DEEP, pre_smooth=3, post_smooth=1)),
    "v20": ("csr", (20, 18, 16), dict(DEEP, pre_smooth=2, post_smooth=0)),
    "v02": ("csr", (20, 18, 16), dict(DEEP, pre_smooth=0, post_smooth=2)),
    "hub": ("hub", (20, 20, 20), dict(coarsest_size=100)),
    "no_diagonal": ("no_diagonal", (20, 18, 16), {}),
}


@pytest.mark.parametrize("name", list(CASES))
def test_fp32_cycle_matches_fp64(dev, name):
    import impes_hip as H

    kind, dims, kw = CASES[name]
    h = H.AmgHierarchy(**kw)
    rng = np.random.default_rng(3)
    for step, sigma in enumerate((1.0, 1.3)):
        A, *st = impes_like(*dims, seed=8, sigma=sigma)
        st = [torch.tensor(a, dtype=torch.float64, device=dev) for a in st]
        if kind == "hub":
            A = hub(dims, 4000) * sigma
        elif kind == "no_diagonal":
            A = no_diagonal(dims) * sigma
        if kind == "st7":
            (h.setup_st7(dims, *st) if step == 0 else h.update_st7(*st))
        else:
            rp, ci, v = to_dev(A, dev)
            (h.setup_csr(rp, ci, v) if step == 0 else h.update_csr(v))
        n = A.shape[0]
        for _ in range(2):
            b = torch.tensor(rng.standard_normal(n), device=dev)
            y = h.vcycle(b, precision=64).cpu().numpy()
            assert rel(h.vcycle(b, precision=32).cpu().numpy(), y) < 2e-5
            z = h.precondition(b, precision=64).cpu().numpy()
            if kind != "no_diagonal":  # the tiled FP64 cycle against the untiled one
                dh = h.dhalf_inv()
                d = torch.tensor(A.diagonal(), device=dev)
                assert rel(z, (dh * h.vcycle(dh * d * b, precision=64)).cpu().numpy()) < 1e-12
            assert rel(h.precondition(b, precision=32).cpu().numpy(), z) < 2e-5


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("dims", [(12, 10, 10), (30, 24, 10)])  # the tail from level 0 on, levels above it
def test_recorded_preparations_are_not_done(dev, dims, precision):
    """A cycle recorded into a caller's graph after an update prepares its matrices when
    the graph runs; an eager cycle before that prepares its own."""
    import impes_hip as H

    first, second = (to_dev(impes_like(*dims, seed=8, sigma=s)[0], dev) for s in (1.0, 1.3))
    fresh, h = H.AmgHierarchy(), H.AmgHierarchy()
    fresh.setup_csr(*first)
    fresh.update_csr(second[2])
    h.setup_csr(*first)
    h.set_graphs(False)
    v = torch.tensor(np.random.default_rng(0).standard_normal(first[0].numel() - 1), device=dev)
    z = torch.empty_like(v)
    h.precondition(v, precision=precision, out=z)
    h.update_csr(second[2])
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        h.precondition(v, precision=precision, out=z)
    ref = fresh.precondition(v, precision=precision)
    assert torch.equal(h.precondition(v, precision=precision), ref)
    for _ in range(3):
        z.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(z, ref)
        assert torch.equal(h.precondition(v, precision=precision), ref)
