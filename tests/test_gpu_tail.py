"""The coarse end of the preconditioner's cycle as one matrix (formed from the
identity once per update) against the cycle run level by level: `precondition`
uses the matrix, `vcycle` does not. Sizes on both sides of the row limit, tails
of one and of several levels, every smoothing count, the pinned coarsest level,
one-column remainders, both precisions, after setup and after an update.

FP64: rounding of sums of up to 2,048 terms. FP32: the matrix is the FP64 cycle's rounded
once (its entries are checked one by one); for a given right-hand side the error
against the FP64 cycle stays within a small multiple of the level-by-level FP32
cycle's own."""
import numpy as np
import pytest
import torch

from matrices import impes_like

pytestmark = pytest.mark.gpu

CASES = {
    "level0": ((12, 10, 10), dict(coarsest_size=200)),
    "level0_odd": ((13, 11, 7), dict(coarsest_size=50)),
    "level0_2048": ((16, 16, 8), dict(coarsest_size=100)),
    "above_2049": ((3, 683, 1), dict(coarsest_size=100)),
    "tiny": ((5, 3, 2), dict(coarsest_size=8, max_levels=25)),
    "many_levels": ((24, 20, 6), dict(coarsest_size=4, max_levels=25)),
    "deeper_than_tail": ((300, 1, 1), dict(coarsest_size=1, max_levels=25)),
    "coarsest_too_large": ((10, 10, 5), dict(coarsest_size=400)),
    "big": ((40, 40, 20), dict(coarsest_size=600, dense_max=600, max_levels=25, theta=0.1)),
    "v32_pinned": ((14, 12, 9), dict(coarsest_size=150, pre_smooth=3, post_smooth=2, omega=0.7, coarse_pin=1)),
    "v10": ((14, 12, 9), dict(pre_smooth=1, post_smooth=0)),
    "v01": ((14, 12, 9), dict(pre_smooth=0, post_smooth=1)),
    "v13": ((14, 12, 9), dict(pre_smooth=1, post_smooth=3)),
    "symmetric_scaling": ((14, 12, 9), dict(equil_mode=0)),
}


@pytest.mark.parametrize("kind", ["csr", "stencil"])
@pytest.mark.parametrize("name", list(CASES))
def test_tail_matrix_equals_the_levels(dev, name, kind):
    import impes_hip as H

    dims, kw = CASES[name]
    h = H.AmgHierarchy(**kw)
    rng = np.random.default_rng(2)
    for step, sigma in enumerate((1.0, 1.3)):
        A, *st = impes_like(*dims, seed=9, sigma=sigma)
        st = [torch.tensor(a, dtype=torch.float64, device=dev) for a in st]
        val = torch.tensor(A.data, dtype=torch.float64, device=dev)
        if step == 0 and kind == "csr":
            h.setup_csr(torch.tensor(A.indptr, dtype=torch.int32, device=dev),
                        torch.tensor(A.indices, dtype=torch.int32, device=dev), val)
        elif step == 0:
            h.setup_st7(dims, *st)
        elif kind == "csr":
            h.update_csr(val)
        else:
            h.update_st7(*st)
        for _ in range(2):  # the second time from the captured graph
            v = torch.tensor(rng.standard_normal(A.shape[0]), device=dev)
            dh = h.dhalf_inv()
            b = dh * st[0] * v
            z = dh * h.vcycle(b)
            z32 = dh * h.vcycle(b, precision=32)
            n = z.norm()
            e = (h.precondition(v, precision=64) - z).norm() / n
            assert e < 1e-12, f"FP64: {e:.1e}"
            e32, own = (h.precondition(v, precision=32) - z).norm() / n, (z32 - z).norm() / n
            assert e32 <= 3.0 * own + 2e-7, f"FP32: {e32:.1e} against {own:.1e}"


@pytest.mark.parametrize("dims,sigma,wells", [((20, 20, 3), 0.3, 0), ((20, 20, 3), 1.0, 2), ((18, 17, 4), 1.5, 0),
                                              ((36, 33, 1), 1.0, 1), ((25, 10, 2), 1.0, 2)])
def test_fp32_matrix_is_the_fp64_cycle_rounded_once(dev, dims, sigma, wells):
    """Columns of the FP32 cycle's matrix (the preconditioner of unit vectors: 1 is exact
    in FP32) against the FP64 cycle's: half an ulp of FP32 an entry, beside the FP64
    cycle's own rounding. Up to about 1,250 rows the matrix starts at level 0."""
    import impes_hip as H

    A, *st = impes_like(*dims, seed=3, sigma=sigma, wells=wells)
    d, *off = [torch.tensor(a, dtype=torch.float64, device=dev) for a in st]
    d = d - (1.0 - 1e-4) * 1.2e-12  # nearly singular without wells: the coarsest solve dominates
    h = H.AmgHierarchy()
    h.setup_st7(dims, d, *off)
    dh = h.dhalf_inv()
    n = d.numel()
    for j in np.random.default_rng(1).choice(n, 24, replace=False):
        e = torch.zeros(n, dtype=torch.float64, device=dev)
        e[j] = 1.0
        ref = h.vcycle(e)
        got = h.precondition(e / (dh * d), precision=32) / dh
        bound = 2.0**-24 * ref.abs() + 1e-12 * ref.abs().max()
        assert ((got - ref).abs() <= 1.01 * bound).all(), f"column {j}: {((got - ref).abs() / bound).max().item():.1f}"
