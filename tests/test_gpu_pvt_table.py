"""PVT table lookups of the device against numpy's interpolation formula, to the last
bit: node counts at the edges of the search, pressures at, beside, between and outside
the nodes, infinities and NaN. Division by 10^6 included (it is formed from the
reciprocal and has to round like the division)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

KEYS = ("Bo", "Bw", "Bg", "mu_o", "mu_w", "mu_g", "Rs", "Rv")


@pytest.mark.parametrize("n", [2, 3, 4, 5, 7, 8, 9, 20, 64, 65, 1000])
def test_lookup_is_the_interpolation(dev, n):
    from impes_hip import ops
    from impes_hip._lib import FluidStruct

    rng = np.random.default_rng(n)
    nodes = np.cumsum(rng.uniform(0.01, 2.0, n))
    cols = rng.uniform(-2.0, 3.0, (8, n))
    fluid = FluidStruct(max_ds=1.0, max_substeps=1)
    model = ops.ImpesModel((4, 3, 2, 10.0, 10.0, 5.0), fluid, np.concatenate([nodes[None], cols]))
    x = np.concatenate([nodes, np.nextafter(nodes, -np.inf), np.nextafter(nodes, np.inf),
                        rng.uniform(nodes[0] - 3.0, nodes[-1] + 3.0, 5000), [-np.inf, np.inf, np.nan, 0.0]])
    p = x * 1e6
    x = p / 1e6
    t = torch.tensor(p, dtype=torch.float64, device=dev)
    seg = np.clip(np.searchsorted(nodes, x, side="right") - 1, 0, n - 2)
    for key, col in zip(KEYS, cols):
        with np.errstate(invalid="ignore"):
            ref = (col[seg + 1] - col[seg]) / (nodes[seg + 1] - nodes[seg]) * (x - nodes[seg]) + col[seg]
        ref = np.where(x < nodes[0], col[0], np.where(x >= nodes[-1], col[-1], ref))
        ref[np.isnan(x)] = np.nan
        got = model.eval_pvt(key, t).cpu().numpy()
        assert np.array_equal(got, ref, equal_nan=True), key
