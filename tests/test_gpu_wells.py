"""The well kernels against the oracle's serial loop over the wells: counts at the edges
of their one workgroup of 256 threads, wells alone in their cells and chains of rate and
BHP wells that share one. Bars: those of the step parity (test_gpu_impes)."""
import json

import numpy as np
import pytest

from test_gpu_impes import PVT_SYNTH, run_parity, solver_cfg

pytestmark = pytest.mark.gpu


def well(rng, n, cell, first, nx, ny):
    # one BHP-type well a cell at most: the direct form the reference takes for two of
    # them multiplies the pressure's rounding by the well index
    k, t = cell % 2, cell // 2
    d = {"name": f"W{n}", "type": ("injector", "producer")[n % 2], "i": t // ny, "j": t % ny, "k": k, "radius": 0.1,
         "injected_phase": ("water", "gas")[n // 2 % 2]}
    if n % 5 < 3 or not first:
        d.update(control_type="rate", control_value=float(rng.uniform(0.5, 2.0)))
        if first and n % 2 and n % 3 == 0:
            d["bhp_min"] = 24.98  # some of these switch to their pressure limit
        if n % 2 and n % 4 == 1:
            d.update(rate_type="surface", surface_phase="liquid")
    else:
        d.update(control_type="bhp", control_value=25.0 + (0.02 if n % 2 == 0 else -0.02))
    return d


@pytest.mark.parametrize("nw,cells", [(2, 1), (5, 2), (255, 255), (256, 256), (257, 200), (600, 40), (600, 600)])
def test_wells_match_oracle(dev, nw, cells):
    nx, ny = 22, 20
    rng = np.random.default_rng(nw + cells)
    at = rng.choice(nx * ny * 2, size=cells, replace=False)
    where = np.concatenate([at, rng.choice(at, size=nw - cells)])
    cfg = {"simulation": {"solver_type": "impes"},
           "reservoir": {"dimensions": [nx, ny, 2], "grid_size": [20, 20, 10], "porosity": 0.25, "permeability": 200.0,
                         "k_vertical_fraction": 0.5},
           "fluid": {"pressure": 25.0, "s_w": 0.45, "s_g": 0.15, "pvt_table": json.load(open(PVT_SYNTH))},
           "wells": [well(rng, n, int(c), n < cells, nx, ny) for n, c in enumerate(where)]}
    run_parity(cfg, None, 20000.0, 2, amg=solver_cfg(64), whole_step=False)
