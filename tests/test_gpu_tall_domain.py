"""Water levels in a domain of more sampling heights than an int counts.

The march steps by dp * 5e-5, so a domain some 1e5 spacings tall has 2e9 heights,
and one a little taller more than an int holds; the level of the water at its
bottom is met within the first thousands and does not depend on the domain's top.
"""
import numpy as np
import pytest

import tinysph_old_amd as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("spacings", [9e4, 1.06e5, 1.08e5, 2e5])
def test_levels_below_a_high_top(spacings):
    dp = 0.01
    x, y = (g.ravel() * dp for g in np.meshgrid(np.arange(12), np.arange(30)))
    arrays = {"type": np.full(x.size, T.FLUID, np.int32), "r": np.stack([x, y], -1),
              "rho": np.full(x.size, 1000.0)}
    levels = []
    for top in (2.0, spacings * dp):
        prm = {"h": dp * 2 ** 0.5, "kap": 2.1, "cs": 20.0, "rho0": 1000.0, "avisc": 0.02, "delta": 0.1,
               "dp": dp, "x_0": -0.03, "x_m": 0.15, "y_0": -0.03, "y_m": top}
        print(f"[case] level below a top of {top} m, np={x.size}", flush=True)
        with T.ParticleSystem(prm, capacity=x.size) as ps:
            ps.upload(arrays)
            ps.particle_to_cell()
            levels.append([ps.water_elevation(0.055, 0.05), ps.water_elevation(0.055, 0.5, inverse=True)])
    print(levels, flush=True)
    assert np.isfinite(levels[0]).all() and levels[0] == levels[1]
