"""Wall densities against the oracle, bit for bit, where a wall has many neighbours.

The pass holds a wall's fluid neighbours in LDS and takes them 16 at a time: none,
fewer than 16, exactly so many that some are left over, and hundreds, in the
reference order; walls at the domain's corners, whose cells lie partly outside.
"""
import numpy as np
import pytest

import tinysph_old_amd as T
from oracle import pyoracle as po
from tests.helpers import oracle_for, oracle_init

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _oracle(oracle_built):
    return oracle_built


@pytest.mark.parametrize("spacing", [4.0, 1.7, 1.0, 0.7, 0.5, 0.25])
@pytest.mark.parametrize("preset", [T.CASE_DAM_BREAK_MDBC, T.CASE_DAM_BREAK_BT])
def test_wall_densities(preset, spacing):
    case = T.build_case(preset, dx=0.02, jitter=0.02, seed=4)
    a, prm, g = case.arrays, case.params, np.random.RandomState(6)
    fluid = np.nonzero(a["type"] == T.FLUID)[0]
    # the fluid on a lattice of `spacing` dp from the lower left corner up
    d, side = spacing * prm["dp"], int(np.sqrt(len(fluid)))
    xy = np.stack(np.meshgrid(np.arange(side), np.arange(side)), -1).reshape(-1, 2)
    low = a["r"][fluid].min(0)
    at = low + d * (xy + 0.1 * g.uniform(-1, 1, xy.shape))
    at = np.clip(at, low, [prm["x_m"] - prm["h"], prm["y_m"] - prm["h"]])
    a["r"][fluid[:len(at)]] = at
    a["rho"][fluid] = 1000.0 + g.normal(0, 10.0, len(fluid))
    for k in ("r_o", "v_o"):
        a.pop(k, None)
    print(f"[case] walls preset {preset} spacing {spacing} np={case.np}", flush=True)
    mdbc = case.wall == T.WALL_MDBC
    O = oracle_for(case)
    oracle_init(O)
    O.call("mdbc_density" if mdbc else "bt_density")
    with T.system_for_case(case) as ps:
        ps.particle_to_cell()
        ps.mdbc_density() if mdbc else ps.bt_density()
        rho = ps.download(("rho",))["rho"]
    assert np.array_equal(rho, O.get(po.F_RHO))
