"""The FP64 pair pass against the oracle, bit for bit.

Every division and square root of a pair term is correctly rounded and every
sum is formed in the oracle's order, so one pass over the same state gives the
same bits, whichever walk the system's size selects.  The exception is the
root in the density-diffusion term, which is within an ulp of libm's: with
delta = 0 that term is zero and drho is bit-identical too.  States have random
velocities, densities and pressures, negative ones among them; sizes lie on
both sides of the walks' limits, the smallest with cells of a few particles;
a cluster puts a neighbourhood beyond the LDS budget, another more than 64
particles into one cell, and coincident particles have r = 0.
"""
import numpy as np
import pytest

import tinysph_old_amd as T
from oracle import pyoracle as po
from tests.helpers import oracle_for, oracle_init, oracle_variant

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _oracle(oracle_built):
    return oracle_built


def state(preset, dx, seed, delta=0.0):
    case = T.build_case(preset, dx=dx, jitter=0.2, seed=seed)
    g = np.random.RandomState(seed)
    n = case.np
    case.params["delta"] = delta
    a = case.arrays
    fluid = a["type"] == T.FLUID
    a["v"] = np.where(fluid[:, None], g.normal(0, 1.0, (n, 2)), 0.0)
    a["rho"] = 1000.0 + g.normal(0, 5.0, n)
    a["p"] = g.normal(0, 3000.0, n)
    return case, fluid, g


def compare(case, what, waves=0):
    print(f"[case] {what} np={case.np}", flush=True)
    O = oracle_for(case)
    oracle_init(O)
    O.call("compute_forces", oracle_variant(case.wall))
    with T.system_for_case(case) as ps:
        if waves:
            ps.set_waves_per_cu(waves)
        ps.particle_to_cell()
        ps.compute_forces(T.forces_variant(case.wall))
        if waves:  # once more, its chunks cut by the times the first pass recorded
            ps.particle_to_cell()
            ps.compute_forces(T.forces_variant(case.wall))
        got = ps.download(("a", "drho"))
    assert np.array_equal(got["a"], O.get(po.F_A), equal_nan=True)
    if case.params["delta"] == 0.0:
        assert np.array_equal(got["drho"], O.get(po.F_DRHO), equal_nan=True)


@pytest.mark.parametrize("delta", [0.0, 0.1])
@pytest.mark.parametrize("preset,dx", [
    (T.CASE_STILL_WATER_DBC, 0.05), (T.CASE_STILL_WATER_DBC, 0.0101), (T.CASE_DAM_BREAK_MDBC, 0.012),
    (T.CASE_DAM_BREAK_MDBC, 0.0033), (T.CASE_DAM_BREAK_MDBC, 0.003), (T.CASE_DAM_BREAK_BT, 0.021),
    (T.CASE_DAM_BREAK_BT, 0.0047), (T.CASE_DAM_BREAK_BT, 0.0015), (T.CASE_STILL_WATER_DBC, 0.0026)])
def test_pair_pass_equals_oracle_bit_for_bit(preset, dx, delta):
    case, _, _ = state(preset, dx, 7, delta)
    compare(case, f"preset {preset} dx {dx} delta {delta}")


@pytest.mark.parametrize("preset,dx", [(T.CASE_STILL_WATER_DBC, 0.0026), (T.CASE_DAM_BREAK_MDBC, 0.003),
                                       (T.CASE_DAM_BREAK_BT, 0.0015)])
def test_pooled_walk_equals_oracle_bit_for_bit(preset, dx):
    """One wavefront per compute unit: enough particles for each that tiles are pooled."""
    case, _, _ = state(preset, dx, 9)
    compare(case, f"preset {preset} dx {dx} pooled", waves=1)


@pytest.mark.parametrize("preset", [T.CASE_STILL_WATER_DBC, T.CASE_DAM_BREAK_MDBC, T.CASE_DAM_BREAK_BT])
@pytest.mark.parametrize("crowd", [2, 12, 40, 100])
def test_crowded_cells_equal_oracle_bit_for_bit(preset, crowd):
    """`crowd` particles moved into one cell, next to its own."""
    case, fluid, g = state(preset, 0.012, 13)
    at = np.nonzero(fluid)[0]
    home = case.arrays["r"][at[len(at) // 2]]
    moved = g.choice(at, crowd, replace=False)
    case.arrays["r"][moved] = home + g.uniform(-0.2, 0.2, (crowd, 2)) * case.params["h"]
    case.arrays["r_o"] = case.arrays["r"].copy()
    compare(case, f"preset {preset} with {crowd} particles in one cell")


@pytest.mark.parametrize("preset", [T.CASE_STILL_WATER_DBC, T.CASE_DAM_BREAK_MDBC])
def test_coincident_particles_equal_oracle_bit_for_bit(preset):
    case, fluid, _ = state(preset, 0.012, 17)
    at = np.nonzero(fluid)[0]
    case.arrays["r"][at[40]] = case.arrays["r"][at[41]]
    compare(case, f"preset {preset}, two coincident particles")
