"""Water levels and point probes against the oracle, over the domain and outside it.

A level comes from chunks of 256 sampling heights, one workgroup each; a march that
leaves the first launch's heights behind goes on in another.  Levels are the
oracle's to the last bit (both march by the same sums, and a threshold is crossed
whole heights away from round-off here); probes to 1e-12.
"""
import numpy as np
import pytest

import tinysph_old_amd as T
from tests.helpers import oracle_for, oracle_init

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _oracle(oracle_built):
    return oracle_built


@pytest.mark.parametrize("preset,dx", [(T.CASE_DAM_BREAK_MDBC, 0.02), (T.CASE_DAM_BREAK_BT, 0.01),
                                       (T.CASE_STILL_WATER_DBC, 0.02)])
def test_levels_and_points(preset, dx):
    case = T.build_case(preset, dx=dx, jitter=0.05, seed=9)
    prm = case.params
    print(f"[case] probes preset {preset} np={case.np}", flush=True)
    O = oracle_for(case)
    oracle_init(O)
    O.call("density_to_pressure")
    width, top = prm["x_m"], prm["y_m"]
    with T.system_for_case(case) as ps:
        ps.particle_to_cell()
        ps.density_to_pressure()
        for x in (0.013, 0.1 * width, 0.3, 0.5 * width, 0.97 * width):
            for y0, inverse in ((0.0, False), (0.21, False), (0.45, True), (0.95 * top, True)):
                fn = "water_elevation_inverse" if inverse else "water_elevation"
                got, ref = ps.water_elevation(x, y0, inverse=inverse), O.call(fn, x, y0)
                assert got == ref or (np.isnan(got) and np.isnan(ref)), (x, y0, inverse, got, ref)
        for x, y in ((0.3, 0.03), (0.013, 0.0), (0.0, 0.2), (0.5 * width, 0.4), (0.3, 0.9 * top)):
            got, ref = np.array(ps.interpolate_point(x, y)), np.array(O.interpolate_point(x, y))
            assert np.allclose(got, ref, rtol=1e-12, atol=1e-12 * 1000.0), (x, y, got, ref)
        assert np.isnan(ps.water_elevation(width + 5.0, 0.95 * top, inverse=True))
