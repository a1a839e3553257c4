"""FP32 pair passes over tiles that hold more than a wavefront or the LDS budget.

The list of a static walk gives a tile of more than 64 particles two entries; the
pooled walk takes it in two rounds.  Both give the same bits, also where a tile is
gathered from global memory.  The ALE passes take a tile that does not fit the LDS
budget in runs of fewer rows, and one row that does not fit from global memory:
both within the FP32 rounding of the FP64 passes.
"""
import numpy as np
import pytest

import tinysph_old_amd as T
from tests.helpers import rel_l2

pytestmark = pytest.mark.gpu


def crowded(preset, dx, spacing, cells, seed=3):
    """Fluid regathered on a lattice of `spacing` dp over `cells` cells of a column."""
    case = T.build_case(preset, dx=dx, jitter=0.02, seed=seed)
    prm, a, g = case.params, case.arrays, np.random.RandomState(seed)
    fluid = np.nonzero(a["type"] == T.FLUID)[0]
    a["rho"] = 1000.0 + g.normal(0, 2.0, case.np)
    a["v"][fluid] = g.normal(0, 0.5, (len(fluid), 2))
    if spacing:
        kh, d = prm["kap"] * prm["h"], spacing * prm["dp"]
        nx, ny = int(kh / d), int(cells * kh / d)
        xy = np.stack(np.meshgrid(np.arange(nx), np.arange(ny)), -1).reshape(-1, 2)
        at = a["r"][fluid[len(fluid) // 2]].copy()
        a["r"][fluid[-len(xy):]] = at + d * (xy + 0.02 * g.uniform(-1, 1, xy.shape))
    for k in ("r_o", "v_o"):
        a.pop(k, None)
    return case


CROWDS = [(0, 0), (0.8, 7), (0.5, 4), (0.25, 2), (0.15, 1)]


@pytest.mark.parametrize("spacing,cells", CROWDS, ids=str)
@pytest.mark.parametrize("preset,variant", [(T.CASE_DAM_BREAK_MDBC, T.FORCES_WCSPH),
                                            (T.CASE_DAM_BREAK_BT, T.FORCES_BT),
                                            (T.CASE_STILL_WATER_DBC, T.FORCES_DBC)])
def test_walks_give_the_same_bits(preset, variant, spacing, cells):
    case = crowded(preset, 0.012, spacing, cells)
    print(f"[case] preset {preset} spacing {spacing} cells {cells} np={case.np}", flush=True)
    out = []
    for pooled in (False, True):
        with T.system_for_case(case, precision=T.PREC_MIXED) as ps:
            ps.set_balanced(pooled)
            if pooled:
                ps.set_waves_per_cu(1)
            ps.particle_to_cell()
            ps.density_to_pressure()
            ps.compute_forces(variant)
            first = ps.download(("a", "drho"))
            ps.step(case.wall, 1e-7, 9)
            out.append((first, ps.download(), ps.counters()))
    for k, v in out[0][0].items():
        assert np.array_equal(v, out[1][0][k], equal_nan=True), k
    for k, v in out[0][1].items():
        assert np.array_equal(v, out[1][1][k], equal_nan=True), k
    for k in ("pairs", "candidates", "active"):
        assert out[0][2][k] == out[1][2][k], k


@pytest.mark.parametrize("spacing,cells", CROWDS, ids=str)
@pytest.mark.parametrize("rows", [7, 24])
def test_ale_passes_beyond_the_budget(spacing, cells, rows):
    case = crowded(T.CASE_ALE_DAM_BREAK, 0.015, spacing, cells)
    print(f"[case] ale spacing {spacing} cells {cells} rows {rows} np={case.np}", flush=True)
    # a position's rounding in the tile's frame, 6e-8 of up to 26 cells of 2.1 h,
    # against the nearest pairs' distance, beside the sums' own rounding
    near = (spacing or 0.9) * case.params["dp"]
    tol = 1e-5 + 6e-8 * (rows + 2) * 2.1 * case.params["h"] / near
    out = []
    for precision in (T.PREC_FP64, T.PREC_MIXED):
        with T.system_for_case(case, precision=precision) as ps:
            ps.set_tile_rows(rows)
            ps.ale_enable()
            ps.particle_to_cell()
            ps.ale_compute_density(False)
            ps.ale_kernel_gradient()
            out.append((ps.ale_download(), ps.counters()))
    fluid = case.arrays["type"] == T.FLUID
    for k in ("domega", "domegarho", "gradrho", "gradvx", "gradvy"):
        err = rel_l2(out[1][0][k][fluid], out[0][0][k][fluid])
        assert err <= tol, (k, err, tol)
    assert out[0][1]["active"] == out[1][1]["active"]
