"""The entries of the tile lists that mixed builds leave.

A list for static walks gives a tile of more than 64 particles two entries, one for a
pooled walk none (it would have to be listed anew), whatever pass the build precedes:
counted against the cell lists.
"""
import numpy as np
import pytest

import tinysph_old_amd as T
from tests.test_gpu_full_tiles import crowded

pytestmark = pytest.mark.gpu


def tiles(ps, rows):
    """Particles of each non-empty tile (`rows` cells of a grid column)."""
    ncx, ncy = ps.grid()
    count = np.diff(ps.cell_lists()[0]).reshape(ncx, ncy)
    own = np.add.reduceat(count, np.arange(0, ncy, rows), axis=1).ravel()
    return own[own > 0]


@pytest.mark.parametrize("waves", [1, 12])
@pytest.mark.parametrize("preset,dx,variant", [(T.CASE_DAM_BREAK_MDBC, 0.005, T.FORCES_WCSPH),
                                               (T.CASE_DAM_BREAK_BT, 0.0025, T.FORCES_BT),
                                               (T.CASE_STILL_WATER_DBC, 0.004, T.FORCES_DBC)])
def test_entries_follow_the_walk(preset, dx, variant, waves):
    case = crowded(preset, dx, 0.5, 4)
    print(f"[case] preset {preset} waves {waves} np={case.np}", flush=True)
    with T.system_for_case(case, precision=T.PREC_MIXED) as ps:
        ps.set_waves_per_cu(waves)
        for _ in range(2):
            ps.particle_to_cell()
            own = tiles(ps, ps.tile_rows)
            full = int((own > 64).sum())
            assert full > 0
            walk, entries = ps.pair_walk(variant)
            assert walk == (2 if waves == 1 else 1)
            assert entries == len(own) + (0 if walk == 2 else full)
            ps.density_to_pressure()
            ps.compute_forces(variant)
            assert ps.pair_walk(variant) == (walk, entries)


@pytest.mark.parametrize("h_dp,split", [(2 ** 0.5, True), (1.6, False)])
def test_entries_of_ale_systems(h_dp, split):
    """Beyond the pooled walk's limit: two entries where few tiles are that full."""
    case = crowded(T.CASE_ALE_DAM_BREAK, 0.005, 0.5, 4)
    case.params["h"] = h_dp * case.params["dp"]
    print(f"[case] ale h/dp {h_dp} np={case.np}", flush=True)
    with T.system_for_case(case, precision=T.PREC_MIXED) as ps:
        ps.set_waves_per_cu(1)
        ps.ale_enable()
        ps.particle_to_cell()
        own = tiles(ps, ps.tile_rows)
        assert ps.pair_walk(T.FORCES_BT)[1] == len(own) + (int((own > 64).sum()) if split else 0)
