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


@pytest.mark.parametrize("precision,dx", [(T.PREC_FP64, 0.0033), (T.PREC_MIXED, 0.005)], ids=["fp64", "mixed"])
def test_passes_stage_by_stage(precision, dx):
    """A build cuts the chunks for a pass of the last variant; one of another variant, of
    other settings or without a pass between gives the same bits as the static walk."""
    case = crowded(T.CASE_DAM_BREAK_MDBC, dx, 0.8, 7)
    print(f"[case] stage by stage np={case.np} precision {precision}", flush=True)
    out = []
    for pooled in (True, False):
        got = []
        with T.system_for_case(case, precision=precision) as ps:
            ps.set_balanced(pooled)
            ps.set_waves_per_cu(1)
            for variant in (T.FORCES_WCSPH, T.FORCES_WCSPH, T.FORCES_DBC, T.FORCES_DBC, T.FORCES_WCSPH):
                ps.particle_to_cell()
                assert ps.pair_walk(variant)[0] == (2 if pooled else 1)
                ps.density_to_pressure()
                ps.compute_forces(variant)
                got.append(ps.download(("a", "drho")))
            ps.particle_to_cell()
            ps.particle_to_cell()
            ps.density_to_pressure()
            if pooled:  # fewer chunks than the build has cut
                ps.set_balanced(False)
                ps.compute_forces(T.FORCES_WCSPH)
                ps.set_balanced(True)
            ps.compute_forces(T.FORCES_WCSPH)
            got.append(ps.download(("a", "drho")))
            out.append(got)
    for x, y in zip(*out):
        for k in x:
            assert np.array_equal(x[k], y[k], equal_nan=True), k
