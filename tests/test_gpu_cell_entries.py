"""The lists that FP64 builds leave: non-empty cells where passes go by cells, else tiles.

Counted against the cell lists, for both ways of ordering the cells; a context whose
passes want one and the other in turn (ALE passes go by cells at any size, the WCSPH
ones up to 70,000 particles) lists anew and gives each pass the bits it has alone.
"""
import numpy as np
import pytest

import tinysph_old_amd as T
from tests.test_gpu_tile_lists import tiles

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", [0, 2])
@pytest.mark.parametrize("dx,walk", [(0.02, 0), (0.0036, 0), (0.0033, 1)])
def test_entries_of_fp64_builds(dx, walk, order):
    case = T.build_case(T.CASE_DAM_BREAK_MDBC, dx=dx, jitter=0.1, seed=5)
    print(f"[case] fp64 entries np={case.np} order {order}", flush=True)
    with T.system_for_case(case) as ps:
        ps.set_cell_order(order)
        for _ in range(2):
            ps.particle_to_cell()
            cells = np.count_nonzero(np.diff(ps.cell_lists()[0]))
            want = len(tiles(ps, ps.tile_rows)) if walk else cells
            assert ps.pair_walk(T.FORCES_WCSPH) == (walk, want)
            ps.density_to_pressure()
            ps.compute_forces(T.FORCES_WCSPH)
            assert ps.pair_walk(T.FORCES_WCSPH) == (walk, want)
            ps.set_tile_rows(5)  # lists of cells do not depend on it
            ps.compute_forces(T.FORCES_WCSPH)
            assert ps.pair_walk(T.FORCES_WCSPH)[1] == (len(tiles(ps, 5)) if walk else cells)


@pytest.mark.parametrize("ale_first", [True, False])
def test_walks_in_turn(ale_first):
    case = T.build_case(T.CASE_DAM_BREAK_BT, dx=0.0015, jitter=0.1, seed=5)
    assert case.np > 70000
    print(f"[case] walks in turn np={case.np}", flush=True)

    def wcsph(ps):
        ps.density_to_pressure()
        ps.compute_forces(T.FORCES_BT)
        return ps.download(("a", "drho"))

    def rale(ps):
        ps.rale_forces()
        f = ps.ale_download()
        return {k: f[k] for k in ("domega", "domegarho", "domegav")}

    alone = []
    for job in (wcsph, rale):
        with T.system_for_case(case) as ps:
            if job is rale:
                ps.ale_enable()
            ps.particle_to_cell()
            alone.append(job(ps))
    with T.system_for_case(case) as ps:
        if ale_first:
            ps.ale_enable()
        ps.particle_to_cell()
        if not ale_first:
            ps.ale_enable()
        for job, want in ((rale, alone[1]), (wcsph, alone[0]), (wcsph, alone[0]), (rale, alone[1])):
            got = job(ps)
            for k in want:
                assert np.array_equal(got[k], want[k], equal_nan=True), k
        ps.step(case.wall, 1e-7, 9)
        ps.step_rale(1e-7, 1, 9)
        assert np.isfinite(ps.download(("r",))["r"]).all()
