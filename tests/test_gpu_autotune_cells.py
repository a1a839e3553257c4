"""The autotuner where the pair pass goes by cells.

FP64 passes of up to 70,000 particles do not depend on the tile settings, so there is
nothing to choose by time: the tuner keeps the context's settings, and rows that
follow the particle count by default go on following it.
"""
import pytest

import tinysph_old_amd as T

pytestmark = pytest.mark.gpu


def balanced_rows_waves(ps):
    rows, waves, bal, ms = T.autotune(ps, T.FORCES_WCSPH)
    assert ms > 0
    return bal, rows, waves


def test_settings_are_kept():
    case = T.build_case(T.CASE_DAM_BREAK_MDBC, dx=0.012, jitter=0.02)
    print(f"[case] autotune by cells np={case.np}", flush=True)
    with T.system_for_case(case) as ps:
        ps.particle_to_cell()
        rows = ps.tile_rows
        assert balanced_rows_waves(ps) == (1, rows, 8) and ps.tile_rows == rows
        ps.set_tile_rows(11)
        ps.set_waves_per_cu(3)
        ps.set_balanced(False)
        assert balanced_rows_waves(ps) == (0, 11, 3) and ps.tile_rows == 11


def test_default_rows_follow_the_particle_count():
    """6 rows below 150 particles per persistent wave (38,400 at one wave per compute
    unit of 256), 7 above."""
    small = T.build_case(T.CASE_DAM_BREAK_MDBC, dx=0.012, jitter=0.02)
    large = T.build_case(T.CASE_DAM_BREAK_MDBC, dx=0.004, jitter=0.02)
    print(f"[case] default rows np={small.np}, {large.np}", flush=True)
    assert small.np < 38400 < large.np < 70000
    with T.ParticleSystem(large.params, capacity=large.np) as ps:
        ps.set_waves_per_cu(1)
        ps.upload(small.arrays)
        ps.particle_to_cell()
        assert ps.tile_rows == 6
        assert balanced_rows_waves(ps) == (1, 6, 1)
        ps.upload(large.arrays)
        assert ps.tile_rows == 7
