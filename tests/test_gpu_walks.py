"""Tile walks and tilings against each other, at sizes that really take them.

FP64 passes go by cells up to 70,000 particles, and a walk is pooled from 95 (FP32
pairs) or 150 (FP64) particles per persistent wave; each test asserts the walk it is
about.  Static and pooled passes, the tile depths of FP64 passes (24 rows, and crowds
under 6 rows, are gathered from global memory) and the scan's fallback give the same
bits and counts.
"""
import numpy as np
import pytest

import tinysph_old_amd as T
from oracle import pyoracle as po
from tests.helpers import oracle_for, oracle_init, oracle_variant
from tests.test_gpu_full_tiles import CROWDS, crowded
from tests.test_gpu_tile_lists import tiles

pytestmark = pytest.mark.gpu

STATIC, POOLED = 1, 2
COUNTS = ("pairs", "candidates", "active", "pair_passes")
FP64_CASES = [(T.CASE_DAM_BREAK_MDBC, 0.0031, T.FORCES_WCSPH), (T.CASE_DAM_BREAK_BT, 0.0016, T.FORCES_BT),
              (T.CASE_STILL_WATER_DBC, 0.0027, T.FORCES_DBC)]


def same(x, y):
    for k in x:
        assert np.array_equal(x[k], y[k], equal_nan=True), k


def forces(ps, variant, walk):
    ps.density_to_pressure()
    ps.reset_counters()
    assert ps.pair_walk(variant)[0] == walk
    ps.compute_forces(variant)
    out, c = ps.download(("a", "drho")), ps.counters()
    assert c["scan_stalls"] == 0
    return out, {k: c[k] for k in COUNTS}


@pytest.mark.parametrize("spacing,cells", CROWDS, ids=str)
@pytest.mark.parametrize("preset,dx,variant", [(T.CASE_DAM_BREAK_MDBC, 0.005, T.FORCES_WCSPH),
                                               (T.CASE_DAM_BREAK_BT, 0.0025, T.FORCES_BT),
                                               (T.CASE_STILL_WATER_DBC, 0.004, T.FORCES_DBC)])
def test_mixed_static_and_pooled(preset, dx, variant, spacing, cells):
    """The static list's two entries against the pooled walk's rounds, tiles gathered
    from global memory among them; then whole steps."""
    case = crowded(preset, dx, spacing, cells)
    print(f"[case] mixed preset {preset} spacing {spacing} cells {cells} np={case.np}", flush=True)
    out = []
    for walk in (STATIC, POOLED):
        with T.system_for_case(case, precision=T.PREC_MIXED) as ps:
            ps.set_waves_per_cu(1 if walk == POOLED else 12)
            ps.particle_to_cell()
            if spacing and walk == STATIC:
                assert ps.pair_walk(variant)[1] > len(tiles(ps, ps.tile_rows))
            first, counts = forces(ps, variant, walk)
            ps.reset_counters()
            ps.step(case.wall, 1e-7, 9)
            c = ps.counters()
            out.append((first, counts, ps.download(), {k: c[k] for k in COUNTS}))
    same(out[0][0], out[1][0])
    same(out[0][2], out[1][2])
    assert out[0][1] == out[1][1] and out[0][3] == out[1][3]


@pytest.mark.parametrize("preset,dx,variant", FP64_CASES)
def test_fp64_static_and_pooled(preset, dx, variant):
    """First with the list cut for the walk by the pass, then by a build; then steps."""
    case = T.build_case(preset, dx=dx, jitter=0.1, seed=11)
    print(f"[case] fp64 walks preset {preset} np={case.np}", flush=True)
    out, steps = [], []
    for pooled, waves in ((False, 8), (True, 1), (True, 2), (False, 1)):
        with T.system_for_case(case) as ps:
            ps.particle_to_cell()
            ps.set_balanced(pooled)
            ps.set_waves_per_cu(waves)
            walk = POOLED if pooled and case.np >= 150 * 256 * waves else STATIC
            out.append(forces(ps, variant, walk))
            ps.particle_to_cell()
            out.append(forces(ps, variant, walk))
            if waves != 2:
                ps.step(case.wall, case.dt, 3)
                steps.append(ps.download())
    for o, counts in out[1:]:
        same(o, out[0][0])
        assert counts == out[0][1]
    for s in steps[1:]:
        same(s, steps[0])


@pytest.mark.parametrize("spacing,cells", [(0, 0), (0.5, 4), (0.25, 2)], ids=str)
@pytest.mark.parametrize("preset,dx,variant", FP64_CASES)
def test_fp64_tile_rows(oracle_built, preset, dx, variant, spacing, cells):
    case = crowded(preset, dx, spacing, cells)
    case.params["delta"] = 0.0  # (the diffusion term's root is libm's to an ulp only)
    print(f"[case] fp64 rows preset {preset} spacing {spacing} np={case.np}", flush=True)
    O = oracle_for(case)
    oracle_init(O)
    O.call("density_to_pressure")
    p = O.get(po.F_P)
    O.call("compute_forces", oracle_variant(case.wall))
    want = {"a": O.get(po.F_A), "drho": O.get(po.F_DRHO)}
    case.arrays["p"] = p
    counts = []
    for rows, waves in ((0, 8), (0, 1), (1, 8), (3, 1), (24, 8), (24, 1)):
        with T.system_for_case(case) as ps:
            ps.set_waves_per_cu(waves)
            if rows:
                ps.set_tile_rows(rows)
            ps.particle_to_cell()
            assert ps.pair_walk(variant)[0] == (POOLED if waves == 1 else STATIC)
            ps.reset_counters()
            ps.compute_forces(variant)
            same(ps.download(("a", "drho")), want)
            c = ps.counters()
            counts.append({k: c[k] for k in COUNTS})
    assert all(c == counts[0] for c in counts)


def test_scan_fallback_cuts_the_same_fp64_chunks():
    case = T.build_case(T.CASE_DAM_BREAK_MDBC, dx=0.0031, jitter=0.01, seed=11)
    print(f"[case] fp64 scan fallback np={case.np}", flush=True)
    out = []
    for wait in (1 << 20, -1):
        with T.system_for_case(case) as ps:
            ps.set_scan_wait(wait)
            ps.set_waves_per_cu(1)
            ps.particle_to_cell()
            lists = ps.cell_lists()
            ps.mdbc_density()
            ps.density_to_pressure()
            assert ps.pair_walk(T.FORCES_WCSPH)[0] == POOLED
            ps.compute_forces(T.FORCES_WCSPH)
            first = ps.download(("a", "drho"))
            ps.step(case.wall, case.dt, 5)
            out.append((lists, first, ps.download(), ps.counters()))
    (l0, f0, s0, n0), (l1, f1, s1, n1) = out
    assert np.array_equal(l0[0], l1[0]) and np.array_equal(l0[1], l1[1])
    same(f0, f1)
    same(s0, s1)
    assert n0["scan_stalls"] == 0 and n1["scan_stalls"] > 0
    assert all(n0[k] == n1[k] for k in COUNTS)
