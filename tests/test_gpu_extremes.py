"""FP64 pair passes over states that hold a zero, infinite or NaN density, pressure
or velocity.

A particle's values reach those within 2h of it and no others: whoever lies farther
away, be it by a rounding error, gets the same bits as from the state without it,
also where a crowded neighbourhood is gathered from global memory.  Sizes take every
walk (by cells, tiles, pooled tiles).
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


def state(preset, dx, crowd):
    """A random state, `crowd` more particles around one cell, and the one to spoil."""
    case = T.build_case(preset, dx=dx, jitter=0.2, seed=7)
    a, g, n = case.arrays, np.random.RandomState(5), case.np
    fluid = np.nonzero(a["type"] == T.FLUID)[0]
    a["v"] = np.where((a["type"] == T.FLUID)[:, None], g.normal(0, 1.0, (n, 2)), 0.0)
    a["rho"] = 1000.0 + g.normal(0, 5.0, n)
    a["p"] = g.normal(0, 3000.0, n)
    home, h = a["r"][fluid[len(fluid) // 2]].copy(), case.params["h"]
    if crowd:
        moved = g.choice(fluid[:len(fluid) // 3], crowd, replace=False)
        a["r"][moved] = home + g.uniform(-0.2, 0.2, (crowd, 2)) * h
    for k in ("r_o", "v_o"):
        a.pop(k, None)
    # beyond the crowd's support, in a cell beside it; another just beyond its own
    d = np.hypot(*(a["r"] - home).T)
    b = fluid[(d[fluid] > 2.3 * h) & (d[fluid] < 2.8 * h)][0]
    a["r"][fluid[1]] = a["r"][b] + 2 * h * (1 + 2e-13) * np.array([0.6, 0.8])
    return case, b


def forces(case, waves):
    with T.system_for_case(case) as ps:
        if waves:
            ps.set_waves_per_cu(waves)
        ps.particle_to_cell()
        ps.compute_forces(T.forces_variant(case.wall))
        return ps.download(("a", "drho"))


# by cells; tiles; pooled tiles
SIZES = {T.CASE_DAM_BREAK_MDBC: (0.012, 0.0033), T.CASE_DAM_BREAK_BT: (0.0101, 0.0015),
         T.CASE_STILL_WATER_DBC: (0.0101, 0.0026)}


WALKS = [(p, w, c) for p in sorted(SIZES) for w in ("cells", "tiles", "pooled") for c in (0, 140)]


def spoilt(preset, walk, crowd):
    """The case, its forces, and for each spoilt value the case's forces with it."""
    dx, waves = SIZES[preset][walk != "cells"], 1 if walk == "pooled" else 0
    case, b = state(preset, dx, crowd)
    print(f"[case] preset {preset} {walk} crowd {crowd} np={case.np}", flush=True)
    a = case.arrays
    x, y = (a["r"] - a["r"][b]).T
    qq = np.sqrt(x * x + y * y) / case.params["h"]
    assert ((qq > 2) & (qq < 2 * (1 + 4e-13))).any()

    def each():
        for field, values in (("rho", (0.0, np.inf, np.nan)), ("p", (np.inf, np.nan)),
                              ("v", (np.inf, -np.inf, np.nan))):
            for value in values:
                kept = a[field].copy()
                a[field].reshape(case.np, -1)[b, 0] = value
                yield (field, value), forces(case, waves)
                a[field] = kept

    return case, qq, forces(case, waves), each()


@pytest.mark.parametrize("preset,walk,crowd", WALKS)
def test_spoilt_particle_reaches_its_support_only(preset, walk, crowd):
    case, qq, clean, each = spoilt(preset, walk, crowd)
    for what, got in each:
        for k in got:
            assert np.array_equal(got[k][qq > 2], clean[k][qq > 2], equal_nan=True), (what, k)


@pytest.mark.parametrize("preset,walk,crowd", WALKS)
def test_sums_over_a_spoilt_particle_are_the_oracles(preset, walk, crowd):
    """Within 2h: the same infinities, and NaN where the oracle's expressions give NaN.
    (No other value is spoilt, so the oracle's sums over nine cells differ from sums
    over the support by exact zeros.)"""
    case, qq, _, each = spoilt(preset, walk, crowd)
    inside = (qq <= 2) & (qq > 0)
    for what, got in each:
        O = oracle_for(case)
        oracle_init(O)
        O.call("compute_forces", oracle_variant(case.wall))
        for k, ref in (("a", O.get(po.F_A)), ("drho", O.get(po.F_DRHO))):
            x, y = got[k][inside], ref[inside]
            assert np.array_equal(np.isnan(x), np.isnan(y)), (what, k)
            inf = np.isinf(y)
            assert np.array_equal(np.isinf(x), inf) and np.array_equal(x[inf], y[inf]), (what, k)
