"""FP64 passes by cells over lattices of more particles per cell than the presets'.

Kernel radii from 1.4 to 2.6 spacings take the narrow form, the wide one, and either
of them with neighbourhoods beyond its staged slots.  Pair passes equal the oracle bit
for bit; ALE passes find the pairs that the host counts, and the density gradient is
the sum over them.
"""
import numpy as np
import pytest

import tinysph_old_amd as T
from oracle import pyoracle as po
from tests.helpers import oracle_for, oracle_init, oracle_variant

pytestmark = pytest.mark.gpu

RADII = (1.4, 1.55, 1.6, 1.8, 2.0, 2.2, 2.35, 2.6)


@pytest.fixture(scope="module", autouse=True)
def _oracle(oracle_built):
    return oracle_built


def state(preset, dx, h_dp, crowd):
    case = T.build_case(preset, dx=dx, jitter=0.2, seed=3)
    case.params["h"] = h_dp * case.params["dp"]
    case.params["delta"] = 0.0
    a, g, n = case.arrays, np.random.RandomState(3), case.np
    fluid = np.nonzero(a["type"] == T.FLUID)[0]
    a["v"] = np.where((a["type"] == T.FLUID)[:, None], g.normal(0, 1.0, (n, 2)), 0.0)
    a["rho"] = 1000.0 + g.normal(0, 5.0, n)
    a["p"] = g.normal(0, 3000.0, n)
    if crowd:
        home = a["r"][fluid[len(fluid) // 2]]
        moved = g.choice(fluid, crowd, replace=False)
        a["r"][moved] = home + g.uniform(-0.2, 0.2, (crowd, 2)) * case.params["h"]
    for k in ("r_o", "v_o"):
        a.pop(k, None)
    return case


@pytest.mark.parametrize("crowd", [0, 60])
@pytest.mark.parametrize("h_dp", RADII)
@pytest.mark.parametrize("preset,dx", [(T.CASE_DAM_BREAK_MDBC, 0.015), (T.CASE_DAM_BREAK_BT, 0.008),
                                       (T.CASE_STILL_WATER_DBC, 0.02)])
def test_pair_pass_equals_oracle_bit_for_bit(preset, dx, h_dp, crowd):
    case = state(preset, dx, h_dp, crowd)
    print(f"[case] preset {preset} h/dp {h_dp} crowd {crowd} np={case.np}", flush=True)
    O = oracle_for(case)
    oracle_init(O)
    O.call("compute_forces", oracle_variant(case.wall))
    with T.system_for_case(case) as ps:
        ps.particle_to_cell()
        assert ps.pair_walk(T.forces_variant(case.wall))[0] == 0
        ps.compute_forces(T.forces_variant(case.wall))
        got = ps.download(("a", "drho"))
    assert np.array_equal(got["a"], O.get(po.F_A), equal_nan=True)
    assert np.array_equal(got["drho"], O.get(po.F_DRHO), equal_nan=True)


def neighbours(case):
    """Ordered pairs (i fluid, j) with qq <= 2, i != j, in blocks."""
    r, h = case.arrays["r"], case.params["h"]
    fluid = np.nonzero(case.arrays["type"] == T.FLUID)[0]
    out = []
    for i0 in range(0, len(fluid), 256):
        i = fluid[i0:i0 + 256]
        x, y = r[i, None, 0] - r[None, :, 0], r[i, None, 1] - r[None, :, 1]
        qq = np.sqrt(x * x + y * y) / h
        near = qq <= 2
        near[np.arange(len(i)), i] = False
        a, b = np.nonzero(near)
        out.append((i[a], b, x[near], y[near], qq[near]))
    return [np.concatenate(z) for z in zip(*out)]


@pytest.mark.parametrize("crowd", [0, 60])
@pytest.mark.parametrize("h_dp", RADII)
def test_ale_passes(h_dp, crowd):
    case = state(T.CASE_ALE_DAM_BREAK, 0.02, h_dp, crowd)
    print(f"[case] ale h/dp {h_dp} crowd {crowd} np={case.np}", flush=True)
    out = []
    with T.system_for_case(case) as ps:
        ps.ale_enable()
        ps.particle_to_cell()
        for job in (ps.ale_kernel_gradient, lambda: ps.ale_compute_density(True),
                    lambda: ps.ale_compute_acceleration(True), ps.rale_forces,
                    lambda: ps.ale_compute_density(False), lambda: ps.ale_compute_acceleration(False)):
            ps.reset_counters()
            job()
            out.append(ps.counters())
            if len(out) == 1:
                grad = ps.ale_download()
    i, j, x, y, qq = neighbours(case)
    for c in out:
        assert c["pairs"] == len(i)
        assert c["active"] == int((case.arrays["type"] == T.FLUID).sum())
    # the density gradient's terms over fluid neighbours and walls in 64 bits; the
    # kernel's factors are rounded to 32 bits on the way (2^-24 each, four of them),
    # against the sum of the terms' magnitudes
    a, prm = case.arrays, case.params
    h, dp = prm["h"], prm["dp"]
    bw, aw = float(np.float32(-2.7852 / h ** 3)), float(np.float32(0.557 / h ** 2))
    w1 = 1 - qq / 2
    with np.errstate(invalid="ignore", divide="ignore"):
        f = np.where(qq > 0, bw * qq * w1 ** 3 / (qq * h), 0.0)
    w = aw * (2 * qq + 1) * w1 ** 4
    wall = a["type"][j] == T.WALL
    d = a["rho"][j] - a["rho"][i]
    for c, dr in ((0, x), (1, y)):
        t = np.where(wall, -d * a["n"][j, c] * w * dp, d * dp * dp * dr * f) * 2
        s, mag = np.bincount(i, t, case.np), np.bincount(i, np.abs(t), case.np)
        assert (np.abs(grad["gradrho"][:, c] - s) <= 1e-6 * mag + 1e-300).all()
