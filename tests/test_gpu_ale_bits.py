"""The FP64 ALE pair passes against the oracle, bit for bit.

Compute_Density, Kernel_gradient_approx and the volume and density rates of the
first-order Riemann pass use no power function, so one pass over the same
state gives the oracle's bits (the acceleration's sound speed and the Riemann
pass's pressure go through libm's pow there; other tests hold those to 1e-9).
Random velocities and densities, every limiter mode, sizes from a few hundred
particles, cells crowded beyond the LDS budget and beyond a wavefront, and a
sparse domain whose grid is walked by its list of occupied tiles.
"""
import numpy as np
import pytest

import tinysph_old_amd as T
from oracle import pyoracle as po
from tests.helpers import oracle_ale

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _oracle(oracle_built):
    return oracle_built


def state(dx, crowd=0, wide=0.0):
    case = T.build_case(T.CASE_ALE_DAM_BREAK, dx=dx, jitter=0.2, seed=3)
    g = np.random.RandomState(5)
    a, fluid = case.arrays, case.arrays["type"] == T.FLUID
    a["v"] = np.where(fluid[:, None], g.normal(0, 1.0, (case.np, 2)), 0.0)
    a["rho"] = 1000.0 + g.normal(0, 5.0, case.np)
    if crowd:
        at = np.nonzero(fluid)[0]
        moved = g.choice(at, crowd, replace=False)
        a["r"][moved] = a["r"][at[len(at) // 2]] + g.uniform(-0.2, 0.2, (crowd, 2)) * case.params["h"]
    if wide:
        case.params["x_m"] = case.params["x_0"] + wide
        case.params["y_m"] = case.params["y_0"] + wide
    return case


CASES = [dict(dx=0.1), dict(dx=0.031), dict(dx=0.006), dict(dx=0.03, crowd=12), dict(dx=0.03, crowd=40),
         dict(dx=0.03, crowd=100), dict(dx=0.02, wide=64.0)]


def same(ps, O, names):
    g = ps.ale_download()
    for k in names:
        assert np.array_equal(g[k], O.get(getattr(po, "F_" + k.upper())), equal_nan=True), k


@pytest.mark.parametrize("kw", CASES, ids=str)
@pytest.mark.parametrize("limited", [False, True])
def test_density_and_gradient_passes(kw, limited):
    case = state(**kw)
    print(f"[case] ale {kw} np={case.np} limited={limited}", flush=True)
    O = oracle_ale(case)
    sfx = "_limited" if limited else ""
    with T.system_for_case(case) as ps:
        ps.ale_enable()
        ps.particle_to_cell()
        for _ in range(2):  # gradients of zero, then the pass's own
            ps.ale_compute_density(limited)
            O.call("ale_compute_density" + sfx)
            ps.ale_kernel_gradient()
            O.call("ale_kernel_gradient")
            same(ps, O, ("domega", "domegarho", "gradrho", "gradvx", "gradvy"))


@pytest.mark.parametrize("kw", CASES, ids=str)
def test_riemann_pass_rates(kw):
    case = state(**kw)
    print(f"[case] rale {kw} np={case.np}", flush=True)
    O = oracle_ale(case)
    with T.system_for_case(case) as ps:
        ps.ale_enable()
        ps.particle_to_cell()
        ps.rale_forces()
        O.call("rale_forces")
        same(ps, O, ("domega", "domegarho"))
