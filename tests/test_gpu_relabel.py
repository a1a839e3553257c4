"""Relabelled reference positions with walls behind fluid that has left.

Walls uploaded after fluid change their position when removed fluid is relabelled
away.  Each keeps its own ghost node: the wall densities, the steps and the fields
kept by position are those of a run without the relabel, bit for bit, for a call
between two stages, between runs of steps and in a run with an inlet.
"""
import numpy as np
import pytest

import tinysph_old_amd as T

pytestmark = pytest.mark.gpu

FIELDS = ("type", "index", "r", "v", "rho", "p", "a", "drho", "gnr")


def fluid_first(preset, dx, seed=4):
    """Fluid before the walls, some of it on the way out of the domain."""
    case = T.build_case(preset, dx=dx, jitter=0.05, seed=seed)
    a, prm = case.arrays, case.params
    order = np.argsort(a["type"] == T.WALL, kind="stable")
    for k in list(a):
        a[k] = a[k][order]
    a["index"] = np.random.RandomState(seed).permutation(case.np).astype(np.int32)
    loose = np.nonzero(a["type"] == T.FLUID)[0][[3, 11, 12, 40]]
    a["r"][loose, 1] = prm["y_m"] + 0.001
    a["v"][loose, 1] = 5.0
    for k in ("r_o", "v_o"):
        a.pop(k, None)
    return case


def same(x, y):
    for k in x:
        assert np.array_equal(x[k], y[k], equal_nan=True), k


@pytest.mark.parametrize("order", [0, 2])
@pytest.mark.parametrize("precision", [T.PREC_FP64, T.PREC_MIXED], ids=["fp64", "mixed"])
def test_wall_densities_after_a_relabel(precision, order):
    case = fluid_first(T.CASE_DAM_BREAK_MDBC, 0.02)
    print(f"[case] relabel np={case.np} precision {precision} order {order}", flush=True)
    out = []
    for relabel in (False, True):
        with T.system_for_case(case, precision=precision) as ps:
            ps.set_cell_order(order)
            ps.particle_to_cell()
            ps.step(case.wall, case.dt, 19)
            assert ps.counters()["removed"] > 0
            if relabel:
                ps.renumber()
            got = [ps.download(FIELDS)]
            ps.mdbc_density()
            got.append(ps.download(FIELDS))
            if relabel:
                ps.renumber()
            ps.step(case.wall, case.dt, 19)
            got.append(ps.download(FIELDS))
            out.append(got)
    walls = out[0][1]["type"] == T.WALL
    assert np.ptp(out[0][1]["rho"][walls]) > 0  # the ghost nodes matter
    for x, y in zip(*out):
        same(x, y)


@pytest.mark.parametrize("precision", [T.PREC_FP64, T.PREC_MIXED], ids=["fp64", "mixed"])
def test_inflow_steps_after_a_relabel(precision):
    case = fluid_first(T.CASE_INFLOW_CHANNEL, 0.02)
    print(f"[case] relabelled inflow np={case.np} precision {precision}", flush=True)
    out = []
    for relabel in (False, True):
        with T.system_for_case(case, precision=precision) as ps:
            ps.particle_to_cell()
            for _ in range(3):
                ps.step_inflow(case.wall, case.dt, 40)
                if relabel:
                    ps.renumber()
            c = ps.counters()
            assert c["removed"] > 0 and c["zone_rejected"] == 0
            out.append(ps.download(FIELDS))
    same(*out)


@pytest.mark.parametrize("n", [1, 33, 8193, 131073, 300001])
def test_relabel_with_removed_particles_still_in_their_slots(n):
    """A relabel between the removal decision and the build that drops the particles:
    every field stays with its particle, and the next decisions (every other one of a
    run of candidates) are those without the relabel."""
    g = np.random.RandomState(n)
    arrays = {k: g.rand(n, 2) for k in ("r", "v", "gnr", "n")}
    arrays["rho"] = 1000.0 + g.rand(n)
    arrays["type"] = np.where(g.rand(n) < 0.2, T.WALL, T.FLUID).astype(np.int32)
    arrays["index"] = g.permutation(n).astype(np.int32)
    out = g.rand(n) < 0.3  # runs of candidates among them
    arrays["r"][out, 0] = 1.1 + 0.015
    prm = {"h": 0.01, "kap": 2.0, "cs": 20.0, "rho0": 1000.0, "avisc": 0.01, "delta": 0.1, "dp": 0.01,
           "x_0": -0.1, "x_m": 1.1, "y_0": -0.1, "y_m": 1.1}
    print(f"[case] relabel of {n} particles, {int(out.sum())} of them leaving", flush=True)
    fields = ("type", "index", "r", "v", "rho", "gnr", "n")
    got = []
    for relabel in (False, True):
        some = []
        with T.ParticleSystem(prm, capacity=n) as ps:
            ps.upload(arrays)
            ps.particle_to_cell()
            for _ in range(3):
                ps.remove_out_of_domain()
                if relabel:
                    ps.renumber()
                some.append(ps.download(fields))
                ps.particle_to_cell()
                if relabel:
                    ps.renumber()
                some.append(ps.download(fields))
            got.append((some, ps.counters()["removed"]))
    assert got[0][1] == got[1][1] and (n == 1 or got[0][1] > 0)
    for x, y in zip(got[0][0], got[1][0]):
        same(x, y)
