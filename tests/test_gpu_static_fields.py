"""Ghost nodes and reference indices, kept by reference position.

The cell builds do not move them; downloads gather them in reference order.  What
was uploaded comes back with its particle after sorting, motion and removals, for
one system (both precisions, runs and single steps) and for each case of a batch.
"""
import numpy as np
import pytest

import tinysph_old_amd as T

pytestmark = pytest.mark.gpu

FIELDS = ("type", "index", "r", "rho", "gnr")


def tagged(case, seed):
    """gnr and index tell the particle; walls keep the ghost nodes they use."""
    a, g = case.arrays, np.random.RandomState(seed)
    fluid = a["type"] == T.FLUID
    a["gnr"][fluid] = g.normal(0, 1, (int(fluid.sum()), 2))
    a["index"] = g.permutation(case.np).astype(np.int32)
    return case


def check(got, a, may_go):
    """The survivors in reference order; only those of may_go may be missing."""
    keep = np.isin(a["index"], got["index"])
    assert np.isin(np.nonzero(~keep)[0], may_go).all()
    assert np.array_equal(got["index"], a["index"][keep])
    assert np.array_equal(got["gnr"], a["gnr"][keep])
    assert np.array_equal(got["type"], a["type"][keep])


@pytest.mark.parametrize("order", [0, 2])
@pytest.mark.parametrize("precision", [T.PREC_FP64, T.PREC_MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("steps", [1, 19])
def test_fields_stay_with_their_particles(precision, order, steps):
    case = tagged(T.build_case(T.CASE_DAM_BREAK_MDBC, dx=0.02, jitter=0.05), 2)
    a, prm = case.arrays, case.params
    fluid = np.nonzero(a["type"] == T.FLUID)[0]
    gone = fluid[[7, 20, len(fluid) // 2]]
    a["r"][gone, 1] = prm["y_m"] + 0.001
    a["v"][gone, 1] = 5.0
    for k in ("r_o", "v_o"):
        a.pop(k, None)
    print(f"[case] static fields np={case.np} precision {precision} order {order}", flush=True)
    with T.system_for_case(case, precision=precision) as ps:
        ps.set_cell_order(order)
        ps.particle_to_cell()
        check(ps.download(FIELDS), a, [])
        ps.step(case.wall, case.dt, steps)
        check(ps.download(FIELDS), a, gone)


@pytest.mark.parametrize("precision", [T.PREC_FP64, T.PREC_MIXED], ids=["fp64", "mixed"])
def test_fields_stay_with_their_particles_in_a_batch(precision):
    cases = [tagged(c, q) for q, c in enumerate(T.build_ensemble(3, 11, 2000, 4000))]
    with T.batch_for_cases(cases, precision) as bs:
        bs.particle_to_cell()
        bs.step(T.WALL_MDBC, 9)
        for q, c in enumerate(cases):
            check(bs.download_case(q, FIELDS), c.arrays, [])
