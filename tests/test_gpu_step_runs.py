"""A run of steps taken from one graph equals the same steps taken one by one.

Inside a graph of several steps the second cell build of a step also takes the
hash of the next step's first build and the wall densities run beside that
build's scan; single steps launch the hash itself.  Every field and counter is
the same bits, for each wall treatment and precision, both in-cell orderings,
with particles that leave the domain on the way, and in a batch.
"""
import numpy as np
import pytest

import tinysph_old_amd as T

pytestmark = pytest.mark.gpu

FIELDS = ("type", "index", "p", "rho", "drho", "r", "v", "a", "r_o", "v_o", "rho_o")
STEPS = 21  # two graphs of eight steps and five single steps
COUNTS = ("pairs", "candidates", "active", "removed", "outside_grid", "density_out_of_range")


def launched(ps, wall, dt, run):
    ps.particle_to_cell()
    for n in ([STEPS] if run else [1] * STEPS):
        ps.step(wall, dt, n) if dt is not None else ps.step(wall, n)
    return ps.counters()


def escape(case):
    """A few fluid particles fly off over the top and one through the side."""
    fluid = np.nonzero(case.arrays["type"] == T.FLUID)[0]
    gone = fluid[[3, 4, 5, 40, len(fluid) // 2, len(fluid) // 2 + 1]]
    prm, r, v = case.params, case.arrays["r"], case.arrays["v"]
    r[gone, 1] = prm["y_m"] - 0.3 * prm["dp"] - 0.2 * prm["dp"] * np.arange(len(gone))
    v[gone, 1] = 0.02 / (STEPS * case.dt) * (1.0 + 0.1 * np.arange(len(gone)))
    for k in ("r_o", "v_o"):
        case.arrays.pop(k, None)


@pytest.mark.parametrize("order", [1, 2])
@pytest.mark.parametrize("precision", [T.PREC_FP64, T.PREC_MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("preset,dx", [(T.CASE_STILL_WATER_DBC, 0.02), (T.CASE_DAM_BREAK_MDBC, 0.02),
                                       (T.CASE_DAM_BREAK_BT, 0.01)])
def test_run_equals_single_steps(preset, dx, precision, order):
    case = T.build_case(preset, dx=dx, jitter=0.05, seed=3)
    escape(case)
    print(f"[case] preset {preset} np={case.np} precision {precision} order {order}", flush=True)
    out = []
    for run in (False, True):
        with T.system_for_case(case, precision=precision) as ps:
            ps.set_cell_order(order)
            cnt = launched(ps, case.wall, case.dt, run)
            out.append((ps.download(FIELDS), cnt))
    (a, ca), (b, cb) = out
    assert ca["removed"] > 0
    for k in FIELDS:
        assert np.array_equal(a[k], b[k], equal_nan=True), k
    for k in COUNTS:
        assert ca[k] == cb[k], k


@pytest.mark.parametrize("precision", [T.PREC_FP64, T.PREC_MIXED], ids=["fp64", "mixed"])
def test_batch_run_equals_single_steps(precision):
    cases = T.build_ensemble(4, 77, 2000, 5000)
    out = []
    for run in (False, True):
        with T.batch_for_cases(cases, precision) as bs:
            cnt = launched(bs, T.WALL_MDBC, None, run)
            out.append(([bs.download_case(q, FIELDS) for q in range(4)], cnt))
    (a, ca), (b, cb) = out
    for q in range(4):
        for k in FIELDS:
            assert np.array_equal(a[q][k], b[q][k]), (q, k)
    for k in COUNTS:
        assert ca[k] == cb[k], k


@pytest.mark.parametrize("precision", [T.PREC_FP64, T.PREC_MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("kind", ["rale", "ale", "leapfrog"])
def test_other_steps_in_runs(kind, precision):
    """Riemann-ALE, ALE-SPH MUSCL and leap-frog steps, the first one included."""
    preset = T.CASE_DAM_BREAK_MDBC if kind == "leapfrog" else T.CASE_ALE_DAM_BREAK
    case = T.build_case(preset, dx=0.02, jitter=0.05, seed=5)
    print(f"[case] {kind} np={case.np} precision {precision}", flush=True)
    out = []
    for run in (False, True):
        with T.system_for_case(case, precision=precision) as ps:
            if kind == "leapfrog":
                ps.history_enable()
            else:
                ps.ale_enable()
            ps.particle_to_cell()
            first = 1
            for n in ([STEPS] if run else [1] * STEPS):
                if kind == "rale":
                    ps.step_rale(case.dt, first, n)
                elif kind == "ale":
                    ps.step_ale(case.dt, first, n, T.MUSCL_MINMOD)
                else:
                    ps.step_leapfrog(case.wall, case.dt, first, n)
                first += n
            more = {} if kind == "leapfrog" else ps.ale_download()
            out.append((ps.download(FIELDS), more, ps.counters()))
    (a, ea, ca), (b, eb, cb) = out
    for k in FIELDS:
        assert np.array_equal(a[k], b[k], equal_nan=True), k
    for k in ea:
        assert np.array_equal(ea[k], eb[k], equal_nan=True), k
    for k in COUNTS:
        assert ca[k] == cb[k], k
