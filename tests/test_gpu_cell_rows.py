"""Cell lists ranked from the hash's rows, where cells hold more than a row.

A row holds 16 to 128 seqs by the particles that the lattice puts in a cell; what
a cell holds beyond its row is chained from heads that cells 4096 apart share.
The lists equal the oracle's for cells of every fill about the row's edges, build
after build over new positions, and the steps from them equal, in every bit, the
steps whose cells are ordered by passes of their own.
"""
import numpy as np
import pytest

import tinysph_old_amd as T
from tests.helpers import oracle_for, oracle_init

pytestmark = pytest.mark.gpu

FILLS = (0, 1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 129, 300)


@pytest.fixture(scope="module", autouse=True)
def _oracle(oracle_built):
    return oracle_built


def clumped(scale, seed):
    """The dam break with its fluid regathered: cell 40 + 61 q and the cell 4096
    on (where the grid has it) get FILLS[q] particles each."""
    case = T.build_case(T.CASE_DAM_BREAK_MDBC, dx=0.01, jitter=0.01)
    prm, r = case.params, case.arrays["r"]
    prm["h"] *= scale
    kh = prm["kap"] * prm["h"]
    of = 0.273 * prm["h"]  # the grid's offset, src/SPH_find_pairs.h:13
    with T.system_for_case(case) as ps:
        ncx, ncy = ps.grid()
    rng = np.random.default_rng(seed)
    fluid = iter(rng.permutation(np.nonzero(case.arrays["type"] == T.FLUID)[0]))
    for q, fill in enumerate(FILLS):
        for cell in (40 + 61 * q, 40 + 61 * q + 4096):
            cx, cy = divmod(cell, ncy)
            if cx >= ncx - 1:
                continue
            for i in [p for _, p in zip(range(fill), fluid)]:
                r[i] = ((cx + rng.uniform(0.2, 0.8)) * kh + prm["x_0"] - of,
                        (cy + rng.uniform(0.2, 0.8)) * kh + prm["y_0"] - of)
    for k in ("r_o", "v_o"):
        case.arrays.pop(k, None)
    return case


@pytest.mark.parametrize("scale", [1.0, 1.7, 2.6, 3.4], ids=["16", "64", "128", "none"])
def test_lists_of_full_cells(scale):
    cases = [clumped(scale, seed) for seed in (1, 2, 3)]
    print(f"[case] clumped dam break scale {scale} np={cases[0].np}", flush=True)
    with T.system_for_case(cases[0]) as ps:
        for case in cases:
            ps.upload(case.arrays)
            O = oracle_for(case)
            oracle_init(O)
            s_o, it_o = O.cell_csr()
            for _ in range(3):
                ps.particle_to_cell()
                s, it = ps.cell_lists()
                assert np.array_equal(s, s_o) and np.array_equal(it, it_o)


@pytest.mark.parametrize("precision", [T.PREC_FP64, T.PREC_MIXED], ids=["fp64", "mixed"])
def test_steps_with_full_cells(precision):
    case = clumped(1.0, 4)
    print(f"[case] clumped dam break steps, precision {precision}", flush=True)
    out = []
    for mode in (0, 1, 2):
        with T.system_for_case(case, precision=precision) as ps:
            ps.set_cell_order(mode)
            ps.particle_to_cell()
            ps.step(case.wall, 1e-7, 17)
            out.append(ps.download())
    for got in out[:2]:
        for k, v in out[2].items():
            assert np.array_equal(got[k], v, equal_nan=True), k
