"""FP32 ALE passes under budgets of LDS records from the least to the most.

The budget follows the waves per compute unit; a tile beyond it is taken in runs of
rows of the same frame, and one row beyond it from global memory.  The bits do not
depend on it.
"""
import numpy as np
import pytest

import tinysph_old_amd as T
from tests.test_gpu_full_tiles import CROWDS, crowded

pytestmark = pytest.mark.gpu


def check(case):
    out = []
    for waves in (1, 5, 8, 11, 12, 13, 24):
        with T.system_for_case(case, precision=T.PREC_MIXED) as ps:
            ps.set_waves_per_cu(waves)
            ps.ale_enable()
            ps.particle_to_cell()
            ps.ale_kernel_gradient()
            ps.ale_compute_density(True)
            ps.ale_compute_acceleration(True)
            out.append((ps.ale_download(), ps.counters()))
    for fields, counts in out[1:]:
        for k, v in out[0][0].items():
            assert np.array_equal(v, fields[k], equal_nan=True), k
        for k in ("pairs", "candidates", "active"):
            assert counts[k] == out[0][1][k], k


@pytest.mark.parametrize("spacing,cells", CROWDS, ids=str)
def test_bits_do_not_depend_on_the_waves(spacing, cells):
    case = crowded(T.CASE_ALE_DAM_BREAK, 0.0042, spacing, cells)
    print(f"[case] ale budget spacing {spacing} cells {cells} np={case.np}", flush=True)
    check(case)


@pytest.mark.parametrize("h_dp", [1.6, 2.0, 2.5, 3.0])
def test_full_lattices(h_dp):
    """Every tile beyond the budget: runs of several rows, of one, none."""
    case = crowded(T.CASE_ALE_DAM_BREAK, 0.0075, 0, 0)
    case.params["h"] = h_dp * case.params["dp"]
    print(f"[case] ale budget h/dp {h_dp} np={case.np}", flush=True)
    check(case)
