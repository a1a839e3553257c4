"""Cell builds whose scan runs in the reorder's launch, at the edges of its range.

On grids of up to 65536 cells the reorder finds its cells' offsets from sums over
16 cells, beside the scan; larger grids scan first.  Both give the oracle's cell
lists: grids of one bin, of a bin's and a scan round's edge, and on either side of
the limit; particles in the first and the last cells, and none in most others.
"""
import numpy as np
import pytest

import tinysph_old_amd as T
from tests.helpers import oracle_for, oracle_init

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _oracle(oracle_built):
    return oracle_built


@pytest.mark.parametrize("ncx,ncy", [(3, 5), (4, 4), (128, 128), (127, 129), (129, 128), (256, 256),
                                     (255, 257), (257, 256), (509, 521)])
@pytest.mark.parametrize("wait", [1 << 20, -1], ids=["wait", "nowait"])
def test_lists_on_grids_about_the_limit(ncx, ncy, wait):
    case = T.build_case(T.CASE_DAM_BREAK_MDBC, dx=0.02, jitter=0.01)
    prm, r = case.params, case.arrays["r"]
    kh, of = prm["kap"] * prm["h"], 0.273 * prm["h"]
    prm["x_m"], prm["y_m"] = (prm["x_0"] + (ncx - 0.5) * kh - of, prm["y_0"] + (ncy - 0.5) * kh - of)
    rng = np.random.default_rng(ncx)
    cells = rng.integers(0, ncx * ncy, len(r))
    cells[:40] = 0
    cells[40:75] = ncx * ncy - 1
    for ax, (c, lo) in enumerate(((cells // ncy, prm["x_0"]), (cells % ncy, prm["y_0"]))):
        r[:, ax] = lo - of + (c + rng.uniform(0.1, 0.9, len(r))) * kh
    for k in ("r_o", "v_o"):
        case.arrays.pop(k, None)
    print(f"[case] {ncx} x {ncy} cells, np={case.np}, scan wait {wait}", flush=True)
    O = oracle_for(case)
    oracle_init(O)
    s_o, it_o = O.cell_csr()
    with T.system_for_case(case) as ps:
        assert ps.grid() == (ncx, ncy)
        ps.set_scan_wait(wait)
        for _ in range(3):
            ps.particle_to_cell()
            s, it = ps.cell_lists()
            assert np.array_equal(s, s_o) and np.array_equal(it, it_o)
