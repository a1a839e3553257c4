"""The download's ordering on the device: every field comes back in reference
order, bit for bit, whatever the cell build did to the slots.  Sizes at the
edges of the bitmap's words (32 positions), of a workgroup's share of the
bitmap scan (4 words per thread, 64 lanes) and of a round of it (131,072
positions); removed particles; a batch's cases."""
import numpy as np
import pytest

import tinysph_old_amd as T

pytestmark = pytest.mark.gpu

FIELDS = ("type", "index", "p", "rho", "drho", "r", "v", "a", "r_o", "v_o", "rho_o", "gnr", "n")


def scattered(n, seed):
    """n fluid particles scattered over a 1 x 1 m box, every field random."""
    g = np.random.RandomState(seed)
    arrays = {k: g.rand(n, 2) for k in ("r", "v", "a", "r_o", "v_o", "gnr", "n")}
    arrays.update({k: 1000.0 + g.rand(n) for k in ("p", "rho", "drho", "rho_o")})
    arrays["type"] = np.where(g.rand(n) < 0.2, T.WALL, T.FLUID).astype(np.int32)
    arrays["index"] = g.permutation(n).astype(np.int32)
    return arrays


def box(h=0.01):
    return {"h": h, "kap": 2.0, "cs": 20.0, "rho0": 1000.0, "avisc": 0.01, "delta": 0.1, "dp": h,
            "x_0": -0.1, "x_m": 1.1, "y_0": -0.1, "y_m": 1.1}


@pytest.mark.parametrize("n", [1, 31, 32, 33, 255, 8191, 8193, 131071, 131072, 131073, 300001])
def test_download_returns_reference_order(n):
    print(f"[case] {n} scattered particles", flush=True)
    arrays = scattered(n, n)
    with T.ParticleSystem(box(), capacity=n) as ps:
        ps.upload(arrays)
        ps.particle_to_cell()
        ps.particle_to_cell()
        got = ps.download(FIELDS)
        some = ps.download(("rho", "r"))  # a part of the fields, on a state already downloaded
        ps.particle_to_cell()             # the build after a download
        again = ps.download(FIELDS)
    for k in FIELDS:
        assert np.array_equal(got[k], arrays[k]), k
        assert np.array_equal(again[k], arrays[k]), k
    for k in some:
        assert np.array_equal(some[k], arrays[k]), k


def test_download_skips_removed_particles():
    n = 5000
    arrays = scattered(n, 3)
    arrays["type"][:] = T.FLUID
    # single particles out of the domain (each is erased: no two are adjacent)
    gone = np.arange(7, n, 37)
    arrays["r"][gone, 0] = 1.1 + 0.015
    print(f"[case] {n} particles, {len(gone)} of them removed", flush=True)
    with T.ParticleSystem(box(), capacity=n) as ps:
        ps.upload(arrays)
        ps.particle_to_cell()
        ps.remove_out_of_domain()
        ps.particle_to_cell()
        got = ps.download(FIELDS)
        assert ps.np == n - len(gone)
    keep = np.setdiff1d(np.arange(n), gone)
    for k in FIELDS:
        assert np.array_equal(got[k], arrays[k][keep]), k


def test_batch_counts_and_downloads_each_case():
    cases = T.build_ensemble(5, 11, 2000, 6000)
    with T.batch_for_cases(cases, T.PREC_FP64) as bs:
        bs.particle_to_cell()
        assert list(bs.np_per_case()) == [c.np for c in cases]
        for q in (4, 0, 2):
            got = bs.download_case(q, ("type", "index", "r", "v", "rho"))
            for k in got:
                assert np.array_equal(got[k], cases[q].arrays[k]), (q, k)
