"""A trace whose sigma |u| dt / dx is past the largest double: the division's
infinity, as in the CPU oracle, not NaN (MakeUtrans, VelPred and the edge states
along the flow; the transverse velocities are zero and keep it on its own faces)."""
import numpy as np
import pytest

from harness import gpu_for, mf_arrays, oracle_for, pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [0, 1, 2])
@pytest.mark.parametrize("ppm", [1, 2])
def test_overflowing_sigma(ppm, d):
    wc, wg = pair(dim=3, n=16, max_grid=16, ppm_type=ppm, all_periodic=True)
    for w in (wc, wg):
        for q in range(3):
            big = 1e308 if q == d else 0.0  # times dt = 1 still finite, over dx = 1/16 not
            w.utrans[q].arrays[0][...] = big
            w.umac[q].arrays[0][...] = big
            w.ufull.arrays[0][q] = big
    out = []
    for w, m in ((wc, oracle_for(wc)), (wg, gpu_for(wg))):
        m.set_dt(1.0, w.params.rel_eps)
        bcs_s, _ = m.bc_setup()
        m.MakeEdgeScal(0, w.scal, w.sedge, w.umac, w.scal_force, False, bcs_s, 4, 4, 2, False)
        m.VelPred(0, w.utilde, w.ufull, w.utrans, w.umac, w.w0mac, w.vel_force, w.w0_cart)
        m.MakeUtrans(0, w.utilde, w.ufull, w.utrans, w.w0mac, w.w0_cart)
        m.sync()
        out.append([mf_arrays(f[d])[0][c] for f, c in
                    ((w.sedge, [4, 5]), (w.umac, [0]), (w.utrans, [0]))])
    for name, a, b in zip(("sedge", "umac", "utrans"), *out):
        assert np.isinf(a).any(), name
        np.testing.assert_array_equal(a, b, err_msg=name)
