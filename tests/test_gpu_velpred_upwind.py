"""GPU parity of the fused VelPred's upwind choice: transverse faces that flow
either way, stand still or stay within rel_eps (both sides averaged) under
tracing velocities of either sign, none and rel_eps, on boxes whose edges lie at
and beside the edges of a tile and of a z chunk, against the CPU oracle, bit for
bit."""
import numpy as np
import pytest

from harness import assert_bitexact, compare_face, gpu_for, oracle_for, pair
from test_gpu_edge_upwind import BOXES, IN, NOSLIP, OUT, SLIP, SYM

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cfg", [
    dict(), dict(phys_bc={2: (SLIP, IN)}), dict(phys_bc={2: (SYM, NOSLIP)}),
    dict(phys_bc={0: (OUT, OUT), 1: (OUT, OUT)}),
    dict(phys_bc={0: (IN, SLIP), 1: (NOSLIP, SYM), 2: (OUT, IN)}), dict(spherical=True),
], ids=["outflow_z", "slip_inflow_z", "symmetry_noslip_z", "open_xy", "all", "spherical"])
@pytest.mark.parametrize("ppm,tz", [(1, 32), (1, 3), (2, 7)])
def test_velpred_still_faces(cfg, ppm, tz):
    wc, wg = pair(dim=3, n=34, boxes=BOXES, ppm_type=ppm, **cfg)
    eps = wc.params.rel_eps
    rng = np.random.default_rng(11)

    def still(shape):
        return rng.choice([-1.0, 1.0], shape) * rng.choice(
            [0.0, 0.5 * eps, eps, 0.3, 1.0], shape, p=[0.1, 0.1, 0.05, 0.35, 0.4])

    for b in range(len(BOXES)):
        for mc, mg in [(wc.ufull, wg.ufull)] + [(wc.utrans[d], wg.utrans[d]) for d in range(3)]:
            u = still(mc.arrays[b].shape)
            mc.arrays[b] = u
            mg.arrays[b] = wg.backend.from_numpy(u)
    mg = gpu_for(wg)
    mg.set_tuning("velpred_fused_tz", tz)
    for w, m in ((wc, oracle_for(wc)), (wg, mg)):
        m.VelPred(0, w.utilde, w.ufull, w.utrans, w.umac, w.w0mac, w.vel_force, w.w0_cart)
        m.sync()
    assert_bitexact(compare_face(wc.umac, wg.umac), "umac")
