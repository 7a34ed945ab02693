"""GPU parity of the fused MakeEdgeScal's upwind choice: faces that flow
either way, stand still, or stay within rel_eps (both sides averaged), on
boxes whose edges lie at and beside the edges of a tile (16 x 11 columns) and
of a z chunk, against the CPU oracle, bit for bit."""
import numpy as np
import pytest

from harness import assert_bitexact, compare_face, gpu_for, oracle_for, pair
from maestroex_amd import _abi as P

pytestmark = pytest.mark.gpu

CUTS = ([0, 1, 17, 34], [0, 11, 23, 34], [0, 2, 34])
BOXES = [((x0, y0, z0), (x1 - 1, y1 - 1, z1 - 1))
         for z0, z1 in zip(CUTS[2], CUTS[2][1:]) for y0, y1 in zip(CUTS[1], CUTS[1][1:])
         for x0, x1 in zip(CUTS[0], CUTS[0][1:])]
OUT, SLIP, IN, SYM, NOSLIP = (P.PHYS_OUTFLOW, P.PHYS_SLIPWALL, P.PHYS_INFLOW, P.PHYS_SYMMETRY,
                              P.PHYS_NOSLIPWALL)


@pytest.mark.parametrize("bc", [{}, {2: (SLIP, IN)}, {2: (SYM, SLIP)},
                                {0: (OUT, OUT), 1: (SYM, OUT)},
                                {0: (IN, SLIP), 1: (NOSLIP, SYM), 2: (OUT, IN)}],
                         ids=["outflow_z", "slip_inflow_z", "symmetry_z", "open_xy", "all"])
@pytest.mark.parametrize("ppm,cons,is_vel,tz", [(1, 0, 0, 32), (2, 0, 0, 3), (1, 1, 0, 5),
                                                (2, 1, 0, 32), (1, 0, 1, 7)])
def test_edge_scal_still_faces(bc, ppm, cons, is_vel, tz):
    wc, wg = pair(dim=3, n=34, boxes=BOXES, ppm_type=ppm, phys_bc=bc or None)
    eps = wc.params.rel_eps
    rng = np.random.default_rng(7)
    for d in range(3):
        for b, a in enumerate(wc.umac[d].arrays):
            u = rng.choice([-1.0, 1.0], a.shape) * rng.choice(
                [0.0, 0.5 * eps, eps, 0.3, 1.0], a.shape, p=[0.1, 0.1, 0.05, 0.35, 0.4])
            wc.umac[d].arrays[b] = u
            wg.umac[d].arrays[b] = wg.backend.from_numpy(u)
    mg = gpu_for(wg)
    mg.set_tuning("edge_scal_tz", tz)
    for w, m in ((wc, oracle_for(wc)), (wg, mg)):
        bcs_s, bcs_u = m.bc_setup()
        if is_vel:
            bu = (P.BCRec * 3)(*[bcs_u[q] for q in range(3)])
            m.MakeEdgeScal(0, w.utilde, w.sedge, w.umac, w.vel_force, True, bu, 0, 0, 3, False)
        else:
            m.MakeEdgeScal(0, w.scal, w.sedge, w.umac, w.scal_force, False, bcs_s, 4, 4, 3,
                           bool(cons))
            m.MakeEdgeScal(0, w.scal, w.sedge, w.umac, w.scal_force, False, bcs_s, 0, 0, 2,
                           bool(cons))
        m.sync()
    comps = [0, 1, 2] if is_vel else [0, 1, 4, 5, 6]
    assert_bitexact(compare_face(wc.sedge, wg.sedge, comps=comps), "sedge")
