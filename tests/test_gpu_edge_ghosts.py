"""GPU parity of the fused MakeEdgeScal with the fewest ghost cells it accepts (3
for ppm_type 1, 4 for ppm_type 2), on boxes that start within the reach of the
domain side's PPM stencils (2 and 3 planes above the low z side, and as far below
the high one), with upward and downward flow through them, against the CPU oracle,
bit for bit.  The planes read beside a box, from the kernel's indices: [lo - ng, hi +
ng] and no further."""
import numpy as np
import pytest

from harness import assert_bitexact, compare_face, gpu_for, oracle_for, pair
from maestroex_amd import _abi as P

pytestmark = pytest.mark.gpu

CUTS = [0, 2, 3, 5, 17, 18, 20]  # boxes of 2, 1, 2, 12, 1 and 2 planes


@pytest.mark.parametrize("side", [P.PHYS_INFLOW, P.PHYS_NOSLIPWALL, P.PHYS_OUTFLOW])
@pytest.mark.parametrize("ppm,ng", [(1, 3), (2, 4)])
@pytest.mark.parametrize("up", [1.0, -1.0])
def test_edge_scal_fewest_ghosts(ppm, ng, side, up):
    boxes = [((x, 0, a), (x + 9, 19, b - 1)) for x in (0, 10) for a, b in zip(CUTS, CUTS[1:])]
    wc, wg = pair(dim=3, n=20, ng=ng, boxes=boxes, ppm_type=ppm, phys_bc={2: (side, side)})
    for b, a in enumerate(wc.umac[2].arrays):
        u = up * (0.5 + 0.5 * np.random.default_rng(b).random(a.shape))
        wc.umac[2].arrays[b] = u
        wg.umac[2].arrays[b] = wg.backend.from_numpy(u)
    for w, m in ((wc, oracle_for(wc)), (wg, gpu_for(wg))):
        bcs_s, bcs_u = m.bc_setup()
        ho = (P.BCRec * len(bcs_s))(*bcs_s)
        for r in ho:  # the other boundary code with a stencil
            r.lo[2] = r.hi[2] = P.BC_HOEXTRAP
        m.MakeEdgeScal(0, w.scal, w.sedge, w.umac, w.scal_force, False, bcs_s, 4, 4, 3, False)
        m.MakeEdgeScal(0, w.scal, w.sedge, w.umac, w.scal_force, False, ho, 0, 0, 2, True)
        m.sync()
    assert_bitexact(compare_face(wc.sedge, wg.sedge, comps=[0, 1, 4, 5, 6]), "sedge")
