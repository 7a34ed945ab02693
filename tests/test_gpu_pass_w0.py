"""GPU parity of the pass's face velocities (and etarhoflux) where Addw0 is part of
their stores (transverse directions periodic; spherical: umac) and where it is a
pass of its own (walls): whole FABs with their ghosts, from fields that hold other
values, two passes in a row, against the CPU oracle, bit for bit."""
import numpy as np
import pytest

from harness import assert_bitexact, compare_face, compare_mf, gpu_for, oracle_for, pair
from test_gpu_edge_upwind import BOXES, IN, NOSLIP, OUT, SLIP, SYM

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tune", [{}, {"velpred_fused": 0}, {"velpred_fused_comp": 0}],
                         ids=["default", "staged", "all_components"])
@pytest.mark.parametrize("cfg", [
    dict(), dict(phys_bc={2: (SLIP, IN)}), dict(phys_bc={2: (SYM, NOSLIP)}),
    dict(phys_bc={0: (OUT, OUT)}), dict(phys_bc={0: (IN, SLIP), 1: (NOSLIP, SYM), 2: (OUT, IN)}),
    dict(spherical=True), dict(ppm_type=2), dict(use_exact_base_state=1),
    dict(dim=2, boxes=[((0, 0, 0), (16, 33, 0)), ((17, 0, 0), (33, 33, 0))]),
    dict(dim=2, phys_bc={1: (SLIP, OUT)}),
], ids=["outflow_z", "slip_inflow_z", "symmetry_z", "open_x", "all", "spherical", "ppm2", "exact_base",
        "2d", "2d_slip"])
def test_pass_face_velocities(cfg, tune):
    cfg = dict(dict(dim=3, n=34, ppm_type=1), **cfg)
    if cfg["dim"] == 3:
        cfg["boxes"] = BOXES
    wc, wg = pair(**cfg)
    rng = np.random.default_rng(3)
    for mc, mg in [(wc.etarhoflux, wg.etarhoflux)] + [
            (f, g) for fc, fg in ((wc.utrans, wg.utrans), (wc.umac, wg.umac))
            for f, g in zip(fc, fg)]:
        for b, x in enumerate(mc.to_numpy()):
            v = rng.standard_normal(x.shape)
            mc.arrays[b] = v
            mg.arrays[b] = wg.backend.from_numpy(v)
    mc, mg = oracle_for(wc), gpu_for(wg)
    for k, v in tune.items():
        mg.set_tuning(k, v)
    for rep in range(2):
        for w, m in ((wc, mc), (wg, mg)):
            m.advance_pass(0, w.pass_fields())
            m.sync()
        assert_bitexact(compare_face(wc.utrans, wg.utrans, region="all"), f"utrans, pass {rep}")
        assert_bitexact(compare_face(wc.umac, wg.umac, region="all"), f"umac, pass {rep}")
        assert_bitexact(compare_mf(wc.etarhoflux, wg.etarhoflux, region="all"), f"eta, pass {rep}")
