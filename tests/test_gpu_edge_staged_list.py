"""GPU parity of the pass's edge states by the staged kernels, whose components
(species, Rho, RhoH: not adjacent) go in one call where their temporaries are
small and in one call each where they are not, against the CPU oracle, bit for
bit."""
import pytest

from harness import assert_bitexact, compare_face, gpu_for, oracle_for, pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cfg", [
    dict(dim=2, n=20, max_grid=12, ppm_type=0), dict(dim=2, n=33, max_grid=16, ppm_type=1, nspec=1),
    dict(dim=2, n=33, max_grid=33, ppm_type=2, nspec=5), dict(dim=3, n=14, max_grid=8, ppm_type=0),
    dict(dim=3, n=14, max_grid=8, ppm_type=1, ppm_trace_forces=1),
    # 5 components' temporaries above the size that goes in one call
    dict(dim=2, n=1000, max_grid=512, ppm_type=1),
], ids=["2d_ppm0", "2d_ppm1", "2d_ppm2", "3d_ppm0", "3d_forces", "2d_large"])
def test_staged_edge_states(cfg):
    wc, wg = pair(**cfg)
    for w, m in ((wc, oracle_for(wc)), (wg, gpu_for(wg))):
        m.advance_pass(0, w.pass_fields())
        m.sync()
    comps = [0, 1] + list(range(4, wc.nscal))
    assert_bitexact(compare_face(wc.sedge, wg.sedge, comps=comps), "sedge")
    assert_bitexact(compare_face(wc.sflux, wg.sflux, comps=comps), "sflux")
