"""GPU parity of the pass with the chunk lengths its launches pick: one thin box
(chunks of a few planes), boxes of unequal heights, more boxes than the chip
holds blocks, against the CPU oracle, bit for bit."""
import pytest

from harness import assert_bitexact, compare_face, gpu_for, oracle_for, pair
from maestroex_amd import _abi as P

pytestmark = pytest.mark.gpu

HEIGHTS = [0, 1, 3, 10, 32, 40]  # boxes of 1, 2, 7, 22 and 8 planes


@pytest.mark.parametrize("ppm", [1, 2])
@pytest.mark.parametrize("cfg", [
    dict(n=20, max_grid=(20, 20, 20)),
    dict(n=40, boxes=[((x, 0, a), (x + 19, 39, b - 1)) for x in (0, 20)
                      for a, b in zip(HEIGHTS, HEIGHTS[1:])]),
    dict(n=48, max_grid=(8, 8, 16)),
], ids=["one_box", "heights", "many_boxes"])
def test_pass_picked_chunks(cfg, ppm):
    wc, wg = pair(dim=3, ppm_type=ppm, **cfg)
    for w, m in ((wc, oracle_for(wc)), (wg, gpu_for(wg))):
        m.advance_pass(0, w.pass_fields())
        m.sync()
    for name in ("utrans", "umac", "sedge", "sflux"):
        comps = None if name in ("utrans", "umac") else [0, 1] + list(range(4, wc.nscal))
        assert_bitexact(compare_face(getattr(wc, name), getattr(wg, name), comps=comps), name)


@pytest.mark.parametrize("ppm", [1, 2])
@pytest.mark.parametrize("bc", [{2: (P.PHYS_SLIPWALL, P.PHYS_INFLOW)},
                                {1: (P.PHYS_NOSLIPWALL, P.PHYS_OUTFLOW),
                                 2: (P.PHYS_INFLOW, P.PHYS_OUTFLOW)}], ids=["z", "yz"])
def test_pass_picked_chunks_walls(bc, ppm):
    """the kernels with the rules of such sides hold fewer blocks, of which the
    chunks are picked: boxes at a wall and boxes out of its reach"""
    wc, wg = pair(dim=3, n=40, ppm_type=ppm, phys_bc=bc, boxes=[
        ((0, y, a), (39, y + 19, b - 1)) for y in (0, 20) for a, b in zip(HEIGHTS, HEIGHTS[1:])])
    for w, m in ((wc, oracle_for(wc)), (wg, gpu_for(wg))):
        m.advance_pass(0, w.pass_fields())
        m.sync()
    for name in ("umac", "sedge", "sflux"):
        comps = None if name == "umac" else [0, 1] + list(range(4, wc.nscal))
        assert_bitexact(compare_face(getattr(wc, name), getattr(wg, name), comps=comps), name)
