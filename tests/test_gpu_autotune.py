"""The autotuner tries the chunks that the launch picks beside fixed ones, and keeps
them on one small box, where any fixed length leaves most of the chip idle; the
tuned pass equals the CPU oracle bit for bit."""
import pytest

from harness import assert_bitexact, compare_face, gpu_for, oracle_for, pair

pytestmark = pytest.mark.gpu


def test_small_box_keeps_picked_chunks():
    wc, wg = pair(dim=3, n=32, max_grid=32, ppm_type=1)
    m = gpu_for(wg)
    cands, best = m.autotune([wg.pass_fields()])
    print("[autotune]", cands, "best", best, flush=True)
    assert {t for t, tz, _ in cands if tz == 0} == {t for t, _, _ in cands}
    assert cands[best][1] == 0  # a third of the next one's time
    mc = oracle_for(wc)
    for w, mm in ((wc, mc), (wg, m)):
        mm.advance_pass(0, w.pass_fields())
        mm.sync()
    comps = [0, 1] + list(range(4, wc.nscal))
    assert_bitexact(compare_face(wc.sedge, wg.sedge, comps=comps), "sedge")
