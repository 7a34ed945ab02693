"""The autotuner tries the chunks that the launch picks beside fixed ones, and keeps
them on one small box, where any fixed length leaves most of the chip idle; the
tuned pass equals the CPU oracle bit for bit.  Every tuning key returns to its
default."""
import ctypes as C

import pytest

from harness import assert_bitexact, compare_face, gpu_for, oracle_for, pair
from maestroex_amd import _abi

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


# a choice other than the default of each key, the ones that are made per launch first
KEYS = dict(edge_scal_tz=64, velpred_fused_tz=64, velpred_fused_tile=3, adjoint_xcd=1,
            edge_scal_fused=0, edge_scal_tile=0, edge_scal_per_box=1, edge_scal_xcd=0, utrans_line=0,
            utrans_chunks=1, velpred_trans_all=0, velpred_ppm_all=0, velpred_fused=0,
            velpred_fused_comp=0, velpred_fused_xcd=0, rhoh_flux_epilogue=0, xcd_remap=1,
            adjoint_state_fused=0, adjoint_face_sums=1, adjoint_trace_rolled=1, adjoint_pow2_index=0)


def kernel_times(m, f):
    """{kernel name: (least ms of a launch's average over 5 runs, launches)} of a pass"""
    out = {}
    for _ in range(5):
        m._check(m.fns["prof_enable"](m.ctx, 1), "prof_enable")
        m.advance_pass(0, f)
        for i in range(m.fns["prof_read"](m.ctx, -1, None, None, None)):
            name, ms, n = C.c_char_p(), C.c_double(), C.c_longlong()
            m.fns["prof_read"](m.ctx, i, C.byref(name), C.byref(ms), C.byref(n))
            k = name.value.decode()
            out[k] = (min(out.get(k, (1e9, 0))[0], ms.value), n.value)
    m._check(m.fns["prof_enable"](m.ctx, 0), "prof_enable")
    return out


def test_keys_return_to_their_defaults():
    _, wg = pair(dim=3, n=32, max_grid=32, ppm_type=1)
    m = gpu_for(wg)
    f = wg.pass_fields()
    start = kernel_times(m, f)
    for key in ("edge_scal_tz", "velpred_fused_tz"):
        m.set_tuning(key, KEYS[key])
    long = kernel_times(m, f)
    for key, val in KEYS.items():
        m.set_tuning(key, val)
    staged = kernel_times(m, f)
    for key in KEYS:
        m.set_tuning(key, None)
    back = kernel_times(m, f)
    print("[tuning]", start, long, staged, back, flush=True)
    launches = {k: n for k, (_, n) in start.items()}
    assert {k: n for k, (_, n) in staged.items()} != launches
    assert {k: n for k, (_, n) in back.items()} == launches
    for k in ("k_es_fused", "k_vp_fused"):  # one 64-plane chunk: some five times the time
        assert long[k][0] > 2 * start[k][0] and back[k][0] < 2 * start[k][0], k
    with pytest.raises(_abi.MxError) as e:
        m.set_tuning("no_such_key", None)
    assert e.value.code == _abi.MX_ERR_ARG
