"""GPU parity of the pass over FABs whose rows do not follow each other at nx doubles:
rows far apart (past the fused kernels' 32-bit byte offsets: the row index is the
slowest, so that the FAB stays small) and rows that run downwards.  Against the CPU
oracle, bit for bit; the autotuner of the fused kernel refuses such levels."""
import pytest

from harness import assert_bitexact, compare_face, gpu_for, oracle_for, pair
from maestroex_amd import _abi
from maestroex_amd.fabs import _FAB

pytestmark = pytest.mark.gpu

FAR = 0x7FFFFFFF // (8 * 26) + 1


def restride(mf, far):
    """Give box 0 of mf rows FAR doubles apart, or (far False) downward rows."""
    import torch
    a = mf.arrays[0]
    nc, nz, ny, nx = a.shape
    x, y, z = mf.begin[0]
    if far:
        js, ks, ns = FAR, nx, nx * nz
        buf = torch.zeros((ny - 1) * js + nc * ns, dtype=a.dtype, device=a.device)
        v = buf.as_strided((nc, nz, ny, nx), (ns, ks, js, 1))
        v.copy_(a)
        mf.arrays[0] = v
        p = buf.data_ptr()
        mf.to_numpy = lambda: [v.cpu().numpy()]
    else:
        js, ks, ns = -nx, nx * ny, nx * ny * nz
        buf = a.flip(2).contiguous()
        p = buf.data_ptr() + 8 * nx * (ny - 1)
        mf.to_numpy = lambda: [buf.flip(2).cpu().numpy()]
    desc = _FAB.pack(p, js, ks, ns, x, y, z, x + nx, y + ny, z + nz, nc)
    mf._pack = lambda b: desc


@pytest.mark.parametrize("far", [True, False], ids=["far", "down"])
@pytest.mark.parametrize("field", ["scal", "umac", "sedge"])
@pytest.mark.parametrize("ppm", [1, 2])
def test_pass_row_strides(ppm, field, far):
    wc, wg = pair(dim=3, n=8, max_grid=8, ppm_type=ppm)
    f = getattr(wg, field)
    restride(f if field == "scal" else f[1], far)
    mg = gpu_for(wg)
    for w, m in ((wc, oracle_for(wc)), (wg, mg)):
        m.advance_pass(0, w.pass_fields())
        m.sync()
    for name in ("utrans", "umac", "sedge", "sflux"):
        comps = None if name in ("utrans", "umac") else [0, 1] + list(range(4, wc.nscal))
        assert_bitexact(compare_face(getattr(wc, name), getattr(wg, name), comps=comps), name)


@pytest.mark.parametrize("far", [True, False], ids=["far", "down"])
def test_autotune_refuses(far):
    _, wg = pair(dim=3, n=8, max_grid=8, ppm_type=1)
    restride(wg.sedge[0], far)
    m = gpu_for(wg)
    with pytest.raises(_abi.MxError) as e:
        m.autotune([wg.pass_fields()])
    assert e.value.code == _abi.MX_ERR_UNSUPPORTED
    m.sync()
