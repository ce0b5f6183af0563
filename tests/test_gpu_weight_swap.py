"""A weight map replaced, or removed, right after analyse_gpu and run_clean without a host
output, in a context of the caller's own: the kernels that are still queued then read the map
they were called with, so the columns are those of a run that is waited for."""
import numpy as np
import pytest

import sexgpu
from test_gpu_weights import weighted_frame

pytestmark = pytest.mark.gpu

COLUMNS = ("npix", "poserr_mx2", "poserr_my2", "flux", "fluxerr", "thresh_obj", "iso", "master")


def analysed(img, p, wt, then):
    """The path as far as run_clean(NULL), then `then`, then the columns."""
    L = sexgpu.gpu()
    H, W = img.shape
    sexgpu.set_weight(wt, p)
    _, bsig = sexgpu.run_background(img, p)
    dthresh, thresh = sexgpu.thresholds(p, bsig)
    L.init_detection()
    sexgpu.apply_filter(p.mask)
    nraw, npix = sexgpu.C.c_size_t(), sexgpu.C.c_size_t()
    L.run_detection(dthresh, thresh, p.ext_minarea, sexgpu.C.byref(nraw), sexgpu.C.byref(npix))
    L.init_deblend(dthresh, p.deblend_nthresh, nraw, npix)
    nobj = L.parcel_out(dthresh, p.deblend_nthresh, min(p.ext_minarea, 3), nraw, npix,
                        p.deblend_mincont)
    sexgpu.check()
    bw = min(p.back_size, W)
    nbx, nby = (W - 1) // bw + 1, (H - 1) // bw + 1
    L.analyse_gpu(sexgpu.FLAG_TRUE_DOUBLE, 1, 1, sexgpu.FLAG_TRUE_FLOAT, bsig, p.gain, 0.0,
                  thresh, dthresh, p.satur_level, 0, 0, 0, p.ext_minarea, p.clean, 0, nbx, nby,
                  bw, bw, W, nobj)
    L.run_clean(None, p.clean_param, p.clean_stacksize, nobj)
    then()
    sexgpu.check()
    assert nobj > 100
    return {k: sexgpu.get_column(k, nobj) for k in COLUMNS}


@pytest.mark.parametrize("removed", [False, True])
def test_next_weight_map_waits_for_queued_kernels(masks, removed):
    img, wt = weighted_frame(seed=27)
    other = None if removed else (wt * np.float32(9.0)).astype(np.float32)
    p = sexgpu.Params(mask=masks["default"])
    L = sexgpu.gpu()
    ctx = L.sxg_ctx_create()
    L.sxg_ctx_bind(ctx)
    try:
        ref = analysed(img, p, wt, L.sxg_sync)
        for k in range(5):
            print("weight map %s, pass %d" % ("removed" if removed else "replaced", k), flush=True)
            got = analysed(img, p, wt, lambda: sexgpu.set_weight(other, p))
            for c in COLUMNS:
                assert np.array_equal(got[c].view(np.uint8), ref[c].view(np.uint8)), c
    finally:
        L.sxg_ctx_bind(None)
        L.sxg_ctx_destroy(ctx)
