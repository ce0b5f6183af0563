"""The survivors' ranks are made once per CLEAN and shared by the segmentation map and the
catalogue rows: any order of the getters, a second CLEAN with other parameters and a second
deblending of the same frame give what a fresh run of the same steps gives."""
import ctypes as C

import numpy as np
import pytest

import sexgpu

pytestmark = pytest.mark.gpu


def upto_analysis(L, img, p, mincont):
    bm, bsig = sexgpu.run_background(img, p)
    dt, at = sexgpu.thresholds(p, bsig)
    L.init_detection()
    nraw, npix = C.c_size_t(), C.c_size_t()
    L.run_detection(dt, at, p.ext_minarea, C.byref(nraw), C.byref(npix))
    return objects(L, img, p, bsig, dt, at, nraw, npix, mincont)


def objects(L, img, p, bsig, dt, at, nraw, npix, mincont):
    L.init_deblend(dt, p.deblend_nthresh, nraw, npix)
    nobj = L.parcel_out(dt, p.deblend_nthresh, min(p.ext_minarea, 3), nraw, npix, mincont)
    L.clear_deblend(p.deblend_nthresh)
    nb = (img.shape[1] - 1) // p.back_size + 1, (img.shape[0] - 1) // p.back_size + 1
    L.analyse_gpu(sexgpu.FLAG_TRUE_DOUBLE, 1, 1, sexgpu.FLAG_TRUE_FLOAT, bsig, p.gain, 0.0, at,
                  dt, p.satur_level, 0, 0, 0, p.ext_minarea, 1, 0, nb[0], nb[1], p.back_size,
                  p.back_size, img.shape[1], nobj)
    sexgpu.check()
    return nobj, (L, img, p, bsig, dt, at, nraw, npix)


def clean(L, nobj, param):
    L.run_clean(None, param, 3000, nobj)
    sexgpu.check()


def seg(L, img):
    out = np.zeros(img.shape, np.int32)
    n = L.sxg_get_segmap(out.ctypes.data)
    sexgpu.check()
    return n, out


@pytest.mark.parametrize("first", ["map", "rows", "twice"])
def test_survivors_shared(first):
    L = sexgpu.gpu()
    img = sexgpu.synth("plain1024")[:384, :448].copy()
    p = sexgpu.Params()
    nobj, args = upto_analysis(L, img, p, 0.005)
    want = {}
    for param in (1.0, 6.0):      # each after a CLEAN of its own
        clean(L, nobj, param)
        want[param] = seg(L, img) + (sexgpu.get_catalog(nobj),)
    assert want[1.0][0] != want[6.0][0], "the two parameters should keep different objects"
    for param in (1.0, 6.0, 1.0):
        clean(L, nobj, param)
        if first == "twice":
            sexgpu.get_catalog(nobj)
            seg(L, img)
        rows = sexgpu.get_catalog(nobj) if first != "map" else None
        n, m = seg(L, img)
        if rows is None:
            rows = sexgpu.get_catalog(nobj)
        assert n == want[param][0] and len(rows) == n
        assert np.array_equal(m, want[param][1])
        assert rows.tobytes() == want[param][2].tobytes()
    # a second deblending of the same frame: more objects, a new CLEAN, new ranks
    nobj2, _ = objects(*args, 0.00001)
    clean(L, nobj2, 1.0)
    rows = sexgpu.get_catalog(nobj2)
    n, m = seg(L, img)
    assert nobj2 > nobj and len(rows) == n == m.max()
    nobj3, _ = upto_analysis(L, img, p, 0.00001)
    clean(L, nobj3, 1.0)
    n3, m3 = seg(L, img)
    assert nobj3 == nobj2 and n3 == n and np.array_equal(m, m3)
    assert sexgpu.get_catalog(nobj3).tobytes() == rows.tobytes()
    L.clear_detection()
