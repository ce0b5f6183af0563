"""The mesh statistics' sequential double sums, found run by run in parallel, against the
oracle's loops: bit for bit.  A wrong last bit of a sum shows in the maps where the sigma is
a small difference of large numbers (a pedestal of 1e6 with a noise of a few float ulps:
sigma^2 is then of the size of the sum's own rounding), and there ties are frequent.  Mesh
sizes on either side of every kernel's range, of the 64 pixels of a run that the walk takes at a
time, and of the parts that a mesh beyond the LDS is taken in, with truncated meshes at the edges, aligned rows and not."""
import numpy as np
import pytest

import sexgpu
import sxo

pytestmark = pytest.mark.gpu


def frame(kind, h, w):
    rng = np.random.default_rng(3)
    z = rng.normal(size=(h, w))
    if kind == "sky":
        a = 1000 + 10 * z
    elif kind == "pedestal":
        a = 1e6 + 0.2 * z
    elif kind == "negative":
        a = -1e6 + 0.2 * z
    elif kind == "subtracted":          # partial sums around zero: no binade lasts
        a = 10 * z
        a[::17, ::13] = 3e5
    elif kind == "zero mean":           # the same without sources: also sums of either sign
        a = 10 * z
    elif kind == "infinite":            # no run keeps a binade
        a = 10 * z
        a[h // 3, w // 3] = np.inf
    elif kind == "range":               # signs and magnitudes in any order
        a = np.sign(z) * 10.0 ** rng.uniform(-18, 18, (h, w))
    elif kind == "coarse":              # few mantissa bits: ties and exact zeros
        a = np.round(z * 4) * 2.0 ** 20 + np.round(rng.normal(size=(h, w))) * 2.0 ** -3
    elif kind == "holes":               # pixels that take no part; a mesh without any
        a = 1e6 + 0.2 * z
        a[rng.random((h, w)) < 0.3] = -2e30
        a[:70, :70] = -2e30
        a[h // 2, w // 2] = np.nan
    else:
        a = np.full((h, w), 7.25)
    return a.astype(np.float32)


KINDS = ["sky", "pedestal", "negative", "subtracted", "zero mean", "infinite", "range", "coarse",
         "holes", "constant"]


@pytest.mark.parametrize("h,w,bs", [(150, 204, 64), (150, 203, 64), (97, 130, 32), (41, 33, 7),
                                    (300, 292, 128), (205, 301, 91), (333, 340, 160),
                                    (210, 431, 210), (256, 300, 256), (262, 517, 260),
                                    (530, 530, 530)])
@pytest.mark.parametrize("kind", KINDS)
def test_mesh_statistics_match_the_sequential_loops(kind, h, w, bs):
    img = frame(kind, h, w)
    print("mesh statistics: %s %dx%d mesh %d" % (kind, w, h, bs), flush=True)
    o = sxo.background(img, bs=bs, fsize=1)
    bm, bsig = sexgpu.run_background(img, sexgpu.Params(back_size=bs, back_fsize=1))
    back, sigma, _, _ = sexgpu.back_maps((w - 1) // bs + 1, (h - 1) // bs + 1)
    assert np.array_equal(back.view(np.int32), o["back"].view(np.int32))
    assert np.array_equal(sigma.view(np.int32), o["sigma"].view(np.int32))
    assert (bm, bsig) == (o["backmean"], o["backsig"])


@pytest.mark.parametrize("h,w,bs", [(3, 40001, 40001), (4, 33280, 33280), (5, 40001, 20003),
                                    (2, 16385, 16385), (4, 16384, 16384)])
@pytest.mark.parametrize("kind", ["sky", "zero mean", "coarse"])
def test_mesh_rows_longer_than_the_part_in_lds(kind, h, w, bs):
    """Meshes beyond the LDS go through it 16,384 pixels at a time: rows as long, and longer."""
    img = frame(kind, h, w)
    print("mesh statistics: %s %dx%d mesh %d" % (kind, w, h, bs), flush=True)
    o = sxo.background(img, bs=bs, fsize=1)
    L = sexgpu.gpu()
    L.init_device(w, h, img.ctypes.data)
    bm, bsig = sexgpu.C.c_float(), sexgpu.C.c_float()
    L.back_estimate(bs, 0.0, sexgpu.C.byref(bm), sexgpu.C.byref(bsig), 1, 1, 0)
    sexgpu.check()
    back, sigma, _, _ = sexgpu.back_maps((w - 1) // bs + 1, 1)
    assert np.array_equal(back.view(np.int32), o["back"].view(np.int32))
    assert np.array_equal(sigma.view(np.int32), o["sigma"].view(np.int32))
    assert (bm.value, bsig.value) == (o["backmean"], o["backsig"])
