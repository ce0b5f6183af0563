"""The mesh statistics' sequential double sums, found run by run in parallel, against the
oracle's loops: bit for bit.  A wrong last bit of a sum shows in the maps where the sigma is
a small difference of large numbers (a pedestal of 1e6 with a noise of a few float ulps:
sigma^2 is then of the size of the sum's own rounding), and there ties are frequent.  Mesh
sizes on either side of every kernel's range, with truncated meshes at the edges, aligned
rows and not."""
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


KINDS = ["sky", "pedestal", "negative", "subtracted", "range", "coarse", "holes", "constant"]


@pytest.mark.parametrize("h,w,bs", [(150, 204, 64), (150, 203, 64), (97, 130, 32), (41, 33, 7),
                                    (300, 292, 128), (205, 301, 91), (333, 340, 160),
                                    (210, 431, 210)])
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
