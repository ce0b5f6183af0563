"""The component trees at the edges of their size classes: frames that are one raw object as
a whole (a textured field above an absolute threshold), with the number of pixels at and
just beyond the largest of each class (512, 1024, 6144 pixels in LDS; 29,696 with the parent
words in LDS; beyond, and beyond 65,535, all in global memory), against the oracle's trees.
The values are smooth (few ties), or on a coarse grid (plateaus and ties everywhere), where
also the bounds of the significance test are most often exact."""
import numpy as np
import pytest

import sexgpu
import sxo
from test_gpu_pipeline import compare

pytestmark = pytest.mark.gpu


def field(h, w, coarse):
    rng = np.random.default_rng(h * 1000 + w)
    z = rng.normal(size=(h + 8, w + 8))
    for axis in (0, 1):
        for _ in range(3):
            z = z + np.roll(z, 1, axis) + np.roll(z, -1, axis)
    z = z[4:-4, 4:-4]
    z = 400.0 * np.exp(0.9 * (z - z.mean()) / z.std())
    z = np.round(z / 64) * 64 if coarse else z
    return np.maximum(z, 32.0).astype(np.float32)


@pytest.mark.parametrize("coarse", [False, True])
@pytest.mark.parametrize("h,w", [(16, 32), (27, 19), (32, 32), (41, 25), (64, 96), (5, 1229),
                                 (232, 128), (171, 174), (300, 291)])
def test_one_object_of_the_frame(h, w, coarse):
    img = field(h, w, coarse)
    kw = dict(back_size=min(h, w, 64), back_type=2, back_value=0.0, thresh_type=1,
              detect_thresh=16.0, analysis_thresh=16.0, deblend_mincont=0.0005)
    print("one object: %dx%d = %d pixels, coarse %d" % (w, h, w * h, coarse), flush=True)
    g = sexgpu.run_frame(img, sexgpu.Params(**kw))
    assert g["nraw"] == 1 and g["npix_raw"] == h * w
    compare(g, sxo.run(img, **kw))
    assert g["nobj"] > 1
