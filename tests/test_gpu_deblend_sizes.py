"""The component trees at the edges of their size classes: frames that are one raw object as
a whole (a textured field above an absolute threshold), with the number of pixels at and
just beyond the largest of each class (512, 1024, 6144 pixels in LDS; 29,696 with the parent
words in LDS; beyond, and beyond 65,535, by the whole chip), against the oracle's trees.
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


KW = dict(back_size=64, back_type=2, back_value=0.0, thresh_type=1, detect_thresh=16.0,
          analysis_thresh=16.0, deblend_mincont=0.0005)


def blends(shape, boxes, coarse, holes=0.0):
    """Textured fields (y, x, height, width), each an object of its own; holes: share of their
    pixels below the threshold."""
    img = np.zeros(shape, np.float32)
    for y, x, h, w in boxes:
        f = field(h, w, coarse)
        f[np.random.default_rng(h + w).random((h, w)) < holes] = 1.0
        img[y:y + h, x:x + w] = f
    return img


# 29,925, 90,300, 59,800, 29,583 and 600 pixels: three that the whole chip builds beside others
BOXES = [(3, 5, 171, 175), (4, 300, 300, 301), (320, 2, 230, 260), (330, 300, 171, 173),
         (560, 310, 20, 30), (600, 0, 64, 64)]


@pytest.mark.parametrize("coarse", [False, True])
@pytest.mark.parametrize("holes", [0.0, 0.15])
def test_several_large_objects(coarse, holes):
    """Objects of more than 29,696 pixels next to each other and to smaller ones in the pixel
    list, at any offset; with holes also lists with gaps inside their rows, and fragments."""
    img = blends((700, 640), BOXES, coarse, holes)
    print("large objects, coarse %d, holes %g" % (coarse, holes), flush=True)
    o = sxo.run(img, **KW)
    assert (np.asarray(o["raw_count"]) > 29696).sum() == (3 if not holes else 2)
    for _ in range(2):
        compare(sexgpu.run_frame(img, sexgpu.Params(**KW)), o)


@pytest.mark.parametrize("kw", [dict(ext_minarea=1), dict(deblend_nthresh=64),
                                dict(deblend_mincont=0.0)])
def test_large_objects_parameter_variants(kw):
    """One-pixel nodes, 64 levels, every node significant."""
    kw = dict(KW, **kw)
    img = blends((260, 330), [(2, 1, 182, 173), (190, 0, 60, 330)], False, 0.05)
    print("large object, %s" % kw, flush=True)
    o = sxo.run(img, **kw)
    assert np.asarray(o["raw_count"]).max() > 29696
    compare(sexgpu.run_frame(img, sexgpu.Params(**kw)), o)


def test_large_objects_in_a_graph():
    """Planned runs: a graph whose calibration had such objects, and one whose had none and
    whose frame then gets one (it runs again eagerly)."""
    plain = blends((700, 640), BOXES[3:], False)
    large = blends((700, 640), BOXES, False, 0.15)
    p = sexgpu.Params(**KW)
    L = sexgpu.gpu()

    def check(frames, reruns):
        infos, _, segs, rerun = sexgpu.process_batch_graph(len(frames), [f.shape for f in frames],
                                                           p, nworkers=2)
        assert rerun == reruns
        for f, fi, seg in zip(frames, infos, segs):
            o = sxo.run(f, **KW)
            assert (fi.nraw, fi.nobj, fi.nsurv) == (o["nraw"], o["nobj"], o["nsurv"])
            assert np.array_equal(seg, o["seg"])

    frames = [plain, large]
    sexgpu.set_batch_frames(frames)
    for k in range(3):
        print("graph with large objects, replay %d" % k, flush=True)
        check(frames, 0)
    assert L.sxg_batch_update_frame(0, large.ctypes.data) == 0
    print("a frame that gets large objects", flush=True)
    check([large, large], 1)
    check([large, large], 0)
