"""The compactions of the detection beyond 4,096 workgroups, where their offsets are scanned in
a launch of their own: a frame of more than 67.1 million pixels (the window masks) with more
than 16.8 million above the threshold (the pixel lists), in bars with one maximum each, of which
every other one is too short to be kept.  The counts, the objects and the map are known in closed
form.  Eagerly, and as a planned run with the counts on the device."""
import numpy as np
import pytest

import sexgpu

pytestmark = pytest.mark.gpu

W, H, LONG, SHORT = 16448, 4098, 61, 4


def bars():
    """The frame, its number of pixels above the threshold, and the map of its objects (-1:
    none).  Every third row has bars of 61 and 4 pixels in turn, rising to their ends."""
    img = np.zeros((H, W), np.float32)
    alloc = np.full((H, W), -1, np.int32)
    above = n = 0
    for shift in range(5):
        row, own = np.zeros(W, np.float32), np.full(W, -1, np.int32)
        x, k = shift, 0
        while x + LONG + 1 + SHORT <= W:
            row[x:x + LONG] = 100.0 + np.arange(LONG)
            own[x:x + LONG] = k
            x, k = x + LONG + 1, k + 1
            row[x:x + SHORT] = 100.0 + np.arange(SHORT)
            x += SHORT + 1
        rows = np.arange(3 * shift, H, 15)
        img[rows] = row
        alloc[rows] = own
        above += rows.size * int((row > 0).sum())
        n = k
    fg = np.arange(0, H, 3)
    alloc[fg] += np.where(alloc[fg] >= 0, (np.arange(fg.size, dtype=np.int32) * n)[:, None], 0)
    return img, above, alloc, fg.size * n


def test_compactions_of_the_largest_frames():
    img, above, alloc, nobj = bars()
    assert img.size > 4096 * 256 * 64 and above > 4096 * 4096
    kw = dict(back_size=64, back_type=2, back_value=0.0, thresh_type=1, detect_thresh=50.0,
              analysis_thresh=50.0, deblend_nthresh=4, clean=0)
    p = sexgpu.Params(**kw)
    print("%d pixels, %d above the threshold, %d objects" % (img.size, above, nobj), flush=True)
    g = sexgpu.run_frame(img, p, outputs=("columns", "alloc"))
    assert (g["npix_above"], g["nraw"], g["nobj"]) == (above, nobj, nobj)
    assert g["npix_raw"] == nobj * LONG
    assert np.array_equal(g["alloc"], alloc)
    first = np.flatnonzero((alloc >= 0) & (np.roll(alloc, 1, 1) != alloc))
    assert np.array_equal(g["firstpix"], first)
    assert (g["fdnpix"] == LONG).all()
    del g
    print("planned", flush=True)
    sexgpu.set_batch_frames([img])
    try:
        for _ in range(2):
            infos, _, segs, rerun = sexgpu.process_batch_graph(1, [img.shape], p, nworkers=1)
            fi = infos[0]
            assert rerun == 0
            assert (fi.npix_above, fi.npix_raw, fi.nraw) == (above, nobj * LONG, nobj)
            assert np.array_equal(segs[0], alloc + 1)
    finally:
        sexgpu.set_batch_frames([])
