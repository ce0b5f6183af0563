"""The compactions and the sort of the detection at the edges of their launch shapes: frames
with an exact number of foreground pixels, in bars of which every third is too short to be kept,
around one and several workgroups of 1024, the 2^16 pixels up to which the sort takes small
tiles and the 2^18 up to which the compaction does, against the oracle."""
import numpy as np
import pytest

import sexgpu
import sxo
from test_gpu_pipeline import compare

pytestmark = pytest.mark.gpu


def bars(n, w):
    """Exactly n pixels above the threshold: bars of 7, 8 and 3 pixels, a free pixel between
    them, every other row free."""
    rows = []
    left = n
    rng = np.random.default_rng(n)
    while left > 0:
        row = np.zeros(w, np.float32)
        x = len(rows) % 5
        for k in range(w):
            m = min((7, 8, 3)[k % 3], left, w - x)
            if m <= 0:
                break
            row[x:x + m] = 100.0 + rng.integers(0, 64, m)
            x += m + 1
            left -= m
        rows += [row, np.zeros(w, np.float32)]
    while len(rows) < 64:
        rows.append(np.zeros(w, np.float32))
    return np.array(rows)


@pytest.mark.parametrize("n,w", [(8, 64), (255, 65), (1023, 96), (1024, 130), (1025, 130),
                                 (4097, 256), (65535, 515), (65537, 515), (98303, 700),
                                 (262143, 1024), (262145, 1024)])
def test_exact_foreground(n, w):
    img = bars(n, w)
    kw = dict(back_size=64, back_type=2, back_value=0.0, thresh_type=1, detect_thresh=50.0,
              analysis_thresh=50.0, deblend_nthresh=4, clean=0)
    print("foreground %d in %s" % (n, img.shape), flush=True)
    g = sexgpu.run_frame(img, sexgpu.Params(**kw))
    assert g["npix_above"] == n
    compare(g, sxo.run(img, **kw))
    assert 0 < g["nraw"] and g["npix_raw"] < n
