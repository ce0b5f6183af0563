"""The spline tables over the numbers of mesh columns and rows where their kernels change: the
recurrences' groups of eight, 64 columns a workgroup, the row tables' LDS limit (168 columns:
131,072 bytes of three tables with a stride of 65 floats) and the column recurrences' (256 rows),
against the oracle bit for bit."""
import numpy as np
import pytest

import sexgpu
import sxo
from test_gpu_background_filter import _bits, _gpu_background

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nbx,nby", [(1, 1), (1, 9), (2, 2), (3, 11), (9, 3), (10, 10), (11, 18),
                                     (32, 5), (33, 2), (65, 7), (85, 3), (168, 3), (169, 2),
                                     (169, 1), (300, 4),
                                     (4, 256), (3, 257)])
@pytest.mark.parametrize("bs", [4, 7])
def test_spline_tables(nbx, nby, bs):
    W, H = nbx * bs - (bs // 2 if nbx > 1 else 0), nby * bs - (1 if nby > 1 else 0)
    rng = np.random.default_rng(nbx * 1000 + nby)
    img = (100.0 + rng.normal(0, 3, (H, W)) + np.arange(W) * 0.3).astype(np.float32)
    print("meshes %d x %d of %d" % (nbx, nby, bs), flush=True)
    o = sxo.background(img, bs=bs, fsize=3)
    g = _gpu_background(img, bs, 3)
    for k in ("back", "sigma", "dback", "dsigma"):
        assert np.array_equal(_bits(g[k]), _bits(o[k])), k
    assert np.array_equal(_bits(sexgpu.subtracted(img.shape)), _bits(o["sub"]))
