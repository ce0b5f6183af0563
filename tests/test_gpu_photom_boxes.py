"""The aperture photometry at the edges of its launch classes: circular AUTO apertures whose
boxes hold just under and over 512 and 2048 pixels, boxes narrower and wider than a
wavefront's and a workgroup's step, boxes cut by the frame, and more large boxes than there
are workgroups for (all objects of a crowded frame), against the oracle bit for bit."""
import pytest

import sexgpu
from test_gpu_photom import compare, run_both

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("diam", [0.5, 7.0, 21.5, 22.0, 23.0, 44.0, 45.0, 46.0, 63.0, 65.0,
                                  255.0, 257.0, 400.0, 1500.0])
def test_circular_boxes(masks, diam):
    img = sexgpu.synth("plain1024")[100:420, 300:690].copy()
    print("aperture %g" % diam, flush=True)
    g, o = run_both(img, masks["default"],
                    phot={"autoaper": (diam, diam),
                          "apert": min(diam, 300.0)})
    compare(g, o)
    assert g["nobj"] > 20


def test_more_large_boxes_than_workgroups(masks):
    img = sexgpu.synth("crowded4096", width=768, height=640, nsrc=167000 // 34, seed=77)
    g, o = run_both(img, masks["default"], phot={"autoaper": (50.0, 50.0)})
    compare(g, o)
    assert g["nobj"] > 600
