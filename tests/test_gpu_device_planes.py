"""The frame's planes by device pointer, in a context of the caller's own and in the default
one: what an entry point has written is there for a copy on another stream when the entry point
returns, whether the pointer was asked for before or after it."""
import ctypes as C

import numpy as np
import pytest

import sexgpu

pytestmark = pytest.mark.gpu


def plane(ptr, shape):
    import torch
    out = torch.empty(shape, dtype=torch.float32, pin_memory=True)
    hip = sexgpu._hiprt()
    assert hip.hipMemcpy(C.c_void_p(out.data_ptr()), C.c_void_p(ptr),
                         C.c_size_t(out.numel() * 4), C.c_int(2)) == 0
    return out.numpy().view(np.int32)


@pytest.fixture(params=["own", "default"])
def context(request):
    """A context of the caller's own, and the default one."""
    L = sexgpu.gpu()
    ctx = L.sxg_ctx_create() if request.param == "own" else None
    L.sxg_ctx_bind(ctx)
    yield L
    L.sxg_ctx_bind(None)
    if ctx:
        L.sxg_ctx_destroy(ctx)
    else:
        L.sxg_release()     # the pointers are no longer out


def noise(h, w):
    rng = np.random.default_rng(5)
    return (100.0 + rng.normal(0, 3, (h, w))).astype(np.float32)


@pytest.mark.parametrize("early", [False, True])
def test_filtered_plane(masks, context, early):
    img = noise(1500, 1700)
    sexgpu.run_background(img, sexgpu.Params())
    ptr = context.sxg_device_frame(1) if early else None
    sexgpu.apply_filter(masks["mexhat_5p0_11x11"])
    if not early:
        ptr = context.sxg_device_frame(1)
    got = plane(ptr, img.shape)
    assert np.array_equal(got, sexgpu.filtered(img.shape).view(np.int32))


@pytest.mark.parametrize("weight_type", ["MAP_WEIGHT", "BACKGROUND"])
def test_subtracted_plane(context, weight_type):
    """back_estimate on planes whose pointers are out already."""
    img = noise(1500, 1700)
    p = sexgpu.Params()
    sexgpu.run_background(img, p)
    ptr = context.sxg_device_frame(0)
    try:
        sexgpu.set_weight(None, p, weight_type)
        img2 = np.ascontiguousarray(img[::-1])
        sexgpu.run_background(img2, p)
        assert context.sxg_device_frame(0) == ptr
        got = plane(ptr, img.shape)
        assert np.array_equal(got, sexgpu.subtracted(img.shape).view(np.int32))
    finally:
        sexgpu.set_weight(None, p)


def test_planes_of_a_frame_without_objects(masks, context):
    img = noise(1200, 1600)
    p = sexgpu.Params(mask=masks["default"], thresh_type=1, detect_thresh=1e6,
                      analysis_thresh=1e6)
    for flip in (1, -1):
        frame = np.ascontiguousarray(img[::flip])
        nobj, _ = sexgpu.process_resident(frame, p)
        got = [plane(context.sxg_device_frame(k), img.shape) for k in (0, 1)]
        assert nobj == 0
        sexgpu.run_background(frame, p)
        sexgpu.apply_filter(p.mask)
        assert np.array_equal(got[1], sexgpu.filtered(img.shape).view(np.int32))
        assert np.array_equal(got[0], sexgpu.subtracted(img.shape).view(np.int32))
