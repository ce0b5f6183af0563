"""The frame's planes by device pointer, in a context of the caller's own: what an entry point
has written is there for a copy on another stream when the entry point returns, whether the
pointer was asked for before or after it."""
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


@pytest.mark.parametrize("early", [False, True])
def test_filtered_plane(masks, early):
    L = sexgpu.gpu()
    L.sxg_device_frame.restype = C.c_void_p
    L.sxg_device_frame.argtypes = [C.c_int]
    ctx = L.sxg_ctx_create()
    L.sxg_ctx_bind(ctx)
    try:
        rng = np.random.default_rng(5)
        img = (100.0 + rng.normal(0, 3, (1500, 1700))).astype(np.float32)
        p = sexgpu.Params()
        sexgpu.run_background(img, p)
        ptr = L.sxg_device_frame(1) if early else None
        sexgpu.apply_filter(masks["mexhat_5p0_11x11"])
        if not early:
            ptr = L.sxg_device_frame(1)
        got = plane(ptr, img.shape)
        assert np.array_equal(got, sexgpu.filtered(img.shape).view(np.int32))
    finally:
        L.sxg_ctx_bind(None)
        L.sxg_ctx_destroy(ctx)
