"""A readback comes after what the caller has queued on the target: a write on the default stream, or on a
stream that the default stream waits for, behind enough copies that it is still pending when the readback is called."""
import ctypes

import numpy as np
import pytest

import hip_mem
import pfh
import scenegen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("own", [True, False])
@pytest.mark.parametrize("named", [False, True])
@pytest.mark.parametrize("pad", [0, 96, 40000])
def test_pending_write_is_read(own, named, pad):
    w, h, big = 600, 400, 256 << 20
    ctx = pfh.Context(0)
    sid = ctx.upload(scenegen.blob_scene(5, w, h, 30))
    pitch = 4 * w + (0 if own else pad)
    target = hip_mem.DeviceBuffer(pitch * h)
    if not own:
        ctx.set_target(sid, target.ptr, pitch)
    ctx.rasterize([sid])
    ptr, _ = ctx.target(sid)
    a, b = hip_mem.DeviceBuffer(big), hip_mem.DeviceBuffer(big)
    hip = hip_mem._lib()
    P, N = ctypes.c_void_p, ctypes.c_size_t
    stream = P()
    if named:
        assert hip.hipStreamCreate(ctypes.byref(stream)) == 0
    for _ in range(60):  # some milliseconds
        assert hip.hipMemcpyAsync(P(a.ptr), P(b.ptr), N(big), 3, stream) == 0
    assert hip.hipMemsetAsync(P(ptr), 0x5A, N(pitch * h), stream) == 0
    assert (ctx.readback(sid) == 0x5A).all()
    assert hip.hipDeviceSynchronize() == 0
    if named:
        assert hip.hipStreamDestroy(stream) == 0
    ctx.close()
    for m in (target, a, b):
        m.free()
