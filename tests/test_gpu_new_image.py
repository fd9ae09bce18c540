"""A scene's own image starts transparent, also in memory that a released scene's image or outlines lay in: read
back at once, and blended over by a first pass that loads its target, in every mode."""
import ctypes

import numpy as np
import pytest

import hip_mem
import pfh
import scenegen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h", [(1, 1), (17, 33), (500, 300), (1024, 1024)])
def test_first_pass_over_a_new_image(w, h):
    r = max(4.0, min(w, h) / 3.0)
    old = scenegen.blob_scene(70, w, h, 60, r_max=r, alpha_min=1.0)
    new = scenegen.blob_scene(71, w, h, 5, r_max=r, alpha_min=0.3)
    ctx = pfh.Context(0)
    sid = ctx.upload(new)
    ctx.rasterize([sid])
    want = ctx.readback(sid)
    load = pfh.PFH_LOAD_DST
    for draw in ("read", "lend", lambda i: ctx.rasterize([i], pfh.PFH_PLAIN | load),
                 lambda i: ctx.rasterize([i], pfh.PFH_BATCHED | pfh.PFH_NO_GRAPH | load),
                 lambda i: ctx.rasterize_noalloc([i], load)):
        ids = [ctx.upload(old) for _ in range(3)]
        ctx.rasterize(ids)
        assert ctx.readback(ids[0]).any()
        for i in ids:
            ctx.release(i)
        sid = ctx.upload(new)
        if draw == "read":
            assert not ctx.readback(sid).any()
        elif draw == "lend":
            got = np.full(4 * w * h, 0xA5, np.uint8)
            assert hip_mem._lib().hipMemcpy(ctypes.c_void_p(got.ctypes.data), ctypes.c_void_p(ctx.target(sid)[0]), ctypes.c_size_t(got.size), 2) == 0
            assert not got.any()
        else:
            draw(sid)
            np.testing.assert_array_equal(ctx.readback(sid), want)
        if draw != "lend":  # once drawn, it is left alone
            ctx.rasterize([sid])
            ptr, _ = ctx.target(sid)
            assert ptr
            np.testing.assert_array_equal(ctx.readback(sid), want)
        ctx.release(sid)
    ctx.close()
