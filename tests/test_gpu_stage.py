"""Copies through the pinned stage (halves of 1 MiB): images below, at and above a half and of several,
with a pitch of the target, of the caller's buffer and of both, far-apart rows; scenes uploaded and
released in turn, so that each takes blocks another gave back, draw what a new context draws; outlines
of more than a half come back from the stroker."""
import ctypes

import numpy as np
import pytest

import hip_mem
import pfh
import scenegen

pytestmark = pytest.mark.gpu


def read(ctx, sid, w, h, pitch):
    out = np.full(pitch * h, 0xA5, np.uint8)
    ctx._check(ctx.lib.pfh_readback_rgba8(ctx.h, sid, ctypes.c_void_p(out.ctypes.data), pitch), "readback")
    return out.reshape(h, pitch)


@pytest.mark.parametrize("w,h", [(1, 1), (512, 512), (513, 511), (16, 20000), (1500, 700), (1024, 1025)])
@pytest.mark.parametrize("dev_pad,host_pad", [(0, 0), (64, 0), (0, 12), (16, 4), (40000, 0)])
def test_readback_pitches(w, h, dev_pad, host_pad):
    if dev_pad > 1000 and h > 2000:
        pytest.skip("a target of 800 MB")
    sc = scenegen.blob_scene(w * 7 + h, w, h, 40, r_max=max(8.0, min(w, h) / 2.0))
    ctx = pfh.Context(0)
    pitch = 4 * w + dev_pad
    buf = hip_mem.DeviceBuffer(pitch * (h - 1) + 4 * w)  # nothing behind the last row
    buf.fill(0x5A)
    sid = ctx.upload(sc)
    ctx.set_target(sid, buf.ptr, pitch)
    ctx.rasterize([sid])
    raw = buf.download()
    rows = np.stack([raw[r * pitch:r * pitch + 4 * w] for r in range(h)])
    got = read(ctx, sid, w, h, 4 * w + host_pad)
    np.testing.assert_array_equal(got[:, :4 * w], rows)
    assert (got[:, 4 * w:] == 0xA5).all()
    ctx.close()
    buf.free()


def test_blocks_change_hands():
    scenes = [scenegen.blob_scene(k, 300 + 40 * k, 500, 30 + 200 * (k % 3)) for k in range(6)]
    scenes += [scenegen.dashed_stroke_scene(9, size=700, n=40), scenegen.blob_scene(8, 64, 64, 12000, r_max=9.0)]
    want = []
    for sc in scenes:
        c = pfh.Context(0)
        sid = c.upload(sc)
        c.rasterize([sid])
        want.append(c.readback(sid))
        c.close()
    ctx = pfh.Context(0)
    live = {}
    for step, k in enumerate(np.random.default_rng(1).integers(0, len(scenes), 60)):
        if k in live:
            ctx.release(live.pop(k))
            continue
        live[k] = ctx.upload(scenes[k])
        ids = list(live.values())
        ctx.rasterize(ids, pfh.PFH_BATCHED | (pfh.PFH_NO_GRAPH if step % 2 else 0))
        for q, sid in live.items():
            np.testing.assert_array_equal(ctx.readback(sid), want[q])
    ctx.close()


def test_long_outlines():
    import oracle

    rng = np.random.default_rng(4)
    pts = (rng.uniform(0, 4000, (60000, 2))).astype(np.float32)
    one = (pts, np.zeros(60000, np.uint8), np.array([0, 60000]), np.zeros(1, np.uint8))
    ctx = pfh.Context(0)
    got = ctx.stroke_outlines(*one, np.array([0, 1]), [(3.0, 0, 1, 4.0)])
    want = oracle.stroke(*one, 3.0, 0, 1, 4.0)
    assert got[0].nbytes > 1 << 20
    np.testing.assert_array_equal(got[0].view(np.uint32), np.asarray(want[0], np.float32).reshape(-1, 2).view(np.uint32))
    ctx.close()
