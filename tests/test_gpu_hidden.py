"""Canvases covered so deep that masks under their translucent layers are left out of the fill: the
pixels equal, byte for byte, those of the run with dumps, which computes every mask.  Each is drawn
after another scene, so that the masks left out hold that scene's.  Layers of few and of many bits, long
runs of whole tiles, tile counts that are no multiple of a block's, gradients, blend ops (no bound
holds: every mask is needed), deep and shallow scenes in one launch, and a loaded target."""
import numpy as np
import pytest

import pfh
import scenegen

pytestmark = pytest.mark.gpu

DEPTH = 96  # path tiles per framebuffer tile from which masks are left out


def blobs(seed, w, h, n, alphas, r_min=20.0):
    sc = scenegen.blob_scene(seed, w, h, n, r_min=r_min, r_max=90.0)
    a = np.random.default_rng(seed).choice(np.asarray(alphas, np.uint32), n)
    sc.path_rgba = (sc.path_rgba & np.uint32(0xffffff)) | (a << 24).astype(np.uint32)
    return sc


SCENES = [("one tile", blobs(1, 16, 16, 300, [200, 254], 4.0)), ("faint", blobs(2, 80, 56, 3000, [3, 8])),
          ("half", blobs(3, 72, 40, 400, [128])), ("near opaque", blobs(4, 200, 136, 900, [250, 254])),
          ("every alpha", blobs(5, 136, 264, 1200, range(256))), ("runs", blobs(6, 48, 48, 900, [0, 90, 254], 60.0)),
          ("gradients", scenegen.gradient_scene(7, 64, 3000)), ("ops", scenegen.blend_scene(8, 64, 3000))]
DECOY = scenegen.blob_scene(99, 320, 320, 3000, r_min=4.0, r_max=60.0)


@pytest.mark.parametrize("flags", [pfh.PFH_PLAIN, pfh.PFH_BATCHED | pfh.PFH_NO_GRAPH, pfh.PFH_BATCHED])
@pytest.mark.parametrize("name,sc", SCENES)
def test_left_out_masks_do_not_show(name, sc, flags):
    ctx = pfh.Context(0)
    decoy, sid = ctx.upload(DECOY), ctx.upload(sc)
    ctx.rasterize([sid], flags | pfh.PFH_DUMP)
    want = ctx.readback(sid)
    full = ctx.stats()
    for _ in range(2):
        ctx.rasterize([decoy], flags)
        ctx.rasterize([sid], flags)
        st = ctx.stats()
        assert st["tiles"] >= DEPTH * st["fb_tiles"]
        assert st["entries"] == full["entries"] and st["alpha_masked"] == st["alpha_entries"]
        np.testing.assert_array_equal(ctx.readback(sid), want)
    ctx.close()


def test_deep_and_shallow_scenes_in_one_launch():
    ctx = pfh.Context(0)
    scenes = [scenegen.blob_scene(30, 100, 60, 5)] + [sc for _, sc in SCENES] + [scenegen.blob_scene(31, 500, 300, 60)]
    decoy, ids = ctx.upload(DECOY), [ctx.upload(sc) for sc in scenes]
    ctx.rasterize(ids, pfh.PFH_BATCHED | pfh.PFH_NO_GRAPH | pfh.PFH_DUMP)
    want = [ctx.readback(i) for i in ids]
    ctx.rasterize([decoy], pfh.PFH_PLAIN)
    ctx.rasterize(ids, pfh.PFH_BATCHED | pfh.PFH_NO_GRAPH)
    for i, img in zip(ids, want):
        np.testing.assert_array_equal(ctx.readback(i), img)
    ctx.close()


def test_left_out_masks_over_a_loaded_target():
    ctx = pfh.Context(0)
    decoy, bg, sid = ctx.upload(DECOY), ctx.upload(scenegen.blob_scene(40, 136, 264, 40)), ctx.upload(SCENES[4][1])
    ctx.set_target(sid, *ctx.target(bg))
    imgs = []
    for dump in (pfh.PFH_DUMP, 0):
        ctx.rasterize([decoy], pfh.PFH_PLAIN)
        ctx.rasterize([bg], pfh.PFH_PLAIN)
        ctx.rasterize([sid], pfh.PFH_PLAIN | pfh.PFH_LOAD_DST | dump)
        imgs.append(ctx.readback(sid))
    np.testing.assert_array_equal(imgs[1], imgs[0])
    ctx.close()
