"""The entries' grouping by framebuffer tile where its steps end, against the oracle's draw order: one
block per scene (at most 256 tiles and 16 384 path tiles) and one past either limit, buckets of no
entries, of one chunk (2 048, or 8 192 with wide blocks) and of many, canvases of more than 65 536 tiles
(two digits below a bucket), empty scenes among others, and the same scenes in one batch."""
import numpy as np
import pytest

import oracle
import pfh
import scenegen

pytestmark = pytest.mark.gpu


def rects(w, h, boxes, reps=1):
    """Translucent rects (x0, y0, x1, y1), the list repeated."""
    b = np.tile(np.asarray(boxes, np.float64), (reps, 1))
    pts = np.stack([b[:, [0, 1]], b[:, [2, 1]], b[:, [2, 3]], b[:, [0, 3]]], 1).reshape(-1, 2)
    n = len(b)
    return scenegen.Scene(w, h, pts.astype(np.float32), np.zeros(4 * n, np.uint8), np.arange(n + 1) * 4,
                          np.ones(n, np.uint8), np.arange(n + 1), np.zeros(n, np.uint8),
                          (0x40000000 + 7919 * np.arange(n)).astype(np.uint32))


SCENES = {
    "one tile": rects(16, 16, [(1, 1, 9, 9)], 5),
    "256 tiles, 16384": rects(256, 256, [(0, 0, 256, 256)], 64),
    "256 tiles, past 16384": rects(256, 256, [(0, 0, 256, 256)], 65),
    "257 tiles": rects(257 * 16, 16, [(3, 2, 4000, 13), (0, 0, 40, 16)], 9),
    "one bucket": rects(1024, 1024, [(5, 5, 60, 11), (30, 2, 200, 12)], 1500),
    "wide, one bucket": rects(4096, 4096, [(0, 0, 4096, 4096)] * 16 + [(0, 33, 4000, 47)] * 400),
    "past 65536 tiles": rects(8192, 4112, [(0, 0, 8192, 900), (100, 3000, 8000, 4100), (8100, 4000, 8192, 4112)], 3),
    "nothing": rects(300, 200, [(900, 900, 950, 950)]),
    "blobs": scenegen.blob_scene(21, 2048, 640, 3000, r_max=300.0),
}


def order(ctx, sc, sid):
    d = ctx.dump(sid)
    canon = oracle.run_oracle(sc, 1)
    np.testing.assert_array_equal(d["entry_fbtile"], canon["entry_fbtile"])
    np.testing.assert_array_equal(d["entry_path"], canon["entry_path"])


@pytest.mark.parametrize("name", list(SCENES))
def test_draw_order(name):
    ctx = pfh.Context(0)
    sid = ctx.upload(SCENES[name])
    ctx.rasterize([sid], pfh.PFH_PLAIN | pfh.PFH_DUMP)
    order(ctx, SCENES[name], sid)
    img = ctx.readback(sid)
    ctx.rasterize([sid], pfh.PFH_PLAIN)
    np.testing.assert_array_equal(ctx.readback(sid), img)
    ctx.close()


@pytest.mark.parametrize("names", [["one tile", "nothing", "256 tiles, 16384"], list(SCENES)])
def test_draw_order_in_a_batch(names):
    ctx = pfh.Context(0)
    ids = [ctx.upload(SCENES[k]) for k in names]
    ctx.rasterize(ids, pfh.PFH_BATCHED | pfh.PFH_NO_GRAPH | pfh.PFH_DUMP)
    for k, sid in zip(names, ids):
        order(ctx, SCENES[k], sid)
    ctx.close()
