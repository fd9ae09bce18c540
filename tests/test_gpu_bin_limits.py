"""Rects on both sides of a bin block's LDS (5 700 tiles, 512 columns) on canvases wider than they are, resolved in
the count pass, through LDS and through global atomics, and beside a scene with clip paths; the same paths
binned in one launch and in one per class; and whole-canvas rects of a destructive blend mode, past that LDS,
within the larger block's (25 000 tiles) and past both."""
import numpy as np
import pytest

import oracle
import pfh
import scenegen
from test_gpu_bin import polygons
from test_gpu_parity import check_scene
from test_gpu_resolve import rects
from test_gpu_scan import small_rects

pytestmark = pytest.mark.gpu

LDS_TILES, LDS_COLS = 5700, 512


def sides(ctx, sid, want):
    """How many of the dumped rects lie within a block's LDS and past it, at least `want` of each."""
    r = ctx.dump(sid)["path_rect"].astype(np.int64).reshape(-1, 4)
    w, h = r[:, 2] - r[:, 0], r[:, 3] - r[:, 1]
    past = (w * h > LDS_TILES) | (w > LDS_COLS)
    assert past.sum() >= want and (~past).sum() >= want


@pytest.mark.parametrize("name,sc", [
    ("tiles", rects([(2, 2, 16 * 75 - 4, 16 * 76 - 4), (2, 2, 16 * 76 - 4, 16 * 76 - 4), (18, 34, 1300, 1310), (5, 5, 700, 90)],
                    1400, 1360)),
    ("columns", rects([(2, 3, 16 * k - 4, 30) for k in (511, 512, 513, 520)], 16 * 530, 64)),
    ("windings", rects([(2, 2, 16 * 75 - 4, 16 * 76 - 4), (2, 2, 16 * 76 - 4, 16 * 76 - 4)], 1300, 1300, turns=130)),
])
def test_alone_and_beside_clips(name, sc):
    ctx = pfh.Context(0)
    alone, img = check_scene(ctx, sc, name=name)
    ids = [ctx.upload(sc), ctx.upload(scenegen.clip_scene(3, size=256, n_draw=20, n_clip=3))]
    ctx.rasterize(ids, pfh.PFH_BATCHED | pfh.PFH_NO_GRAPH | pfh.PFH_DUMP)
    sides(ctx, ids[0], 1)
    beside = ctx.dump(ids[0])
    for k in oracle.CANONICAL_KEYS + ("masks",):
        np.testing.assert_array_equal(beside[k], alone[k], err_msg=k)
    np.testing.assert_array_equal(ctx.readback(ids[0]), img)
    for flags in (pfh.PFH_PLAIN, pfh.PFH_BATCHED | pfh.PFH_NO_GRAPH, pfh.PFH_BATCHED):
        ctx.rasterize(ids[:1], flags)
        np.testing.assert_array_equal(ctx.readback(ids[0]), img)
    ctx.close()


def test_one_launch_and_two():
    sc = polygons([5] * 2 + [90] * 4, [175.0, 192.0, 590.0, 600.0, 612.0, 640.0], 1500)
    ctx = pfh.Context(0)
    _, img = check_scene(ctx, sc, name="polygons")
    ids = [ctx.upload(sc), ctx.upload(small_rects(30000))]
    ctx.rasterize(ids[:1], pfh.PFH_BATCHED | pfh.PFH_NO_GRAPH | pfh.PFH_DUMP)
    sides(ctx, ids[0], 1)
    ctx.rasterize(ids, pfh.PFH_BATCHED | pfh.PFH_NO_GRAPH)
    np.testing.assert_array_equal(ctx.readback(ids[0]), img)
    ctx.close()


@pytest.mark.parametrize("w,h", [(200, 130), (1200, 1216), (1216, 1216), (1500, 1100), (2560, 2560)])
def test_whole_canvas_blends(w, h):
    sc = scenegen.blob_scene(24, w, h, 40, r_max=min(w, h) / 2.0)
    sc.path_blend = np.full(sc.n_paths, 4, np.uint8)
    sc.path_blend[:3] = 2  # source-in: its rect is the view box (built_path.cpp:21)
    ctx = pfh.Context(0)
    _, img = check_scene(ctx, sc, name=f"{w}x{h}")
    sid, other = ctx.upload(sc), ctx.upload(small_rects(30000))
    for ids in ([sid], [sid, other]):
        for flags in (pfh.PFH_PLAIN, pfh.PFH_BATCHED | pfh.PFH_NO_GRAPH, pfh.PFH_BATCHED):
            if flags == pfh.PFH_PLAIN and len(ids) > 1:
                continue
            ctx.rasterize(ids, flags)
            np.testing.assert_array_equal(ctx.readback(sid), img)
    ctx.close()
