"""Backdrops, tile status and z-buffer from the count pass (batches without clip paths) and from the
column walk (batches with one): the oracle's tiles drawn alone, and the same dump, bit for bit, drawn
beside a scene with clip paths.  Rects one tile wide and one tile high, heights on both sides of the 8-row
groups, more columns than a wave or a block has threads, rects beyond LDS, opaque and even-odd paths, and
windings past int8."""
import numpy as np
import pytest

import oracle
import pfh
import scenegen
from test_gpu_parity import check_scene

pytestmark = pytest.mark.gpu


def rects(boxes, w, h, turns=1):
    """A path per (x, y, width, height) box, its outline traced `turns` times; opaque and not, both rules."""
    n = len(boxes)
    pts = np.concatenate([np.tile([[x, y], [x + bw, y + 0.25], [x + bw - 0.5, y + bh], [x + 0.25, y + bh - 0.5]],
                                  (turns, 1)) for x, y, bw, bh in boxes]).astype(np.float32)
    a = np.array([(0xff if i % 3 else 0x80) << 24 | 0x203040 * (i + 1) & 0xffffff for i in range(n)], np.uint32)
    return scenegen.Scene(w, h, pts, np.zeros(len(pts), np.uint8), np.arange(n + 1) * 4 * turns, np.ones(n, np.uint8),
                          np.arange(n + 1), np.arange(n) // 2 % 2, a)


SCENES = [
    ("thin", rects([(3, 2, 20, 16 * k) for k in (1, 7, 8, 9, 40, 300)], 64, 5000)),
    ("flat", rects([(1, 5, 16 * k, 20) for k in (1, 63, 64, 65, 128, 129, 600)], 9700, 48)),
    ("wave and group", rects([(7, 9, 350, 350), (5, 5, 360, 380), (2, 3, 700, 16 * 8), (0, 0, 900, 900)], 1000, 1000)),
    ("beyond lds", rects([(4, 4, 1100, 1120), (40, 9, 16 * 68, 16 * 67)], 1200, 1200)),
    ("windings", rects([(8, 8, 200, 150), (60, 20, 500, 500)], 640, 640, turns=130)),
]


@pytest.mark.parametrize("name,sc", SCENES)
def test_tiles_from_the_count_pass_and_the_column_walk(name, sc):
    ctx = pfh.Context(0)
    alone, img = check_scene(ctx, sc, name=name)
    ids = [ctx.upload(sc), ctx.upload(scenegen.clip_scene(3, size=256, n_draw=20, n_clip=3))]
    ctx.rasterize(ids, pfh.PFH_BATCHED | pfh.PFH_NO_GRAPH | pfh.PFH_DUMP)
    beside = ctx.dump(ids[0])
    for k in oracle.CANONICAL_KEYS + ("masks",):
        np.testing.assert_array_equal(beside[k], alone[k], err_msg=k)
    np.testing.assert_array_equal(ctx.readback(ids[0]), img)
    for flags in (pfh.PFH_PLAIN, pfh.PFH_BATCHED | pfh.PFH_NO_GRAPH, pfh.PFH_BATCHED):
        ctx.rasterize(ids[:1], flags)
        np.testing.assert_array_equal(ctx.readback(ids[0]), img)
    ctx.close()


@pytest.mark.parametrize("cols,rows", [(1, 1), (1, 513), (31, 9), (32, 16), (33, 17), (65, 130), (130, 3)])
def test_strips_of_clips_and_clipped_paths(cols, rows):
    """Strips of 32 columns with 16 or more threads to a column: rects, and clips nested in each other, of
    about a strip's width and its stretches' heights."""
    w, h = 16.0 * cols, 16.0 * rows
    boxes = [(1 + i, 2, w - 3 - i, h - 4) for i in range(6)] + [(3, 1, w - 4, h - 2), (2.5, 2, w * 0.75, h - 3),
                                                               (4, 3, w * 0.5, h * 0.75)]
    sc = rects(boxes, 16 * cols + 8, 16 * rows + 8)
    sc.n_clip_paths = 3
    sc.path_clip = np.array([-1, 0, 1, 2, 0, 2, -1, 0, 1], np.int32)
    ctx = pfh.Context(0)
    _, img = check_scene(ctx, sc, name=f"{cols}x{rows} tiles")
    sid = ctx.upload(sc)
    for flags in (pfh.PFH_PLAIN, pfh.PFH_BATCHED | pfh.PFH_NO_GRAPH, pfh.PFH_BATCHED):
        ctx.rasterize([sid], flags)
        np.testing.assert_array_equal(ctx.readback(sid), img)
    ctx.close()


def whole_canvas(sc, n):
    """The first n paths in a blend mode whose rect is the view box (built_path.cpp:21)."""
    sc.path_blend = np.full(sc.n_paths, 4, np.uint8)
    sc.path_blend[:n] = 5  # source-in
    return sc


@pytest.mark.parametrize("name,sc", [
    # rects on both sides of a bin block's LDS (5 700 tiles, 512 columns) and of the larger one's (25 000, 1 024)
    ("square", rects([(0, 0, 16 * 75, 16 * 76), (0, 0, 16 * 76, 16 * 76), (5, 5, 2500, 2500), (0, 0, 2560, 2560)],
                     2560, 2560)),
    ("whole", rects([(0, 0, 16 * 158, 16 * 158), (0, 0, 16 * 60, 16 * 60)], 16 * 158, 16 * 158)),
    ("wide", rects([(0, 3, 16 * k, 30) for k in (512, 513, 1024, 1025)], 16 * 1030, 48)),
    ("small whole canvas", whole_canvas(scenegen.blob_scene(21, 200, 130, 40), 3)),
    ("large whole canvas", whole_canvas(scenegen.blob_scene(22, 1500, 1100, 60), 3)),
])
def test_large_rects(name, sc):
    ctx = pfh.Context(0)
    _, img = check_scene(ctx, sc, name=name)
    sid, other = ctx.upload(sc), ctx.upload(scenegen.blob_scene(23, 1024, 1024, 20000, r_max=300.0))  # entries by 4 waves
    for ids in ([sid], [sid, other]):
        for flags in (pfh.PFH_BATCHED | pfh.PFH_NO_GRAPH, pfh.PFH_BATCHED):
            ctx.rasterize(ids, flags)
            np.testing.assert_array_equal(ctx.readback(sid), img)
    ctx.close()


@pytest.mark.parametrize("seed", range(4))
def test_first_plain_pass_with_clips(seed):
    """A new context's first stage-by-stage pass grows its buffers half way, in memory that earlier
    contexts have used: the set of mask rows already listed starts empty there too."""
    sc = scenegen.clip_scene(60 + seed, size=900, n_draw=150, n_clip=12)
    imgs = []
    for _ in range(3):
        ctx = pfh.Context(0)
        sid = ctx.upload(sc)
        for _ in range(2):
            ctx.rasterize([sid], pfh.PFH_PLAIN)
            imgs.append(ctx.readback(sid))
        ctx.rasterize([sid], pfh.PFH_BATCHED | pfh.PFH_NO_GRAPH | pfh.PFH_DUMP)
        imgs.append(ctx.readback(sid))
        ctx.close()
    for img in imgs[1:]:
        np.testing.assert_array_equal(img, imgs[0])
