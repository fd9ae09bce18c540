"""The flattener where its kernels' limits lie, bit for bit against the oracle's depth-first recursion:
chunks of 8 to 64 segments with a remainder, 64 curves of one depth whose pending halves overfill
the shared stack, curves flat exactly at the depth the curves' bits reach, one past it and two,
and the allocation-free entry without room for the bits."""
import numpy as np
import pytest

import pfh
import scenegen
from test_gpu_parity import check_scene

pytestmark = pytest.mark.gpu


def curves_scene(contours, size=512):
    """One closed path per (points, flags)."""
    pts = np.concatenate([np.asarray(p, np.float32).reshape(-1, 2) for p, _ in contours])
    flg = np.concatenate([np.asarray(f, np.uint8) for _, f in contours])
    cst = np.concatenate([[0], np.cumsum([len(f) for _, f in contours])])
    n = len(contours)
    return scenegen.Scene(size, size, pts, flg, cst, np.ones(n, np.uint8), np.arange(n + 1), np.arange(n) % 2,
                          np.array([0xff204060 + 0x10203 * i for i in range(n)], np.uint32))


def cubics(n, reach, seed):
    """A chain of n cubics, every fourth a quadratic, whose control points lie `reach` px off their ends."""
    rng = np.random.default_rng(seed)
    pts, flg = [rng.uniform(100, 400, 2)], [0]
    for i in range(n):
        end = rng.uniform(100, 400, 2)
        a = rng.uniform(0, 2 * np.pi)
        off = reach * np.array([np.cos(a), np.sin(a)])
        pts += [pts[-1] + off, end] if i % 4 == 3 else [pts[-1] + off, end - off, end]
        flg += [1, 0] if i % 4 == 3 else [1, 2, 0]
    return np.array(pts, np.float32), np.array(flg, np.uint8)


def flat_lines(n, seed):
    """A path of n short lines (the filler that sets how many segments a flattener wave takes)."""
    a = np.arange(n + 1) * (2 * np.pi / (n + 1))
    p = 256 + (200 + 20 * np.sin(40 * a + seed))[:, None] * np.stack([np.cos(a), np.sin(a)], 1)
    return p.astype(np.float32), np.zeros(n + 1, np.uint8)


# segments of a wave: 8 below 32 768 segments (count; emit), 16 and 32 above, 64 from 131 072
@pytest.mark.parametrize("lines", [0, 33000, 66000, 132000])
@pytest.mark.parametrize("n", [1, 7, 8, 9, 63, 64, 65])
def test_chunks_of_deep_curves(lines, n):
    ctx = pfh.Context(0)
    contours = [cubics(n, 700.0, 900 + n)] + ([flat_lines(lines, 3)] if lines else [])
    check_scene(ctx, curves_scene(contours), flags=pfh.PFH_BATCHED | pfh.PFH_NO_GRAPH, name=f"{n} curves, {lines} lines")
    ctx.close()


@pytest.mark.parametrize("reach", [1e-3, 1.0, 300.0, 1400.0, 2800.0, 9000.0, 4e4])
def test_curve_depths_around_the_bits(reach):
    """Depths 0 to 8: the bits hold 6, deeper curves take the whole-wave walk."""
    ctx = pfh.Context(0)
    check_scene(ctx, curves_scene([cubics(12, reach, 5), cubics(3, reach / 3, 6)]), name=f"reach {reach}")
    ctx.close()


@pytest.mark.parametrize("n", [3, 5000])
def test_noalloc_without_room_for_the_bits(n):
    """Thousands of curves over a few tiles: the tile arrays cannot hold the bits."""
    rng = np.random.default_rng(n)
    pts = rng.uniform(2, 30, (3 * n + 1, 2)).astype(np.float32)
    flg = np.concatenate([[0], np.tile([1, 2, 0], n)]).astype(np.uint8)
    ctx = pfh.Context(0)
    sid = ctx.upload(curves_scene([(pts, flg)], size=64))
    ctx.rasterize([sid])
    want = ctx.readback(sid)
    ctx.rasterize_noalloc([sid])
    np.testing.assert_array_equal(ctx.readback(sid), want)
    ctx.close()
