"""The bin passes as one launch and as one per class: scenes on both sides of every class limit (rects of
about 512 and 4 600 tiles, 64 and 65 segments, blocks of 8 wave-class paths with a remainder) against
the oracle in one launch, and equal to that drawn together with enough paths for two."""
import numpy as np
import pytest

import pfh
import scenegen
from test_gpu_parity import check_scene
from test_gpu_scan import small_rects

pytestmark = pytest.mark.gpu


def polygons(sides, radii, size):
    """One closed polygon per (sides, radius), round the canvas' middle, corners on 1/512 px."""
    pts, cst = [], [0]
    for n, r in zip(sides, radii):
        a = np.arange(n) * (2 * np.pi / n)
        pts.append(np.round((size / 2 + r * np.stack([np.cos(a), np.sin(a)], 1)) * 512) / 512)
        cst.append(cst[-1] + n)
    k = len(sides)
    return scenegen.Scene(size, size, np.concatenate(pts).astype(np.float32), np.zeros(cst[-1], np.uint8),
                          np.array(cst), np.ones(k, np.uint8), np.arange(k + 1), np.arange(k) % 2,
                          np.array([0x60000000 + 0x123456 * (i + 1) for i in range(k)], np.uint32))


@pytest.mark.parametrize("sides,radii", [
    ([3], [5.0]),
    ([64, 65], [300.0, 300.0]),
    ([8] * 9, [10.0 + 20 * i for i in range(9)]),
    ([5] * 4 + [90] * 3, [175.0, 180.0, 186.0, 192.0, 530.0, 545.0, 560.0]),
])
def test_one_launch_and_two(sides, radii):
    sc = polygons(sides, radii, 1200)
    ctx = pfh.Context(0)
    _, img = check_scene(ctx, sc, name=str(sides))
    ids = [ctx.upload(sc), ctx.upload(small_rects(30000))]
    ctx.rasterize(ids, pfh.PFH_BATCHED | pfh.PFH_NO_GRAPH)
    np.testing.assert_array_equal(ctx.readback(ids[0]), img)
    ctx.close()
