"""The one-launch scan at the sizes where its tiles end (4096 items), through the paths' offsets: scenes
of that many paths, one below, one above and over more than 64 tiles (two rounds of look-back), and
the same scenes cut into a batch; the pixels of a batch equal the scene drawn alone, plain."""
import numpy as np
import pytest

import pfh
import scenegen

pytestmark = pytest.mark.gpu


def small_rects(n, size=256):
    """n small rects, every pixel column count and colour of their own."""
    rng = np.random.default_rng(n)
    p0 = rng.uniform(0, size - 8, (n, 2))
    d = rng.uniform(1, 8, (n, 2))
    pts = np.stack([p0, p0 + d * [1, 0], p0 + d, p0 + d * [0, 1]], 1).astype(np.float32)
    return scenegen.Scene(size, size, pts.reshape(-1, 2), np.zeros(4 * n, np.uint8), np.arange(n + 1) * 4,
                          np.ones(n, np.uint8), np.arange(n + 1), np.arange(n) % 2,
                          rng.integers(0, 2**32, n, dtype=np.uint64).astype(np.uint32))


@pytest.mark.parametrize("n", [1, 4095, 4096, 4097, 12289, 270000])
def test_offsets_over_tile_edges(n):
    sc = small_rects(n)
    cut = max(1, min(n - 1, 4096)) if n > 1 else 1
    parts = [sc.subset(np.arange(a, b)) for a, b in ((0, cut), (cut, n)) if b > a] if n <= 12289 else [sc]
    ctx = pfh.Context(0)
    ids = [ctx.upload(s) for s in parts]
    want = []
    for s in ids:
        ctx.rasterize([s], pfh.PFH_PLAIN | pfh.PFH_DUMP)
        d = ctx.dump(s)
        assert d["fill_off"][-1] == d["fill_seg"].shape[0] and (np.diff(d["fill_off"]) >= 0).all()
        want.append(ctx.readback(s))
    ctx.rasterize(ids, pfh.PFH_BATCHED | pfh.PFH_NO_GRAPH)
    for s, img in zip(ids, want):
        np.testing.assert_array_equal(ctx.readback(s), img)
    if n <= 4097:  # the oracle's fills per path
        import oracle

        sid = ctx.upload(sc)
        ctx.rasterize([sid], pfh.PFH_PLAIN | pfh.PFH_DUMP)
        canon = oracle.full_model(sc, zmode=1)["canon"]
        got = ctx.dump(sid)
        for k in oracle.CANONICAL_KEYS:
            np.testing.assert_array_equal(got[k], canon[k], err_msg=k)
    ctx.close()
