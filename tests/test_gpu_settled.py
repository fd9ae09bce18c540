"""Tiles the composite leaves early, once nothing below can change their bytes: deep stacks of
translucent layers, of whole tiles alone (folded runs, over several chunks of 64 entries) and with
edges, cleared and over a loaded target.  The bytes equal the rounded FP64 composite of the device's
own masks wherever that is further than 0.01 from a rounding boundary (fp32 over the ~60 layers that
matter: 60 x 3 roundings x 255 x 2^-24 < 0.003), and lie within 1 elsewhere."""
import numpy as np
import pytest

import oracle
import pfh
import scenegen

pytestmark = pytest.mark.gpu


def stack(n, alpha, size, seed):
    """n rects over the whole canvas, dark to bright, of one alpha."""
    rng = np.random.default_rng(seed)
    sq = np.array([[0, 0], [size, 0], [size, size], [0, size]], np.float32)
    rgb = rng.integers(0, 256, n) | rng.integers(0, 256, n) << 8 | (rng.integers(0, 4, n)) << 16
    return scenegen.Scene(size, size, np.tile(sq, (n, 1)), np.zeros(4 * n, np.uint8), np.arange(n + 1) * 4,
                          np.ones(n, np.uint8), np.arange(n + 1), np.zeros(n, np.uint8),
                          (rgb | alpha << 24).astype(np.uint32))


SCENES = [("stack", stack(n, a, 64, n + a)) for n, a in ((3, 128), (64, 40), (65, 40), (129, 20), (300, 254), (700, 3))]
SCENES += [("blobs", scenegen.blob_scene(40 + n, 200, 152, n, r_max=100.0, alpha_min=a))
           for n, a in ((60, 0.2), (700, 0.02), (4000, 0.6))]


@pytest.mark.parametrize("name,sc", SCENES)
@pytest.mark.parametrize("load", [False, True])
def test_settled_tiles_keep_their_bytes(name, sc, load):
    ctx = pfh.Context(0)
    sid = ctx.upload(sc)
    back = None
    if load:
        bg = ctx.upload(stack(1, 255, max(sc.width, sc.height), 9))
        ptr, pitch = ctx.target(bg)
        ctx.set_target(sid, ptr, pitch)
        ctx.rasterize([bg])
        back = ctx.readback(bg)[:sc.height, :sc.width].astype(np.float64) / 255.0
    ctx.rasterize([sid], pfh.PFH_PLAIN | pfh.PFH_DUMP | (pfh.PFH_LOAD_DST if load else 0))
    img, got = ctx.readback(sid).astype(np.int64), ctx.dump(sid)
    m = oracle.full_model(sc, zmode=1)
    cov = got["masks"].astype(np.float64).reshape(m["coverage"].shape) / 255.0
    want = oracle.composite_fp64(m["canon"], m["alpha"], cov, sc)
    if load:
        want = want + (1.0 - want[..., 3:]) * back
    want = np.clip(want, 0.0, 1.0) * 255.0
    err = np.abs(img - np.rint(want))
    assert err.max() <= 1
    clear = np.abs(want - np.floor(want) - 0.5) > 0.01
    assert not err[clear].any()
    ctx.close()
