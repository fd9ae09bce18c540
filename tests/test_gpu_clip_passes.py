"""Passes of scenes with clip paths that differ in nothing but what came before them: a new context's first
stage-by-stage pass, in memory that held ones, against the FP64 composite of the oracle."""
import numpy as np
import pytest

import hip_mem
import oracle
import pfh
import scenegen

pytestmark = pytest.mark.gpu


def leave_ones():
    """Freed device memory full of ones, blocks of every size that a small context takes; between blocks that
    are returned, to be freed later, so that the runtime keeps the memory for what is allocated next."""
    bufs = [hip_mem.DeviceBuffer(256 << k) for k in range(17) for _ in range(16)]
    for b in bufs:
        b.fill(0xFF)
    for b in bufs[::2]:
        b.free()
    return bufs[1::2]


@pytest.mark.parametrize("seed", range(3))
def test_first_plain_pass_in_used_memory(seed):
    """The set of clip mask rows already listed grows with the mask rows, after the pass has begun: it has to
    start empty there, or rows that solid tiles sample are never computed."""
    sc = scenegen.clip_scene(60 + seed, size=900, n_draw=150, n_clip=12)
    want = np.rint(np.clip(oracle.full_model(sc, zmode=1)["image"], 0.0, 1.0) * 255.0).astype(np.int64)
    for _ in range(2):
        kept = leave_ones()
        ctx = pfh.Context(0)
        sid = ctx.upload(sc)
        for p in range(2):
            ctx.rasterize([sid], pfh.PFH_PLAIN)
            off = np.abs(ctx.readback(sid).astype(np.int64) - want)
            assert off.max() <= 1, f"pass {p}: {int((off > 1).sum())} bytes off, by up to {int(off.max())}"
        ctx.close()
        for b in kept:
            b.free()


def test_every_pass_draws_the_same_bytes():
    """A tile's fills come in any order; where a clipped path's mask meets its clip's, the coverage is a sum
    over them and has to be the same one in every pass.  This scene has a pixel next to half a byte step."""
    sc = scenegen.stress_scene(scenegen.BASE_SEED ^ (32 * 7919 + 13), 1278, 948, 237, 94)
    ctx = pfh.Context(0)
    sid = ctx.upload(sc)
    ctx.rasterize([sid], pfh.PFH_PLAIN)
    first = ctx.readback(sid)
    for p in range(23):
        ctx.rasterize([sid], pfh.PFH_PLAIN if p % 2 else pfh.PFH_BATCHED | pfh.PFH_NO_GRAPH)
        np.testing.assert_array_equal(ctx.readback(sid), first, err_msg=f"pass {p}")
    want = np.rint(np.clip(oracle.full_model(sc, zmode=1)["image"], 0.0, 1.0) * 255.0).astype(np.int64)
    assert np.abs(first.astype(np.int64) - want).max() <= 1
    ctx.close()
