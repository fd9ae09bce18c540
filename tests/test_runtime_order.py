"""The host runtime's calls in their order, on a HIP runtime that only records them (hip_recorder.cpp; no GPU):
what the host waits for before it reads memory that the device wrote, and before memory changes hands."""
import ctypes
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
NO_FENCE = 0x20000000   # hipEventDisableSystemFence
COHERENT = 0x40000000   # hipHostMallocCoherent


@pytest.fixture(scope="module")
def recorder(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("hip") / "hip_recorder.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", os.path.join(HERE, "hip_recorder.cpp"), "-o", so], check=True)
    return so


def run(recorder, scenario):
    """A scenario of this file in a process whose HIP runtime is the recorder."""
    code = f"import sys; sys.path.insert(0, {HERE!r}); import test_runtime_order as t; t.{scenario}(t.Hip({recorder!r}))"
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-4000:]


class Hip:
    """The recorder, loaded before the library so that the library's calls go to it."""

    def __init__(self, so):
        import conftest  # noqa: F401  (import paths)

        self.lib = ctypes.CDLL(so, mode=ctypes.RTLD_GLOBAL)
        self.lib.rec_log.restype = ctypes.c_char_p
        self.lib.rec_held.restype = ctypes.c_size_t
        self.lib.rec_limit.argtypes = [ctypes.c_size_t]

    def take(self):
        """The calls since the last time, as lists of words."""
        calls = [line.split() for line in self.lib.rec_log().decode().splitlines()]
        self.lib.rec_clear()
        return calls


def waits_scenario(hip):
    import pfh
    import scenegen

    ctx = pfh.Context(0)
    sid = ctx.upload(scenegen.blob_scene(1, 1024, 1024, 6000))  # several halves of the stage, both ways
    ctx.rasterize([sid])
    ctx.readback(sid)
    ctx.features(sid)
    calls = hip.take()
    flags = {c[1]: int(c[2], 16) for c in calls if c[0] == "hipEventCreate"}
    pinned = [(int(c[1], 16), int(c[2]), int(c[3], 16)) for c in calls if c[0] == "hipHostMalloc"]
    waited = {c[1] for c in calls if c[0] == "hipEventSynchronize"}
    assert len(waited) >= 2
    for e in waited:
        assert not flags[e] & NO_FENCE, "the host waits on an event after which device writes need not be visible"
    read = [c for c in calls if c[0] == "hipMemcpyAsync" and c[4] == "2"]
    assert read
    for c in read:
        p = [f for base, n, f in pinned if base <= int(c[1], 16) < base + n]
        assert p and p[0] & COHERENT, "a copy for the host goes to memory whose coherence depends on the environment"
    last = max(k for k, c in enumerate(calls) if c in read)
    assert ["hipStreamSynchronize", calls[last][5]] in calls[last + 1:]


def test_the_host_waits_for_what_it_reads(recorder):
    run(recorder, "waits_scenario")


def release_scenario(hip):
    import pfh
    import scenegen

    ctx = pfh.Context(0)
    for own_target in (False, True):
        sid = ctx.upload(scenegen.blob_scene(2, 500, 300, 20))
        if own_target:  # and back again
            ctx.set_target(sid, ctx.target(ctx.upload(scenegen.blob_scene(3, 500, 300, 20)))[0], 2000)
            ctx.set_target(sid, None, 0)
        ctx.rasterize([sid])
        image, _ = ctx.target(sid)  # a caller's kernel on a stream of its own may read it from here on
        hip.take()
        ctx.release(sid)
        calls = hip.take()
        assert ["hipDeviceSynchronize"] in calls or ["hipFree", hex(image)] in calls


def test_release_waits_for_work_on_a_lent_image(recorder):
    run(recorder, "release_scenario")


def readback_scenario(hip):
    import numpy as np
    import pfh
    import scenegen

    ctx = pfh.Context(0)
    sc = scenegen.blob_scene(4, 500, 300, 20)
    mine = np.zeros(2400 * 300, np.uint8)  # device memory of the caller's
    for lent, pitch in ((True, 2000), (False, 2000), (False, 2400)):
        sid = ctx.upload(sc)
        if lent:
            ctx.target(sid)
        else:
            ctx.set_target(sid, mine.ctypes.data, pitch)
        ctx.rasterize([sid])
        hip.take()
        ctx.readback(sid)
        calls = hip.take()
        behind = set()  # streams that have waited for the default stream
        recorded = set()
        for c in calls:
            if c[0] == "hipEventRecord" and c[2] in ("(nil)", "0x0"):
                recorded.add(c[1])
            elif c[0] == "hipStreamWaitEvent" and c[2] in recorded:
                behind.add(c[1])
            elif c[0] == "hipMemcpyAsync":
                assert c[5] in behind, "the copy may pass work on the default stream"


def test_readback_follows_the_default_stream(recorder):
    run(recorder, "readback_scenario")


def large_blocks_scenario(hip):
    import numpy as np
    import pfh
    import scenegen

    def whole_canvas(seed, w, h):  # a blend mode whose rect is the view box
        sc = scenegen.blob_scene(seed, w, h, 10)
        sc.path_blend = np.full(sc.n_paths, 2, np.uint8)  # source-in
        return sc

    a, b = pfh.Context(0), pfh.Context(0)
    ids = [(c, c.upload(whole_canvas(k, w, h))) for k, (c, w, h) in enumerate([(a, 2500, 2400), (b, 1300, 1200), (a, 1400, 1200)])]
    for c, sid in ids:
        for flags in (pfh.PFH_PLAIN, pfh.PFH_BATCHED | pfh.PFH_NO_GRAPH):
            c.rasterize([sid], flags)
    limits, launches = {}, 0
    for call in hip.take():
        if call[0] == "hipFuncSetAttribute":
            assert limits.setdefault(call[1], int(call[3])) == int(call[3]), "the limit is the process's: another thread's launch may need more"
        elif call[0] == "hipLaunchKernel" and int(call[2]) > 0:
            assert int(call[2]) <= limits[call[1]]
            launches += 1
    assert launches >= 12
    hip.lib.rec_attr_error(1)
    with pytest.raises(pfh.PfhError):
        c = pfh.Context(0)
        c.rasterize([c.upload(whole_canvas(9, 1300, 1200))])


def test_one_limit_for_large_blocks(recorder):
    run(recorder, "large_blocks_scenario")


def kept_blocks_scenario(hip):
    import numpy as np
    import pfh
    import scenegen

    MB = 1 << 20
    big, other = scenegen.blob_scene(6, 3000, 3000, 50), scenegen.blob_scene(7, 900, 900, 300)

    def kept(ctx):  # what two uploads leave with the context
        before = hip.lib.rec_held()
        for sid in [ctx.upload(big) for _ in range(2)]:
            ctx.release(sid)
        assert hip.lib.rec_held() - before >= 100 * MB

    def work(use):  # how much `use` allocates
        held = hip.lib.rec_held()
        use()
        return hip.lib.rec_held() - held

    for flags in (pfh.PFH_PLAIN, pfh.PFH_BATCHED | pfh.PFH_NO_GRAPH):
        ctx = pfh.Context(0)
        ids = [ctx.upload(other)]
        need = work(lambda: ctx.rasterize(ids, flags))
        ctx.close()
        ctx = pfh.Context(0)
        ids = [ctx.upload(other)]
        kept(ctx)
        assert MB < need < 100 * MB
        hip.lib.rec_limit(hip.lib.rec_held() + need // 2)  # enough once the kept blocks are given back
        ctx.rasterize(ids, flags)
        hip.lib.rec_limit(1 << 40)
        ctx.close()
    ctx = pfh.Context(0)  # the request loop's slots
    ids = [ctx.upload(other)]
    kept(ctx)
    ctx.server_start(slots=1, memory_budget=1 << 30, max_batch=4, flags=pfh.PFH_NO_GRAPH)
    hip.lib.rec_limit(hip.lib.rec_held() + MB)
    ctx.submit(ids[0])
    assert len(ctx.poll(wait_ms=5.0)) == 1
    ctx.server_stop()
    hip.lib.rec_limit(1 << 40)
    kept(ctx)  # the predictor's buffers
    x = np.zeros((40000, 12), np.float32)
    hip.lib.rec_limit(hip.lib.rec_held() + MB)
    ctx.mlp_eval(np.zeros(pfh.MLP_PARAMS, np.float32), x)
    hip.lib.rec_limit(1 << 40)
    ctx.close()


def test_kept_blocks_make_room(recorder):
    run(recorder, "kept_blocks_scenario")


def device_scenario(hip):
    import pfh
    import scenegen

    ctx = pfh.Context(1)

    def use(call, keeps=True):
        """`call` while another library has device 0 current."""
        hip.lib.hipSetDevice(0)
        hip.take()
        got = call()
        device = 0
        for c in hip.take():
            if c[0] == "hipSetDevice":
                device = int(c[1])
            elif c[0] in ("hipMalloc", "hipHostMalloc", "hipEventCreate", "hipLaunchKernel", "hipDeviceSynchronize") or \
                    c[0] == "hipEventRecord" and c[2] in ("(nil)", "0x0"):
                assert device == 1, f"{c[0]} goes to the caller's device, not the context's"
        assert device == 0 or not keeps, "the caller's device is another one afterwards"
        return got

    def strokes():  # the recorder's kernels leave no outlines: the stroker may refuse what it reads back
        try:
            ctx.upload(scenegen.dashed_stroke_scene(9, size=200, n=6))
        except pfh.PfhError:
            pass

    use(strokes, keeps=False)
    scene = scenegen.blob_scene(8, 500, 300, 20)
    ids = [use(lambda: ctx.upload(scene), keeps=False) for _ in range(2)]
    use(lambda: ctx.readback(ids[0]))
    use(lambda: ctx.target(ids[1]))
    use(lambda: ctx.rasterize(ids), keeps=False)
    use(lambda: ctx.readback(ids[1]))
    use(lambda: ctx.features(ids[0]))
    for i in ids:
        use(lambda: ctx.release(i))


def test_calls_go_to_the_context_s_device(recorder):
    run(recorder, "device_scenario")
