"""Performance cases of the rasterizer, through its public entry points (pathfinder-cpp_amd/pfh.py).

Each case is a program's steady state: scenes resident on the device (uploaded in ``prepare``,
with their targets in the program's own device memory), drawn once per pass; the ``frame`` cases
take host outlines through the whole call, as a program that builds a new scene every frame does.
Outputs are the RGBA8 framebuffers, whole.

A case's fields: ``kind`` (what is drawn), ``mode`` (plain: stage by stage; batched: one
predictor-sized pass, eager launches; noalloc: the allocation-free entry; layers: a second scene
drawn over the first's pixels; frame: upload, draw, read back, release; serve: the request loop),
the canvas ``w`` x ``h``, ``n`` paths per scene, ``scenes`` per launch and, for mixed batches, the
seed ``mix`` of the scenes' sizes.  ``deep`` selects the launch schedule the autotuner picks for
scenes that are bound by their longest curves and columns; 0 keeps the default schedule.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pathfinder-cpp_amd"))

import pfh  # noqa: E402
import scenegen  # noqa: E402

WEIGHTS = os.path.join(os.path.dirname(os.path.abspath(pfh.__file__)), "predictor_weights.npy")
# eager launches: a process that has torch loaded runs on torch's HIP runtime, whose stream capture
# refuses the event nodes of the replayed mode
BATCHED = pfh.PFH_BATCHED | pfh.PFH_PREDICT | pfh.PFH_NO_GRAPH
DEEP = {"flatten_deep": 3, "flatten_segs": 64, "column_rows": 8, "composite_block": 128}
SERVE = {"slots": 3, "memory_budget": 64 << 30, "max_batch": 16, "flags": pfh.PFH_PREDICT | pfh.PFH_NO_GRAPH}


def listed():
    return [
        # the smallest call: an icon or avatar of 64 closed cubic paths, drawn stage by stage
        dict(name="icon_plain", kind="cubic", mode="plain", w=512, h=512, n=64, scenes=1),
        # an illustration (the size of an SVG drawing) that changes every frame: host outlines in, host pixels out
        dict(name="frame_900", kind="blob", mode="frame", w=900, h=900, n=304, scenes=1),
        # a document page drawn by a host that may not allocate while it draws
        dict(name="page_noalloc", kind="blob", mode="noalloc", w=1240, h=1754, n=1500, scenes=1),
        # an HD canvas of two layers, the upper drawn over the lower's pixels
        dict(name="layers_hd", kind="blob", mode="layers", w=1920, h=1080, n=700, scenes=2),
        # gradients and blend modes on a mid-size canvas
        dict(name="paint_2k", kind="paint", mode="batched", w=2048, h=2048, n=400, scenes=1),
        # the large single scene: a map of 10 000 paths, default launch schedule
        dict(name="map_4k", kind="blob", mode="batched", w=4096, h=4096, n=10000, scenes=1),
        # heavy overlap, strokes and nested clip paths, with its tuned schedule
        dict(name="stress_4k", kind="stress", mode="batched", w=4096, h=4096, n=2500, scenes=1, deep=3),
        # thumbnails or glyph-sized drawings, many per launch
        dict(name="thumbs_256", kind="blob", mode="batched", w=96, h=96, n=30, scenes=256, mix=5),
        # a render farm's launch: scenes of every size and density in one pass
        dict(name="batch_48", kind="mixed", mode="batched", w=4096, h=4096, n=20000, scenes=48, mix=7),
        # requests for resident mid-size scenes through the request loop, until all are drawn
        dict(name="serve_48", kind="mixed", mode="serve", w=1024, h=1024, n=2000, scenes=48, mix=3),
        # line art that changes every frame: open polylines stroked on the device at upload, half of them dashed
        dict(name="sketch_2k", kind="stroke", mode="frame", w=2048, h=2048, n=400, scenes=1),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the listed ones' families, sizes log-uniform over the range each stands for."""
    kind = rng.choice(["icon", "frame", "noalloc", "layers", "paint", "map", "stress", "thumbs", "batch", "serve",
                       "sketch"])
    mix = rng.randrange(1 << 20)
    if kind == "icon":
        return dict(kind=rng.choice(["cubic", "blob"]), mode=rng.choice(["plain", "batched"]), w=(s := _log(rng, 32, 700)),
                    h=s, n=_log(rng, 4, 96), scenes=1)
    if kind == "frame":
        return dict(kind="blob", mode="frame", w=_log(rng, 200, 2000), h=_log(rng, 200, 2000), n=_log(rng, 20, 2000),
                    scenes=1)
    if kind == "noalloc":
        return dict(kind="blob", mode="noalloc", w=_log(rng, 300, 1400), h=_log(rng, 300, 1754), n=_log(rng, 50, 1500),
                    scenes=1)
    if kind == "layers":
        return dict(kind="blob", mode="layers", w=_log(rng, 640, 3840), h=_log(rng, 360, 2160), n=_log(rng, 50, 3000),
                    scenes=2)
    if kind == "paint":
        s = _log(rng, 256, 2048)
        return dict(kind="paint", mode=rng.choice(["plain", "batched"]), w=s, h=s, n=_log(rng, 20, 500), scenes=1)
    if kind == "map":
        return dict(kind="blob", mode=rng.choice(["plain", "batched"]), w=_log(rng, 1024, 4096), h=_log(rng, 1024, 4096),
                    n=_log(rng, 500, 20000), scenes=1, deep=rng.choice([0, 0, 3]))
    if kind == "stress":
        s = _log(rng, 1024, 4096)
        return dict(kind="stress", mode=rng.choice(["plain", "batched"]), w=s, h=s, n=_log(rng, 250, 2500), scenes=1,
                    deep=rng.choice([0, 3]))
    if kind == "thumbs":
        s = _log(rng, 24, 200)
        return dict(kind="blob", mode="batched", w=s, h=s, n=_log(rng, 5, 60), scenes=rng.randint(32, 256), mix=mix)
    if kind == "batch":
        return dict(kind="mixed", mode="batched", w=(s := _log(rng, 512, 4096)), h=s, n=_log(rng, 200, 20000),
                    scenes=rng.randint(4, 24), mix=mix)
    if kind == "serve":
        s = _log(rng, 400, 1024)
        return dict(kind="mixed", mode="serve", w=s, h=s, n=_log(rng, 100, 2000), scenes=rng.randint(8, 48), mix=mix)
    s = _log(rng, 300, 2048)
    return dict(kind="stroke", mode="frame", w=s, h=s, n=_log(rng, 10, 500), scenes=1)


def _sizes(case):
    """(width, height, paths) of every scene of a case: the case's own, or for mixed batches square
    canvases and path counts log-uniform up to them."""
    if "mix" not in case:
        return [(case["w"], case["h"], case["n"])] * case["scenes"]
    rng = np.random.Generator(np.random.PCG64(case["mix"]))
    out = []
    for _ in range(case["scenes"]):
        if case["kind"] == "mixed":
            s = int(round(math.exp(rng.uniform(math.log(case["w"] / 16), math.log(case["w"])))))
            n = int(round(math.exp(rng.uniform(math.log(10), math.log(case["n"])))))
        else:
            s = int(rng.integers(case["w"] * 2 // 3, case["w"] * 4 // 3 + 1))
            n = int(rng.integers(case["n"] // 2, case["n"] * 3 // 2 + 1))
        out.append((s, s, max(n, 1)))
    return out


def _scene(case, seed, w, h, n):
    if case["kind"] == "cubic":
        return scenegen.cubic_scene(seed, w, n)
    if case["kind"] == "paint":
        return scenegen.blend_scene(seed, w, n)
    if case["kind"] == "stroke":
        return scenegen.dashed_stroke_scene(seed, w, n)
    if case["kind"] == "stress":
        return scenegen.stress_scene(seed, w, n * 4 // 5, n // 5, max(4, n * 2 // 25))
    return scenegen.blob_scene(seed, w, h, n, r_max=max(8.0, min(512.0, min(w, h) / 2.0)))


def prepare(case, seed):
    seed = scenegen.BASE_SEED ^ (seed * 7919 + 13)
    st = {"mode": case["mode"], "ctx": pfh.Context(0)}
    ctx = st["ctx"]
    ctx.set_predictor(np.load(WEIGHTS))
    if case.get("deep"):
        ctx.set_schedule(**DEEP)
    sizes = _sizes(case)
    scenes = [_scene(case, seed + 1000003 * k, w, h, n) for k, (w, h, n) in enumerate(sizes)]
    if case["mode"] == "frame":
        st["scene"] = scenes[0]
        return st
    st["ids"] = [ctx.upload(sc) for sc in scenes]
    # the program's own framebuffers: one allocation, an image per scene (layers share one)
    offs, total = [], 0
    for w, h, _ in sizes:
        offs.append(total)
        if case["mode"] != "layers":
            total += (4 * w * h + 255) // 256 * 256
    total = total or 4 * case["w"] * case["h"]
    st["out"] = torch.zeros(total, dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    for sid, off, (w, _, _) in zip(st["ids"], offs, sizes):
        ctx.set_target(sid, st["out"].data_ptr() + off, 4 * w)
    if case["mode"] == "serve":
        ctx.server_start(**SERVE)
    return st


def run(st):
    ctx, mode = st["ctx"], st["mode"]
    if mode == "frame":
        sid = ctx.upload(st["scene"])
        ctx.rasterize([sid], BATCHED)
        img = ctx.readback(sid)
        ctx.release(sid)
        return img
    if mode == "plain":
        ctx.rasterize(st["ids"], pfh.PFH_PLAIN)
    elif mode == "noalloc":
        ctx.rasterize_noalloc(st["ids"])
    elif mode == "layers":
        ctx.rasterize(st["ids"][:1], BATCHED)
        ctx.rasterize(st["ids"][1:], BATCHED | pfh.PFH_LOAD_DST)
    elif mode == "serve":
        for sid in st["ids"]:
            ctx.submit(sid)
        left = len(st["ids"])
        while left:
            left -= len(ctx.poll(wait_ms=5.0))
    else:
        ctx.rasterize(st["ids"], BATCHED)
    return st["out"]


def work(case):
    """Bytes of the outlines read once (points, flags, colours) and of the pixels written once.  No
    figure for operations: what a path costs depends on the tiles it crosses."""
    per = {"cubic": 25, "blob": 70, "mixed": 70, "paint": 70, "stress": 1000, "stroke": 31}[case["kind"]]
    sizes = _sizes(case)
    points = sum(n * per for _, _, n in sizes)
    images = sizes[:1] if case["mode"] == "layers" else sizes
    return {"bytes": 9 * points + sum(8 * n for _, _, n in sizes) + sum(4 * w * h for w, h, _ in images), "flops": 0}


def exact(case, seed):
    """None: framebuffers are bytes."""
    return None
