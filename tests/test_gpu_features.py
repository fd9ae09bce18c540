"""The sizing network's per-path inputs (pfh_scene_features) against the same sums in float64: paths of 1
to 65 and 200 segments (a wave takes 64 at a time), every segment kind, several contours, zero-length
edges (skipped where directions turn), paths off the canvas and paths with no segment.  Tolerance:
fp32 sums of at most 800 terms and an arc cosine of an fp32 dot product (3.5e-4 for parallel edges)."""
import numpy as np
import pytest

import pfh
import scenegen

pytestmark = pytest.mark.gpu


def segments(sc, p):
    """Control polygons of a path's segments (closing lines included), as SegmentsIter gives them."""
    out = []
    for c in range(sc.path_contour_start[p], sc.path_contour_start[p + 1]):
        a, e = sc.contour_start[c], sc.contour_start[c + 1]
        pts, flg, i = sc.points[a:e], sc.point_flags[a:e], 0
        while i + 1 < len(pts):
            k = 1
            while flg[i + k]:
                k += 1
            out.append(pts[i:i + k + 1])
            i += k
        if len(pts) > 1 and np.hypot(*(pts[0] - pts[-1])) > 1e-4:
            out.append(np.stack([pts[-1], pts[0]]))
    return out


def expect(sc, p, side):
    segs = segments(sc, p)
    n = [sum(len(s) == k + 2 for s in segs) for k in range(3)]
    poly = turn = 0.0
    prev = None
    for s in segs:
        for d in np.diff(s.astype(np.float32), axis=0):
            ln = np.float32(np.sqrt(np.float32(d[0] * d[0]) + np.float32(d[1] * d[1])))
            poly += float(ln)
            if ln > 0:
                u = (d / ln).astype(np.float32)
                if prev is not None:
                    turn += float(np.arccos(np.clip(np.float32(u[0] * prev[0]) + np.float32(u[1] * prev[1]), -1, 1)))
                prev = u
    al = np.concatenate(segs) if segs else np.zeros((1, 2))
    lo, hi = al.min(0) / side, al.max(0) / side
    return [lo[0], lo[1], hi[0], hi[1], np.log1p(poly), np.log1p(turn)] + [np.log1p(k) for k in n]


def test_path_features():
    rng = np.random.default_rng(8)
    outs = []
    for n in (1, 2, 63, 64, 65, 200):
        for kind in range(4):  # lines, quads, cubics, mixed; every third segment repeats a point
            pts, flg = [rng.uniform(0, 300, 2)], [0]
            for i in range(n):
                k = kind if kind < 3 else i % 3
                new = rng.uniform(-50, 350, (k + 1, 2))
                if i % 3 == 2:
                    new[0] = pts[-1]
                pts += list(new)
                flg += [1, 2][:k] + [0]
            cut = [0, len(flg)]
            if n == 65 and kind == 0:  # a second contour
                cut = [0, n // 2, len(flg)]
            outs.append((np.array(pts), flg, cut, np.zeros(len(cut) - 1)))
    outs.append((np.array([[900.0, 900], [950, 910], [940, 960]]), [0, 0, 0], [0, 3], [1]))   # off the canvas
    outs.append((np.array([[5.0, 5]]), [0], [0, 1], [0]))                                     # no segment
    P = len(outs)
    sc = scenegen.outlines_scene(320, 240, outs, np.arange(P) % 2, np.full(P, 0xff112233, np.uint32))
    ctx = pfh.Context(0)
    got = ctx.features(ctx.upload(sc)).astype(np.float64)
    for p in range(P):
        np.testing.assert_allclose(got[p, :9], expect(sc, p, 320.0), rtol=2e-5, atol=4e-4, err_msg=str(p))
    np.testing.assert_allclose(got[:, 10], np.log(320.0), rtol=1e-6)
    np.testing.assert_array_equal(got[:, 11], sc.path_fill_rule)
    ctx.close()
