// gfx950 kernels of the rasterization pipeline.
//
// Stage map (reference GLSL compute stage -> kernel here):
//   dice.comp                   -> k_flatten_count / k_flatten_emit: the hybrid tiler's recursive
//                                  flatten (core/d3d9/tiler.cpp:284-315), chords in DFS order
//   bin.comp                    -> k_bin<COUNT/EMIT>: the tile walk of
//                                  each chord (tiler.cpp:131-279), exact float order, per path
//                                  with LDS counters; also writes every tile of the path's rect
//   bound.comp                  -> (the bin count pass initialises each path's tiles)
//   propagate.comp              -> k_propagate (prepare_tiles, tiler.cpp:369-439) + z-buffer
//   sort.comp                   -> k_entries + stable grouping by framebuffer tile
//   fill.comp / fill.frag       -> k_fill_masks: analytic box-filtered area, fixed-point
//   tile.comp / tile.frag       -> k_composite: premultiplied src-over in fp32, one RGBA8 store
//
// This translation unit is built with -ffp-contract=off: the flatten/bin
// arithmetic must round exactly like the reference's SSE code (no FMA).
#include "pfh_internal.h"

namespace pfh {

// ---------------------------------------------------------------------------
// helpers
// ---------------------------------------------------------------------------

// Sets up to ZERO_SPANS arrays in one launch (the per-launch clears, and the tables the host wrote to
// pinned memory: one dispatch and one tail instead of one per array and copy): index i of their
// concatenation lies in the first span whose end is past it.
__global__ void k_zero_spans(ZeroSpans z) {
    const uint64_t total = z.n ? z.end[z.n - 1] : 0;
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += stride) {
#pragma unroll
        for (int k = 0; k < ZERO_SPANS; k++) {
            const uint64_t start = k ? z.end[k - 1] : 0;
            if (k < z.n && i >= start && i < z.end[k]) z.p[k][i - start] = z.src[k] ? z.src[k][i - start] : 0u;
        }
    }
}

// _mm_max_ps(a, b) / _mm_min_ps(a, b): the second operand wins on NaN or equality.
__device__ __forceinline__ float sse_max(float a, float b) { return a > b ? a : b; }
__device__ __forceinline__ float sse_min(float a, float b) { return a < b ? a : b; }

struct Seg4 {
    float2 p0, c0, c1, p1;
};

__device__ __forceinline__ float2 f2add(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 f2sub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ float2 f2muls(float2 a, float s) { return make_float2(a.x * s, a.y * s); }

// core/data/segment.cpp:12-20 is_flat_cubic
__device__ __forceinline__ bool flat_cubic(const Seg4 &s) {
    float u0 = 3.0f * s.c0.x - s.p0.x - s.p0.x - s.p1.x;
    float u1 = 3.0f * s.c0.y - s.p0.y - s.p0.y - s.p1.y;
    float u2 = 3.0f * s.c1.x - s.p1.x - s.p1.x - s.p0.x;
    float u3 = 3.0f * s.c1.y - s.p1.y - s.p1.y - s.p0.y;
    u0 = u0 * u0;
    u1 = u1 * u1;
    u2 = u2 * u2;
    u3 = u3 * u3;
    return sse_max(u0, u2) + sse_max(u1, u3) <= 1.0f;  // FLATTENING_TOLERANCE, tiler.cpp:15
}

// core/data/segment.cpp:22-36 is_flat_quadratic
__device__ __forceinline__ bool flat_quad(const Seg4 &s) {
    float2 mid = f2muls(f2add(s.p0, s.p1), 0.5f);
    float2 dev = f2sub(s.c0, mid);
    return dev.x * dev.x + dev.y * dev.y <= 1.0f * 0.25f;
}

// ---------------------------------------------------------------------------
// Tile walk of one chord (hybrid semantics)
// ---------------------------------------------------------------------------

// The walk's side effects go either to global counters (atomics) or, when one wave or
// workgroup owns the whole path, to LDS arrays indexed by the tile's position in the path's
// rect (LDS = true): l_cnt holds fill counts (COUNT) or the tiles' next free fill slots
// (EMIT), l_delta the backdrop deltas and l_col the above-rect column backdrops.
// PACK: l_delta holds two tiles per word, 16 bits each biased by 0x8000, so that ±1 steps of
// either half never carry into the other while |sum| < 2^15 (a chord steps a tile at most once:
// callers use it for paths with fewer than 2^15 chords).
template <bool EMIT, bool LDS = false, bool PACK = false>
struct Walker {
    // scene / path state
    float vb_l, vb_r, vb_b;
    int32_t tl, tt, tr, tb, tw, th;
    uint32_t tbase, cbase;
    uint32_t *tile_cnt;
    int32_t *tile_delta, *col_bd;
    uint32_t *l_cnt;
    int32_t *l_delta, *l_col;
    uint4 *out;              // EMIT with dumps: fills in emission order
    uint2 *fills;            // EMIT: fills grouped by tile
    const uint32_t *tile_fill_off;
    uint32_t cap_fills;
    uint32_t count;          // fills emitted by this chord so far
    uint32_t out_base;       // first emission slot of this chord (EMIT)
    uint32_t guard;

    // One coordinate of a point in a tile's 8.8 units, as the low 12 bits of the result
    // (core/d3d9/object_builder.cpp:26-41): rint(clamp((v - origin) * 256, 0, 4095)), the origin given
    // times 256.  The product by 256 only moves the exponent, so one fma rounds as the subtraction
    // does; v_med3 takes a NaN to 0 as the reference's max and min do; adding 2^23 rounds to
    // nearest even into the low mantissa bits.
    __device__ __forceinline__ static uint32_t quant(float v, float origin256) {
        const float t = __builtin_amdgcn_fmed3f(fmaf(v, 256.0f, -origin256), 0.0f, 4095.0f);
        return __float_as_uint(t + 8388608.0f);
    }
    __device__ __forceinline__ static uint32_t pack(uint32_t x, uint32_t y) {
        return __builtin_amdgcn_perm(y, x, 0x05040100u);  // the low halves, x below y
    }

    __device__ __forceinline__ void put(uint32_t pos, uint32_t a, uint32_t c, uint32_t j) {
        if (pos < cap_fills) fills[pos] = make_uint2(a, c);
        if (out) {
            const uint32_t d = out_base + count;
            if (d < cap_fills) out[d] = make_uint4(a, c, tbase + j, 0u);
        }
        count++;
    }

    // core/d3d9/object_builder.cpp:19-64 add_fill, for the fills of one step of a chord in tile
    // (tx, ty): its piece from -> to, then, with `up`, (to, corner) or, with `down`, (corner, from),
    // corner being the tile's origin, whose 8.8 coordinates are 0.  A fill with equal x ends is dropped.
    // Both go to one tile: one cursor add.
    __device__ __forceinline__ void add_fills(float2 from, float2 to, int tx, int ty, bool up, bool down) {
        const uint32_t ox = (uint32_t)tx - (uint32_t)tl, oy = (uint32_t)ty - (uint32_t)tt;
        if (ox >= (uint32_t)tw || oy >= (uint32_t)th) return;
        const float ox256 = (float)tx * 4096.0f;
        const uint32_t fx = quant(from.x, ox256), ex = quant(to.x, ox256);
        const bool piece = fx != ex;
        const bool aux = (up || down) && ((up ? ex : fx) & 0xffffu) != 0;
        if (!piece && !aux) return;
        const uint32_t n = (piece ? 1u : 0u) + (aux ? 1u : 0u);
        // tile within the path's rect (rect sides are below 2^24 tiles: a 24-bit multiply-add)
        const uint32_t j = __umul24(oy, (uint32_t)tw) + ox;
        if (!EMIT) {
            if (LDS) atomicAdd(&l_cnt[j], n);
            else atomicAdd(&tile_cnt[tbase + j], n);
            count += n;
        } else {
            // straight into the tile's range; order inside a tile is free (coverage is
            // accumulated in fixed point)
            uint32_t pos;
            if (LDS) {
                pos = atomicAdd(&l_cnt[j], n);
            } else {
                const uint32_t slot = atomicSub(&tile_cnt[tbase + j], n) - n;
                // written by this block in this launch: read from L2
                pos = __hip_atomic_load(&tile_fill_off[tbase + j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + slot;
            }
            const float oy256 = (float)ty * 4096.0f;
            const uint32_t a = pack(fx, quant(from.y, oy256)), c = pack(ex, quant(to.y, oy256));
            if (piece) put(pos, a, c, j);
            if (aux) put(pos + n - 1u, up ? c : 0u, up ? 0u : a, j);
        }
    }

    // core/d3d9/object_builder.cpp:96-114 adjust_alpha_tile_backdrop
    __device__ __forceinline__ void adjust(int tx, int ty, int delta) {
        if (EMIT) return;  // backdrops are accumulated once, in the count pass
        int ox = tx - tl, oy = ty - tt;
        if (ox < 0 || ox >= tw || oy >= th) return;
        if (oy < 0) {
            if (LDS) atomicAdd(&l_col[ox], delta);
            else atomicAdd(&col_bd[cbase + ox], delta);
            return;
        }
        const uint32_t j = __umul24((uint32_t)oy, (uint32_t)tw) + (uint32_t)ox;
        if (LDS && PACK) atomicAdd(reinterpret_cast<uint32_t *>(l_delta) + (j >> 1), (uint32_t)delta << (16 * (j & 1)));
        else if (LDS) atomicAdd(&l_delta[j], delta);
        else atomicAdd(&tile_delta[tbase + j], delta);
    }

    __device__ __forceinline__ static uint32_t outcode(float2 p, float l, float t, float r, float bb) {
        uint32_t f = 0;
        if (p.x < l) f |= 1;
        else if (p.x > r) f |= 2;
        if (p.y < t) f |= 4;
        else if (p.y > bb) f |= 8;
        return f;
    }

    // common/math/basic.h:45-53 lerp with t clamped to [0, 1]
    __device__ __forceinline__ static float lerpc(float a, float bv, float t) {
        t = t < 0.0f ? 0.0f : (t > 1.0f ? 1.0f : t);
        return a + (bv - a) * t;
    }

    // core/d3d9/tiler.cpp:65-125 Cohen–Sutherland against the view box with top = -inf
    __device__ bool clip(float2 &from, float2 &to) {
        const float l = vb_l, t = -INFINITY, r = vb_r, bb = vb_b;
        uint32_t of = outcode(from, l, t, r, bb), ot = outcode(to, l, t, r, bb);
        for (int iter = 0; iter < 64; iter++) {
            if (of == 0 && ot == 0) return true;
            if ((of & ot) != 0) return false;
            bool clip_from = of > ot;
            uint32_t oc = clip_from ? of : ot;
            // the first edge of the outcode (left, right, top, bottom): a vertical edge fixes x and
            // interpolates y, a horizontal one the reverse.  The operands are selected first so
            // that one division serves every case (lanes clipping different edges run it once).
            const bool vert = (oc & 3u) != 0;
            const float edge = (oc & 1u) ? l : ((oc & 2u) ? r : ((oc & 4u) ? t : bb));
            const float a0 = vert ? from.x : from.y, a1 = vert ? to.x : to.y;
            const float b0 = vert ? from.y : from.x, b1 = vert ? to.y : to.x;
            const float other = lerpc(b0, b1, (edge - a0) / (a1 - a0));
            const float2 p = vert ? make_float2(edge, other) : make_float2(other, edge);
            if (clip_from) {
                from = p;
                of = outcode(p, l, t, r, bb);
            } else {
                to = p;
                ot = outcode(p, l, t, r, bb);
            }
        }
        guard++;
        return false;
    }

    // core/d3d9/tiler.cpp:131-279 process_line_segment
    __device__ void line(float2 from, float2 to) {
        if (!isfinite(from.x) || !isfinite(from.y) || !isfinite(to.x) || !isfinite(to.y)) return;
        if (!clip(from, to)) return;
        const float inv = 1.0f / 16.0f;
        int fx = (int)floorf(from.x * inv), fy = (int)floorf(from.y * inv);
        int ex = (int)floorf(to.x * inv), ey = (int)floorf(to.y * inv);
        float2 vec = f2sub(to, from);
        int stx = vec.x < 0 ? -1 : 1, sty = vec.y < 0 ? -1 : 1;
        float crx = ((float)fx + (vec.x >= 0 ? 1.0f : 0.0f)) * 16.0f;
        float cry = ((float)fy + (vec.y >= 0 ? 1.0f : 0.0f)) * 16.0f;
        float tmx = (crx - from.x) / vec.x, tmy = (cry - from.y) / vec.y;
        float tdx = fabsf(16.0f / vec.x), tdy = fabsf(16.0f / vec.y);
        float2 cur = from;
        int cx = fx, cy = fy;
        int last = 0;  // 0 none, 1 X, 2 Y
        const int64_t dx = (int64_t)ex - fx, dy = (int64_t)ey - fy;
        // steps before the guard trips (a count of 2^31 or more, for chords of 2^31 tiles, is cut there)
        const int64_t lim = (dx < 0 ? -dx : dx) + (dy < 0 ? -dy : dy) + 2;
        for (uint32_t left = (uint32_t)(lim < 0x7fffffff ? lim : 0x7fffffff) + 1u;; left--) {
            if (left == 0) {
                guard++;
                break;
            }
            int next;
            if (tmx < tmy) next = 1;
            else if (tmx > tmy) next = 2;
            else next = stx > 0 ? 1 : 2;
            float nt = next == 1 ? tmx : tmy;
            nt = (1.0f < nt) ? 1.0f : nt;  // std::min(next_t, 1.0f)
            if (cx == ex && cy == ey) next = 0;
            float2 npos = f2add(from, f2muls(vec, nt));  // LineSegmentF::sample
            // with the auxiliary fill along the tile's left edge: (npos, corner) when stepping up out of
            // the tile, (corner, cur) when having stepped down into it
            add_fills(cur, npos, cx, cy, sty < 0 && next == 2, sty > 0 && last == 2);
            // the backdrop step when leaving to the right or having entered from the left
            if ((stx < 0 && last == 1) || (stx > 0 && next == 1)) adjust(cx, cy, stx < 0 ? 1 : -1);
            if (next == 1) {
                tmx += tdx;
                cx += stx;
            } else if (next == 2) {
                tmy += tdy;
                cy += sty;
            } else {
                break;
            }
            cur = npos;
            last = next;
        }
    }
};

// Orders the LDS accesses of a wave's lanes before and after it.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ---------------------------------------------------------------------------
// Flatten: chords of every segment, in depth-first order
// ---------------------------------------------------------------------------
//
// core/d3d9/tiler.cpp:284-315 process_segment (depth first, first half first) and
// core/data/segment.cpp:42-126 split_cubic / split_quadratic at t = 0.5.
//
// A curve's subdivision tree to depth FLAT_LEVELS is described by 64 bits: bit i is set when a
// leaf (a flat piece) starts at i / 64 of the parameter range.  The count pass finds the bits, in
// any order and with every lane of a wave busy; the emit pass needs no flatness test and no
// stack: chord i of a curve ends where leaf i + 1 starts, at a dyadic parameter e / 64 that at
// most 6 halvings from the curve's ends reach, so a lane takes one output point, and consecutive
// lanes store consecutive points.  A curve that is not flat at depth FLAT_LEVELS (its halves there
// are longer than the benchmark generators' curves at the size of a 4096^2 canvas ever give) has no
// bits and is flattened by its whole wave (flatten_wave), down to MAX_FLATTEN_DEPTH.
constexpr int FLAT_LEVELS = 6;
constexpr uint32_t FLAT_STACK = 128;     // pending nodes per wave (36 B each): 6 workgroups per CU

// The halves of a piece at t = 0.5 (core/data/segment.cpp:42-126), one path for both kinds (lanes
// holding quads and cubics run it once).  A quad is held as (p0, c, c, p1): p01 = lerp(p0, c) and
// p23 = lerp(c, p1) are its qa and qb, and taking them in place of p012 and p123 makes
// p0123 = lerp(qa, qb), its midpoint: halves (p0, qa, qa, qc), (qc, qb, qb, p1).  lerp at 0.5 is
// a + (b - a) * 0.5, whose product only changes the exponent: one fma rounds as the two operations do.
__device__ __forceinline__ float2 mid2(float2 a, float2 b) {
    return make_float2(fmaf(b.x - a.x, 0.5f, a.x), fmaf(b.y - a.y, 0.5f, a.y));
}
__device__ __forceinline__ void split_mid(const Seg4 &s, bool quad, Seg4 &a, Seg4 &r) {
    const float2 p01 = mid2(s.p0, s.c0), p12 = mid2(s.c0, s.c1), p23 = mid2(s.c1, s.p1);
    const float2 m0 = mid2(p01, p12), m1 = mid2(p12, p23);
    const float2 p012 = quad ? p01 : m0, p123 = quad ? p23 : m1;
    const float2 p0123 = mid2(p012, p123);
    a = Seg4{s.p0, p01, p012, p0123};
    r = Seg4{p0123, p123, p23, s.p1};
}

// A segment as the flattener takes it: its points (a quad as p0, c, c, p1; a line's ends in p0 and
// p1) and kind; kind 0 when nothing comes of it (no kind, or a non-finite point: every piece of it
// is non-finite, and process_line_segment drops those, tiler.cpp:133-136).
struct FlatSeg {
    Seg4 s;
    uint32_t kind;  // SegKind
    bool brk;       // starts a chain of chords: a separator and its start point come first
};
__device__ __forceinline__ FlatSeg load_flat_seg(const BatchDev &b, int k, uint32_t g) {
    FlatSeg f{};
    while (g >= b.seg_bases[k + 1]) k++;  // k: a scene at or before g's
    const SceneDev &sc = b.scenes[k];
    const uint2 sg = sc.segs[g - sc.seg_base];
    const uint32_t kd = sg.y & SEG_KIND_MASK;
    if (kd == 0) return f;
    const float2 *P = sc.pts + sg.x;
    f.s.p0 = P[0];
    f.s.p1 = f.s.c0 = f.s.c1 = P[1];
    if (kd != SEG_LINE) f.s.p1 = P[2];
    if (kd == SEG_CUBIC) {
        f.s.c1 = f.s.p1;
        f.s.p1 = P[3];
    }
    const Seg4 &s = f.s;
    const bool finite = isfinite(s.p0.x) && isfinite(s.p0.y) && isfinite(s.c0.x) && isfinite(s.c0.y) &&
                        isfinite(s.c1.x) && isfinite(s.c1.y) && isfinite(s.p1.x) && isfinite(s.p1.y);
    f.kind = finite ? kd : 0u;
    f.brk = finite && (sg.y & SEG_CHAIN_BREAK) != 0;
    return f;
}

__device__ __forceinline__ uint32_t mbcnt64(uint64_t m) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// One curve by a whole wave (every lane holds it): lane j owns the j-th node of depth FLAT_LEVELS,
// left to right, and walks down to it from the root by the same splits and flatness tests as the
// depth-first recursion; where a node on the way is flat, the leftmost lane under it takes the
// chord.  The chords below a lane's node are reached one by one from that node (no stack): the
// next leaf starts where the last one ended, at t in units of 2^-(MAX_FLATTEN_DEPTH - FLAT_LEVELS)
// of the node.  Lanes in order hold the curve's chords in order.  Returns their number; EMIT:
// writes their end points at out[0 .. room).
template <bool EMIT>
__device__ uint32_t flatten_wave(const Seg4 &root, bool quad, float2 *out, uint32_t room, uint32_t &guard) {
    const uint32_t lane = threadIdx.x & 63;
    Seg4 node = root;
    bool leaf = false, mine = false;
    for (int lv = 0; lv < FLAT_LEVELS; lv++) {
        if (quad ? flat_quad(node) : flat_cubic(node)) {
            leaf = true;
            mine = (lane & ((1u << (FLAT_LEVELS - lv)) - 1u)) == 0;
            break;
        }
        Seg4 a, r;
        split_mid(node, quad, a, r);
        node = ((lane >> (FLAT_LEVELS - 1 - lv)) & 1u) ? r : a;
    }
    constexpr uint32_t SPAN = 1u << (MAX_FLATTEN_DEPTH - FLAT_LEVELS);
    auto walk = [&](bool emit, uint32_t at) {
        uint32_t n = 0;
        for (uint32_t t = 0; t < SPAN;) {
            Seg4 q = node;
            int d = FLAT_LEVELS;
            bool flat;
            while (true) {
                flat = quad ? flat_quad(q) : flat_cubic(q);
                if (flat || d >= MAX_FLATTEN_DEPTH) break;
                Seg4 a, r;
                split_mid(q, quad, a, r);
                q = ((t >> (MAX_FLATTEN_DEPTH - 1 - d)) & 1u) ? r : a;
                d++;
            }
            if (!emit && !flat) guard++;
            if (emit && at + n < room) out[at + n] = q.p1;
            n++;
            t += 1u << (MAX_FLATTEN_DEPTH - d);
        }
        return n;
    };
    const uint32_t cnt = leaf ? (mine ? 1u : 0u) : walk(false, 0);
    const uint32_t incl = wave_inclusive_sum(cnt);
    if (EMIT) {
        const uint32_t at = incl - cnt;
        if (!leaf) walk(true, at);
        else if (mine && at < room) out[at] = node.p1;
    }
    return __shfl(incl, 63, 64);
}

// Count pass.  A wave takes a chunk of consecutive segments (at most 64, one per lane): lines and flat
// curves are finished at once, the other curves go to a stack of nodes still to be halved, in LDS,
// that the wave's lanes share.  Each step a lane halves its node and tests both halves: a flat one
// sets its bit, one that is not the lane keeps, and where both are not it pushes the right one; a
// lane left without a node takes the top of the stack.  So a wave takes about (its inner nodes) / 64
// steps instead of its deepest curve's depth-first walk, which is what bounded small launches:
// the 512^2 cubic scene's 512 curves (37 chords each) took 83 us with a lane per curve, 9 us so; the
// 4096^2 scene (341 k segments) 89 -> 25 us, the 48-scene batch (4.4 M) 321 -> 130 us.  Bound by
// VALU and scalar issue.  Several chunks per wave, the next one loaded ahead, gain 2 % on the batch
// and lose up to half on the smaller ones: fewer waves.
__global__ __launch_bounds__(256) void k_flatten_count(BatchDev b, uint32_t chunk) {
    __shared__ float4 s_p0c0[4][FLAT_STACK], s_c1p1[4][FLAT_STACK];
    __shared__ uint32_t s_meta[4][FLAT_STACK];  // slot | first 64th << 6 | depth << 12 | quad << 15
    __shared__ unsigned long long s_mask[4][64], s_deep[4];
    const uint32_t lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const uint64_t w0 = ((uint64_t)blockIdx.x * 4 + wv) * chunk;
    if (w0 >= b.n_segs) return;  // whole wave: no block-wide barriers below
    const uint32_t g = (uint32_t)w0 + lane;
    const bool in = lane < chunk && g < b.n_segs;
    const int k0 = find_scene_wave(b.seg_bases, b.n_scenes, (uint32_t)w0);
    FlatSeg f{};
    if (in) f = load_flat_seg(b, k0, g);
    const bool curve = f.kind > SEG_LINE;
    // stream points of a segment: its chords' ends, and a chain's separator and start point
    const uint32_t extra = f.brk ? 2u : 0u;
    uint32_t top;  // pending nodes (wave-uniform)
    {
        const bool quad = f.kind == SEG_QUAD;
        const bool flat = quad ? flat_quad(f.s) : flat_cubic(f.s);
        const bool node = curve && !flat;
        const uint64_t m = __ballot(node);
        s_mask[wv][lane] = flat ? 1ull : 0ull;
        if (lane == 0) s_deep[wv] = 0ull;
        if (node) {
            const uint32_t at = mbcnt64(m);
            s_p0c0[wv][at] = make_float4(f.s.p0.x, f.s.p0.y, f.s.c0.x, f.s.c0.y);
            s_c1p1[wv][at] = make_float4(f.s.c1.x, f.s.c1.y, f.s.p1.x, f.s.p1.y);
            s_meta[wv][at] = lane | (quad ? 1u << 15 : 0u);
        }
        top = (uint32_t)__popcll(m);
    }
    wave_sync();
    Seg4 s{};
    uint32_t meta = 0;
    bool active = false;
    while (true) {
        // idle lanes take the top nodes
        const uint64_t idle = __ballot(!active);
        if (idle && top) {
            const uint32_t rank = mbcnt64(idle);
            if (!active && rank < top) {
                const uint32_t at = top - 1 - rank;
                const float4 u = s_p0c0[wv][at], v = s_c1p1[wv][at];
                s = Seg4{make_float2(u.x, u.y), make_float2(u.z, u.w), make_float2(v.x, v.y), make_float2(v.z, v.w)};
                meta = s_meta[wv][at];
                active = true;
            }
            top -= min(top, (uint32_t)__popcll(idle));
            wave_sync();  // read before the pushes below overwrite the slots
        } else if (idle == ~0ull) {
            break;
        }
        const bool quad = (meta & (1u << 15)) != 0;
        const uint32_t depth = (meta >> 12) & 7u, key = (meta >> 6) & 63u, slot = meta & 63u;
        Seg4 a, r;
        split_mid(s, quad, a, r);
        const bool flat_a = quad ? flat_quad(a) : flat_cubic(a), flat_r = quad ? flat_quad(r) : flat_cubic(r);
        // halves at the last level that are not flat: their curve is left to the whole wave
        const bool inner = depth + 1 < FLAT_LEVELS;
        const bool push = active && inner && !flat_a && !flat_r;
        const uint64_t pm = __ballot(push);
        const uint32_t rank = mbcnt64(pm), room = FLAT_STACK - top;
        const uint32_t half = 32u >> depth;
        if (active && !(push && rank >= room)) {  // a lane without room for its right half waits with its node
            const uint64_t bits = (flat_a ? 1ull << key : 0ull) | (flat_r ? 1ull << (key + half) : 0ull);
            if (bits) atomicOr(&s_mask[wv][slot], bits);
            if (!inner && !(flat_a && flat_r)) atomicOr(&s_deep[wv], 1ull << slot);
            meta += 1u << 12;
            if (push) {
                const uint32_t at = top + rank;
                s_p0c0[wv][at] = make_float4(r.p0.x, r.p0.y, r.c0.x, r.c0.y);
                s_c1p1[wv][at] = make_float4(r.c1.x, r.c1.y, r.p1.x, r.p1.y);
                s_meta[wv][at] = meta + (half << 6);
            }
            if (flat_a) meta += half << 6;
            s = flat_a ? r : a;
            active = inner && !(flat_a && flat_r);
        }
        // a full stack and every lane waiting: the first lane's curve is left to the whole wave
        if (room == 0 && pm == ~0ull && lane == 0) {
            atomicOr(&s_deep[wv], 1ull << slot);
            active = false;
        }
        top += min((uint32_t)__popcll(pm), room);
        wave_sync();
    }
    uint64_t deep = s_deep[wv];
    deep = ((uint64_t)__builtin_amdgcn_readfirstlane((uint32_t)(deep >> 32)) << 32) | __builtin_amdgcn_readfirstlane((uint32_t)deep);
    uint32_t cnt = f.kind == SEG_LINE ? 1u + extra : 0u;
    if (curve) {
        const uint64_t m = (deep >> lane) & 1ull ? 0ull : s_mask[wv][lane];
        if (b.seg_mask) b.seg_mask[g] = m;
        cnt = (uint32_t)__popcll(m) + extra;
    }
    uint32_t guard = 0;
    while (deep) {  // wave-uniform
        const uint32_t i = (uint32_t)__builtin_ctzll(deep);
        deep &= deep - 1;
        const FlatSeg d = load_flat_seg(b, k0, (uint32_t)w0 + i);
        const uint32_t n = flatten_wave<false>(d.s, d.kind == SEG_QUAD, nullptr, 0u, guard);
        if (lane == i) cnt += n;
    }
    if (in) b.seg_cnt[g] = cnt;
    // the totals of the emit pass's chunks (this wave's segments are one of them or two)
    const uint32_t incl = wave_inclusive_sum(cnt);
    for (uint32_t c = 0; c < chunk; c += b.seg_chunk) {
        const uint32_t first = (uint32_t)w0 + c, below = c ? __shfl(incl, (int)c - 1, 64) : 0u;
        const uint32_t sum = __shfl(incl, (int)(c + b.seg_chunk - 1), 64) - below;
        if (lane == 0 && first < b.n_segs) b.chunk_off[first / b.seg_chunk] = sum;
    }
    if (guard) atomicAdd(&b.counters[C_GUARD], guard);
}

// Position of the n-th (from 0) set bit of m.
__device__ __forceinline__ uint32_t nth_bit(uint64_t m, uint32_t n) {
    uint32_t w = (uint32_t)m, pos = 0, c = (uint32_t)__popc(w);
    if (n >= c) {
        n -= c;
        w = (uint32_t)(m >> 32);
        pos = 32;
    }
#pragma unroll
    for (uint32_t h = 16; h >= 1; h >>= 1) {
        c = (uint32_t)__popc(w & ((1u << h) - 1u));
        const bool up = n >= c;
        n -= up ? c : 0u;
        w = up ? w >> h : w;
        pos += up ? h : 0u;
    }
    return pos;
}

// Emit pass: a wave per chunk of segments, a lane per stream point, 64 points at a time.  The
// segment owning a point is the last one starting at or before it: marks at the segments' first
// points, their ballot, and for the points before a window's first mark the last owner of the
// window before.  A chord's end at e / 64 (e the next leaf's start) is the midpoint of the node that
// e splits: the node's 6 - ctz(e) - 1 ancestors halved on the way, by e's top bits.  Stores are
// consecutive (a lane per curve scattered 8-byte stores, lines written back several times):
// 4096^2 scene 93 -> 27 us, 48-scene batch 417 -> 159 us, passes over lines included.
__global__ __launch_bounds__(256) void k_flatten_emit(BatchDev b) {
    __shared__ float4 s_p0c0[4][64], s_c1p1[4][64];
    __shared__ unsigned long long s_mask[4][64];
    __shared__ uint32_t s_start[4][64];  // first point in the chunk | quad << 30 | chain start << 31
    __shared__ uint8_t s_mark[4][64];    // of a window: owner + 1 where its points start
    const uint32_t lane = threadIdx.x & 63, wv = threadIdx.x >> 6, chunk = b.seg_chunk;
    const uint64_t w0 = ((uint64_t)blockIdx.x * 4 + wv) * chunk;
    if (w0 >= b.n_segs) return;  // whole wave
    const uint32_t g = (uint32_t)w0 + lane;
    const bool in = lane < chunk && g < b.n_segs;
    const int k0 = find_scene_wave(b.seg_bases, b.n_scenes, (uint32_t)w0);
    const uint32_t base = __builtin_amdgcn_readfirstlane(b.chunk_off[(uint32_t)w0 / chunk]);
    uint32_t cnt = 0;
    uint64_t mask = 0;
    FlatSeg f{};
    if (in) {
        cnt = b.seg_cnt[g];
        f = load_flat_seg(b, k0, g);
        // a line is one leaf over the whole range
        // (without room for the bits every curve is flattened again by the whole wave)
        mask = f.kind > SEG_LINE ? (b.seg_mask ? b.seg_mask[g] : 0ull) : 1ull;
    }
    const uint32_t incl = wave_inclusive_sum(cnt);
    const uint32_t total = __builtin_amdgcn_readlane(incl, 63), start = incl - cnt;
    if (in) b.seg_cnt[g] = base + start;  // from here on a segment's offset
    const uint64_t deep = __ballot(cnt != 0 && mask == 0);
    s_p0c0[wv][lane] = make_float4(f.s.p0.x, f.s.p0.y, f.s.c0.x, f.s.c0.y);
    s_c1p1[wv][lane] = make_float4(f.s.c1.x, f.s.c1.y, f.s.p1.x, f.s.p1.y);
    s_mask[wv][lane] = mask;
    s_start[wv][lane] = start | (f.kind == SEG_QUAD ? 1u << 30 : 0u) | (f.brk ? 1u << 31 : 0u);
    uint32_t last = 0;  // owner + 1 of the points before the window's first mark
    for (uint32_t q0 = 0; q0 < total; q0 += 64) {  // wave-uniform
        s_mark[wv][lane] = 0;
        wave_sync();
        if (cnt != 0 && start - q0 < 64u) s_mark[wv][start - q0] = (uint8_t)(lane + 1);
        wave_sync();
        const uint32_t mk = s_mark[wv][lane];
        const uint64_t marks = __ballot(mk != 0);
        const uint64_t upto = marks & (~0ull >> (63 - lane));
        const uint32_t owner = upto ? s_mark[wv][63 - __clzll(upto)] : last;
        const uint32_t q = q0 + lane;
        if (q < total && owner) {
            const uint32_t o = owner - 1, st = s_start[wv][o];
            const uint64_t m = s_mask[wv][o];
            const float4 u = s_p0c0[wv][o], v = s_c1p1[wv][o];
            Seg4 s{make_float2(u.x, u.y), make_float2(u.z, u.w), make_float2(v.x, v.y), make_float2(v.z, v.w)};
            const bool quad = (st & (1u << 30)) != 0;
            int i = (int)(q - (st & 0x3fffffffu)) - ((st >> 31) ? 2 : 0);
            float2 p;
            if (i < 0) {  // the chain's separator (a NaN point: its chords emit nothing) and start
                p = i == -2 ? make_float2(__builtin_nanf(""), __builtin_nanf("")) : s.p0;
            } else {
                const uint32_t key = nth_bit(m, (uint32_t)i);
                const uint64_t after = (m >> key) >> 1;  // leaves past this one
                const uint32_t e = after ? key + 1 + (uint32_t)__builtin_ctzll(after) : 64u;
                const int n = FLAT_LEVELS - (int)__builtin_ctz(e);
                for (int lv = 0; lv < n; lv++) {
                    Seg4 a, r;
                    split_mid(s, quad, a, r);
                    s = ((e >> (FLAT_LEVELS - 1 - lv)) & 1u) ? r : a;
                }
                p = n ? s.p0 : s.p1;  // e's lowest bit is set: the last half taken starts there
            }
            if ((m != 0 || i < 0) && base + q < b.cap_lines) b.lines[base + q] = p;
        }
        last = marks ? (uint32_t)__builtin_amdgcn_readlane(mk, 63 - __clzll(marks)) : last;
        wave_sync();  // the next window rewrites the marks
    }
    uint64_t dm = deep;
    uint32_t guard = 0;
    while (dm) {  // wave-uniform
        const uint32_t i = (uint32_t)__builtin_ctzll(dm);
        dm &= dm - 1;
        const float4 u = s_p0c0[wv][i], v = s_c1p1[wv][i];
        const uint32_t st = s_start[wv][i];
        const uint32_t at = base + (st & 0x3fffffffu) + ((st >> 31) ? 2u : 0u);
        if (at >= b.cap_lines) continue;
        flatten_wave<true>(Seg4{make_float2(u.x, u.y), make_float2(u.z, u.w), make_float2(v.x, v.y), make_float2(v.z, v.w)},
                           (st & (1u << 30)) != 0, b.lines + at, b.cap_lines - at, guard);
    }
}

// ---------------------------------------------------------------------------
// Device-wide exclusive scan, 4096 items per block
// ---------------------------------------------------------------------------

constexpr int SCAN_THREADS = 256;
constexpr int SCAN_ITEMS = 16;
constexpr int SCAN_TILE = SCAN_THREADS * SCAN_ITEMS;

struct U2 {
    uint32_t x, y;
    __device__ __forceinline__ U2 operator+(const U2 &o) const { return U2{x + o.x, y + o.y}; }
};

__device__ __forceinline__ uint32_t shfl_up_val(uint32_t v, int d) { return __shfl_up(v, d, 64); }
__device__ __forceinline__ U2 shfl_up_val(U2 v, int d) { return U2{__shfl_up(v.x, d, 64), __shfl_up(v.y, d, 64)}; }

template <typename T>
__device__ __forceinline__ T zero_of() { return T{}; }

// Exclusive scan of one value per thread across a block of THREADS threads; returns the block total.
template <typename T, int THREADS = SCAN_THREADS>
__device__ T block_exclusive_scan(T v, T &total) {
    __shared__ T wave_tot[THREADS / 64];
    int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    T inc = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        T o = shfl_up_val(inc, d);
        if (lane >= d) inc = inc + o;
    }
    if (lane == 63) wave_tot[wave] = inc;
    __syncthreads();
    T base = zero_of<T>();
    T all = zero_of<T>();
#pragma unroll
    for (int w = 0; w < THREADS / 64; w++) {
        if (w < wave) base = base + wave_tot[w];
        all = all + wave_tot[w];
    }
    __syncthreads();
    total = all;
    T excl_in_wave = shfl_up_val(inc, 1);
    if (lane == 0) excl_in_wave = zero_of<T>();
    return base + excl_in_wave;
}

// ---------------------------------------------------------------------------
// Bin: per path, one wave (small rects) or one workgroup (large rects or many segments)
// ---------------------------------------------------------------------------
//
// The chords of a path are contiguous (flatten emits in segment order, segments are in
// path order), and every tile and column of the path's rect belongs to it alone.  So the
// owner counts fills and accumulates backdrop deltas in LDS with LDS atomics and stores
// the whole rect once (COUNT), then hands out fill slots from LDS cursors seeded with the
// tiles' scanned offsets (EMIT).  No global atomics, and the work arrays need no clearing.

// Chord range [c0, c1) of local path p of scene sc (seg_cnt holds the scanned offsets).
__device__ __forceinline__ void path_chords(const BatchDev &b, const SceneDev &sc, uint32_t p, uint32_t &c0,
                                            uint32_t &c1) {
    const uint32_t g0 = sc.seg_base + sc.path_seg_off[p], g1 = sc.seg_base + sc.path_seg_off[p + 1];
    const uint32_t total = b.counters[C_LINES];
    c0 = g0 < b.n_segs ? b.seg_cnt[g0] : total;
    c1 = g1 < b.n_segs ? b.seg_cnt[g1] : total;
    c0 = min(c0, b.cap_lines);
    c1 = min(c1, b.cap_lines);
}

// The chords [c0, c1) of a path, thread `first` of `stride` taking every stride-th.  Most
// chords lie inside one tile, where process_line_segment emits exactly one fill (from, from +
// vec) and no auxiliary fill or backdrop step: the tile crossings it would compute are all at
// t >= 1.  Those are emitted at once; the others (crossing a tile boundary) are queued per wave
// in LDS (wq, WALK_QUEUE slots) and walked 64 at a time, so the DDA's divisions and steps run
// with every lane on a chord that needs them.
template <bool EMIT, bool LDS, bool PACK = false>
__device__ __forceinline__ void walk_chords(const BatchDev &b, const SceneDev &sc, const int4 &rect, uint32_t tbase,
                                            uint32_t cbase, uint32_t *l_cnt, int32_t *l_delta, int32_t *l_col,
                                            uint32_t c0, uint32_t c1, uint32_t first, uint32_t stride,
                                            uint32_t *wq) {
    const uint32_t lane = threadIdx.x & 63;
    const uint64_t lt_mask = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    uint32_t guard = 0;
    Walker<EMIT, LDS, PACK> w;
    w.vb_l = sc.vb_l;
    w.vb_r = sc.vb_r;
    w.vb_b = sc.vb_b;
    w.tl = rect.x;
    w.tt = rect.y;
    w.tr = rect.z;
    w.tb = rect.w;
    w.tw = rect.z - rect.x;
    w.th = rect.w - rect.y;
    w.tbase = tbase;
    w.cbase = cbase;
    w.tile_cnt = b.tile_cnt;
    w.tile_delta = b.tile_delta;
    w.col_bd = b.col_bd;
    w.l_cnt = l_cnt;
    w.l_delta = l_delta;
    w.l_col = l_col;
    w.out = b.dump ? b.dump_fills : nullptr;
    w.fills = b.fills;
    w.tile_fill_off = b.tile_fill_off;
    w.cap_fills = b.cap_fills;
    auto begin = [&](uint32_t i) {
        w.count = 0;
        w.guard = 0;
        w.out_base = (EMIT && b.dump) ? b.line_cnt[i] : 0u;
    };
    auto end = [&](uint32_t i) {
        if (!EMIT && b.dump) b.line_cnt[i] = w.count;  // fills per chord: canonical dump order only
        guard += w.guard;
    };
    uint32_t qn = 0;  // queued chords (wave-uniform)
    // chord i: stream points i and i + 1 of the path's range (the last point pairs with a NaN:
    // nothing is emitted, and the dump's per-chord count there is 0)
    auto chord = [&](uint32_t i) {
        const float2 a = b.lines[i];
        const float2 e = i + 1 < c1 ? b.lines[i + 1] : make_float2(__builtin_nanf(""), __builtin_nanf(""));
        return make_float4(a.x, a.y, e.x, e.y);
    };
    // count pass: the next chunk's chord is loaded while this one is processed (measured: the
    // count passes gain ~5 %, the emit passes, whose stores also wait, lose ~1 %)
    const float4 zero4 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    float4 ln_next = !EMIT && c0 + first < c1 ? chord(c0 + first) : zero4;
    for (uint32_t base = c0; base < c1; base += stride) {  // uniform over the wave
        const uint32_t i = base + first;
        const float4 ln_cur = ln_next;
        if (!EMIT && base + stride + first < c1) ln_next = chord(base + stride + first);
        bool multi = false;
        if (i < c1) {
            const float4 ln = EMIT ? chord(i) : ln_cur;
            float2 from = make_float2(ln.x, ln.y), to = make_float2(ln.z, ln.w);
            begin(i);
            if (isfinite(from.x) && isfinite(from.y) && isfinite(to.x) && isfinite(to.y) && w.clip(from, to)) {
                const float inv = 1.0f / 16.0f;
                const int fx = (int)floorf(from.x * inv), fy = (int)floorf(from.y * inv);
                const int ex = (int)floorf(to.x * inv), ey = (int)floorf(to.y * inv);
                const float2 vec = f2sub(to, from);
                // a -0 component makes a crossing time -inf: left to the full walk
                const bool neg_zero = (vec.x == 0.0f && signbit(vec.x)) || (vec.y == 0.0f && signbit(vec.y));
                if (fx == ex && fy == ey && !neg_zero) w.add_fills(from, f2add(from, vec), fx, fy, false, false);
                else multi = true;
            }
            if (!multi) end(i);
        }
        const uint64_t m = __ballot(multi);
        if (multi) wq[qn + (uint32_t)__popcll(m & lt_mask)] = i;
        qn += (uint32_t)__popcll(m);
        wave_sync();
        if (qn >= 64) {  // at most 127 queued: one full batch
            qn -= 64;
            const uint32_t ci = wq[qn + lane];
            wave_sync();  // read before the next chunk's chords overwrite the slots
            const float4 ln = chord(ci);
            begin(ci);
            w.line(make_float2(ln.x, ln.y), make_float2(ln.z, ln.w));
            end(ci);
        }
    }
    if (lane < qn) {  // the rest of the queue
        const uint32_t ci = wq[lane];
        const float4 ln = chord(ci);
        begin(ci);
        w.line(make_float2(ln.x, ln.y), make_float2(ln.z, ln.w));
        end(ci);
    }
    wave_sync();  // the queue is read before the caller reuses the wave's LDS
    if (!EMIT && guard) atomicAdd(&b.counters[C_GUARD], guard);
}


// Per-path totals and offsets.  The count pass stores each path's {fills, alpha tiles}
// (path_tot, batch path order); after their scan the emit pass turns its rect's tile counts
// into the tiles' fill offsets and alpha-tile indices (a local scan, row-major), writes
// them, and uses the fill offsets as its LDS cursors.  The batch-wide order of tiles is
// path order then row-major within the rect, so this equals a scan over all tiles.

__device__ __forceinline__ U2 wave_sum_u2(U2 v) {
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) {
        v.x += __shfl_xor(v.x, d, 64);
        v.y += __shfl_xor(v.y, d, 64);
    }
    return v;
}

// Mask rows per alpha tile: 2 for a clip path's tiles, whose coverage is kept under both fill rules.
__device__ __forceinline__ uint32_t alpha_rows(const BinItem &it) { return it.level != 0 ? 2u : 1u; }

// Whether a path's tiles are resolved in the bin passes: not where they depend on a clip path's (k_propagate).
__device__ __forceinline__ bool resolved_here(const BinItem &it) { return it.level == 0 && it.clip == CLIP_NONE; }

// Backdrops, tile status and z-buffer (core/d3d9/tiler.cpp:369-439) of a path that no clip path
// concerns, at the end of its count pass, whose counts and deltas are still in LDS: a column's backdrop
// is its running sum from the step above the rect down, which resolve_columns puts in the deltas'
// place.
// As a walk of its own down the batch's columns, a thread each, this took 155 us for 48 scenes (20
// million tiles), 30 us at 4096^2 and 25 us at 1240 x 1754, where it waited 14 times for a group of rows;
// the count pass is longer instead: 367 -> 424 us, 65 -> 81 and 30 -> 32 (the emit pass as long as before).
// A thread per column, 8 rows at a time: each group's reads go out before the first is used.  (Several
// threads to a column where the rect is narrower than the block, with a sum pass before: no faster, and
// 189 -> 209 us for the wave class of the 48 scenes.)
template <int N, typename D>
__device__ __forceinline__ void resolve_columns(const BatchDev &b, const BinItem &it, uint32_t tw, uint32_t th,
                                                D *delta, int32_t bias, const int32_t *col, uint32_t t) {
    for (uint32_t x = t; x < tw; x += N) {
        int32_t run = col[x];
        for (uint32_t r0 = 0; r0 < th; r0 += 8) {
            int32_t d[8];
#pragma unroll
            for (uint32_t i = 0; i < 8; i++) d[i] = r0 + i < th ? (int32_t)delta[(r0 + i) * tw + x] - bias : 0;
#pragma unroll
            for (uint32_t i = 0; i < 8; i++) {
                if (r0 + i < th) delta[(r0 + i) * tw + x] = (D)((int32_t)(int8_t)run + bias);
                run += (int8_t)d[i];
            }
        }
        if (b.dump) b.col_bd[it.cbase + x] = run;
    }
}

// Tile j of the rect (row-major, tw wide), its fills and backdrop known: its status, and for an opaque
// solid tile the z-buffer.  An alpha tile's backdrop waits in tile_delta for its mask record, which the
// emit pass writes once it knows the tile's place (store_tile_offset).
__device__ __forceinline__ void resolve_tile(const BatchDev &b, const BinItem &it, const SceneDev &sc, uint32_t tw,
                                             float inv_w, uint32_t j, uint32_t fills, int32_t bd) {
    const uint32_t t = it.tbase + j;
    const bool clear = (it.rule & 1u) && (bd & 1) == 0;
    b.tile_st[t] = fills ? TILE_ALPHA : (bd == 0 ? TILE_EMPTY : (clear ? TILE_CLEAR : TILE_SOLID));
    if (b.dump) b.tile_bd[t] = (int8_t)bd;
    if (fills) {
        b.tile_delta[t] = bd;
    } else if ((it.rgba >> 24) == 255u && bd != 0 && !clear) {
        uint32_t row = (uint32_t)((float)j * inv_w);  // off by at most one below 2^24 tiles
        if (row * tw > j) row--;
        else if ((row + 1) * tw <= j) row++;
        const int x = it.rect.x - sc.fb_x0 + (int)(j - row * tw), y = it.rect.y - sc.fb_y0 + (int)row;
        atomicMax(&b.zbuf[sc.fb_base + (uint32_t)(y * sc.fb_w + x)], it.p);
    }
}

// Emit pass: where tile t's fills start (`fills` of them) and its mask row.  bd: its tile_delta, read
// beside the counts (anything where it has no fills).  cursors: the fills are placed through tile_fill_off.
__device__ __forceinline__ void store_tile_offset(const BatchDev &b, const BinItem &it, uint32_t t, uint32_t off,
                                                  uint32_t fills, uint32_t ai, int32_t bd, bool cursors) {
    if (b.has_clips || b.dump || cursors) b.tile_fill_off[t] = off;  // dumps read it back
    b.tile_alpha_idx[t] = ai;  // all: whole lines (stored for alpha tiles alone, the entry pass 26 -> 34 us at 4096^2)
    if (fills && ai < b.cap_alpha && resolved_here(it))
        b.alpha_rec[ai] = make_uint4(off, off + fills, (uint32_t)(uint8_t)bd | ((it.rule & 1u) << 8), t);
}

// Inclusive prefix sums of (count, count > 0) across the wave.
__device__ __forceinline__ U2 wave_inclusive_u2(uint32_t c) {
    U2 v{c, c > 0 ? 1u : 0u};
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const U2 o = shfl_up_val(v, d);
        if (lane >= d) v = v + o;
    }
    return v;
}

// Wave: tile offsets of a rect of `area` tiles (counts in cnt_src, global) from the path's
// scanned base; offsets go to the tile arrays and, when given, to the LDS cursors.
// The masks of tiles resolved in the count pass are complete here: see resolve_tile.
__device__ __forceinline__ void wave_tile_offsets(const BatchDev &b, const BinItem &it, uint32_t area, U2 base,
                                                  uint32_t *l_cur) {
    const uint32_t tbase = it.tbase, aw = alpha_rows(it);
    const uint32_t lane = threadIdx.x & 63;
    for (uint32_t j0 = 0; j0 < area; j0 += 64) {
        const uint32_t j = j0 + lane;
        const uint32_t c = j < area ? b.tile_cnt[tbase + j] : 0u;
        const int32_t bd = j < area ? b.tile_delta[tbase + j] : 0;
        const U2 inc = wave_inclusive_u2(c);
        if (j < area) {
            const uint32_t off = base.x + inc.x - c;
            store_tile_offset(b, it, tbase + j, off, c, base.y + aw * (inc.y - (c > 0 ? 1u : 0u)), bd, l_cur == nullptr);
            if (l_cur) l_cur[j] = off;
        }
        base = base + U2{__shfl(inc.x, 63, 64), aw * __shfl(inc.y, 63, 64)};
    }
}

// Block version, called by every thread of a block of THREADS.
template <int THREADS>
__device__ __forceinline__ void block_tile_offsets(const BatchDev &b, const BinItem &it, uint32_t area, U2 base,
                                                   uint32_t *l_cur) {
    const uint32_t tbase = it.tbase, aw = alpha_rows(it);
    // tiles of a thread: a chunk costs a block-wide scan (50 whole-canvas rects 36 -> 24 us; no use to small rects)
    constexpr uint32_t ITEMS = THREADS == 1024 ? 4 : 1;
    for (uint32_t j0 = 0; j0 < area; j0 += THREADS * ITEMS) {
        const uint32_t j = j0 + threadIdx.x * ITEMS;
        uint32_t c[ITEMS];
        int32_t bd[ITEMS];
        U2 own{0, 0};
#pragma unroll
        for (uint32_t i = 0; i < ITEMS; i++) {
            c[i] = j + i < area ? b.tile_cnt[tbase + j + i] : 0u;
            bd[i] = j + i < area ? b.tile_delta[tbase + j + i] : 0;
        }
#pragma unroll
        for (uint32_t i = 0; i < ITEMS; i++) own = own + U2{c[i], c[i] > 0 ? 1u : 0u};
        U2 tot;
        U2 ex = block_exclusive_scan<U2, THREADS>(own, tot);
#pragma unroll
        for (uint32_t i = 0; i < ITEMS; i++) {
            if (j + i < area) {
                store_tile_offset(b, it, tbase + j + i, base.x + ex.x, c[i], base.y + aw * ex.y, bd[i], l_cur == nullptr);
                if (l_cur) l_cur[j + i] = base.x + ex.x;
            }
            ex = ex + U2{c[i], c[i] > 0 ? 1u : 0u};
        }
        base = base + U2{tot.x, aw * tot.y};
    }
}

// Block sum over a block's THREADS threads; `part` is a slot of LDS per wave the block no longer reads.
template <int THREADS>
__device__ __forceinline__ U2 block_sum_u2(U2 v, U2 *part) {
    v = wave_sum_u2(v);
    __syncthreads();  // part may alias data read just before
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
    __syncthreads();
    U2 t = part[0];
#pragma unroll
    for (int w = 1; w < THREADS / 64; w++) t = t + part[w];
    __syncthreads();
    return t;
}

// Group-class paths whose rect is the whole framebuffer, as destructive blend modes make it, past a bin
// block's LDS, that fit a block with more of it (k_bin_big).
__device__ __forceinline__ bool is_big(const BinItem &it, const SceneDev &sc) {
    const uint32_t tw = (uint32_t)max(it.rect.z - it.rect.x, 0), th = (uint32_t)max(it.rect.w - it.rect.y, 0);
    const uint64_t area = (uint64_t)tw * th;
    return tw == (uint32_t)sc.fb_w && area == sc.n_fb && (area > (uint32_t)BIN_GROUP_TILES || tw > (uint32_t)BIN_GROUP_COLS) &&
           area <= (uint32_t)BIN_BIG_TILES && tw <= (uint32_t)BIN_BIG_COLS && it.c1 - it.c0 < (1u << 15);
}

// One descriptor per binned path: thread per item, the first blocks for the wave class, the others for
// the group class.
__global__ __launch_bounds__(256) void k_bin_items(BatchDev b, uint32_t wave_blocks) {
    const bool grp = blockIdx.x >= wave_blocks;  // uniform over the block
    const uint32_t n = grp ? b.n_bin_group : b.n_bin_wave;
    const uint32_t *bases = grp ? b.bin_group_bases : b.bin_wave_bases;
    const uint32_t i = (blockIdx.x - (grp ? wave_blocks : 0u)) * blockDim.x + threadIdx.x;
    // every lane searches (lanes past the end with the last item), then those leave
    const int k = find_scene_lanes(bases, b.n_scenes, min(i, n - 1));
    if (i >= n) return;
    const SceneDev &sc = b.scenes[k];
    const uint32_t p = sc.bin_paths[(grp ? sc.n_bin_wave : 0u) + (i - bases[k])];
    BinItem it;
    it.rect = sc.path_rect[p];
    it.tbase = sc.tile_base + sc.path_tile_off[p];
    it.cbase = sc.col_base + sc.path_col_off[p];
    path_chords(b, sc, p, it.c0, it.c1);
    it.p = p;
    it.gp = sc.path_base + p;
    it.k = (uint32_t)k;
    it.rgba = sc.path_rgba[p];
    it.rule = sc.path_rule[p] | (sc.clip_own_rules ? RULE_CLIP_OWN : 0u);
    uint32_t cr = sc.path_clip ? sc.path_clip[p] : CLIP_NONE;
    if (cr < CLIP_EMPTY)
        cr = (cr & CLIP_GROUP) ? b.n_bin_wave + sc.bin_group_base + (cr & ~CLIP_GROUP) : sc.bin_wave_base + cr;
    it.clip = cr;
    it.level = sc.path_level ? (uint32_t)sc.path_level[p] : 0u;
    it.paint = sc.path_paint ? sc.path_paint[p] : PAINT_NONE;
    const uint32_t gi = (grp ? b.n_bin_wave : 0u) + i;
    b.bin_items[gi] = it;
    if (b.n_big && is_big(it, sc)) b.big_list[atomicAdd(&b.counters[C_BIG], 1u)] = gi;
    if (!b.has_clips) return;
    // for the propagate launches: the strips of clip paths and clipped draw paths, one add per wave and kind
    const uint64_t here = __ballot(true);
    const bool lead = (threadIdx.x & 63) == (uint32_t)__builtin_ctzll(here);
    const uint32_t strips = resolved_here(it) ? 0u : ((uint32_t)max(it.rect.z - it.rect.x, 0) + PROP_COLS - 1) / PROP_COLS;
    for (int kind = 0; kind < 2; kind++) {
        const uint32_t left = (it.level != 0) == (kind == 0) ? strips : 0u;
        uint32_t total = 0, before = 0;
        // sums over the wave's active lanes, a bit of the counts at a time
        for (uint32_t bit = 0; __ballot(left >> bit) != 0; bit++) {
            const uint64_t m = __ballot((left >> bit) & 1u);
            total += (uint32_t)__popcll(m) << bit;
            before += __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u)) << bit;
        }
        if (total == 0) continue;
        uint32_t first = 0;
        if (lead) first = atomicAdd(&b.counters[kind == 0 ? C_CLIP_STRIPS : C_DRAW_STRIPS], total);
        first = __builtin_amdgcn_readfirstlane(first) + before;
        for (uint32_t q = 0; q < left; q++)
            b.prop_strips[kind == 0 ? first + q : b.cap_strips - 1 - (first + q)] = make_uint2(gi, q * PROP_COLS);
    }
}

// LDS of a bin block: its path's arrays (group class), or a slice per wave (wave class).
template <bool EMIT, int THREADS>
struct BinPath {
    uint32_t cnt[BIN_GROUP_TILES];
    uint32_t delta[EMIT ? 1 : (BIN_GROUP_TILES + 1) / 2];  // packed, two tiles per word
    int32_t col[EMIT ? 1 : BIN_GROUP_COLS];
    uint32_t queue[THREADS / 64][WALK_QUEUE];
};
template <bool EMIT>
struct BinSlice {
    uint32_t cnt[BIN_WAVE_TILES];
    int32_t delta[EMIT ? 1 : BIN_WAVE_TILES];
    int32_t col[EMIT ? 1 : BIN_WAVE_COLS];
    uint32_t queue[WALK_QUEUE];
};
template <bool EMIT, int THREADS>
union BinLds {
    BinPath<EMIT, THREADS> g;
    BinSlice<EMIT> w[THREADS / 64];
};

// Wave class: a path per wave, in its own slice.
template <bool EMIT, int THREADS, typename Lds>
__device__ __forceinline__ void bin_wave(const BatchDev &b, Lds &lds, uint32_t item) {
    const uint32_t wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (item >= b.n_bin_wave) return;  // whole wave: no block-wide barriers below
    const BinItem it = b.bin_items[item];
    const SceneDev &sc = b.scenes[it.k];
    const int4 rect = it.rect;
    const uint32_t tw = (uint32_t)max(rect.z - rect.x, 0), th = (uint32_t)max(rect.w - rect.y, 0);
    const uint32_t area = tw * th;
    if (area > (uint32_t)BIN_WAVE_TILES || tw > (uint32_t)BIN_WAVE_COLS) return;  // not this class (host sorts)
    const uint32_t tbase = it.tbase, cbase = it.cbase;
    uint32_t *l_cnt = lds[wv].cnt;
    int32_t *l_delta = lds[wv].delta, *l_col = lds[wv].col;
    const uint32_t gp = it.gp;
    if (EMIT) {
        const uint2 base = b.path_tot[gp];
        wave_tile_offsets(b, it, area, U2{base.x, base.y}, l_cnt);
    } else {
        for (uint32_t j = lane; j < area; j += 64) {
            l_cnt[j] = 0;
            l_delta[j] = 0;
        }
        for (uint32_t j = lane; j < tw; j += 64) l_col[j] = 0;
    }
    wave_sync();
    walk_chords<EMIT, true>(b, sc, rect, tbase, cbase, l_cnt, l_delta, l_col, it.c0, it.c1, lane, 64, lds[wv].queue);
    if (!EMIT) {
        wave_sync();
        const bool resolve = resolved_here(it);
        if (resolve) {
            resolve_columns<64>(b, it, tw, th, l_delta, 0, l_col, lane);
            wave_sync();
        }
        const float inv_w = 1.0f / (float)(int)tw;
        U2 tot{0, 0};
        for (uint32_t j = lane; j < area; j += 64) {
            const uint32_t c = l_cnt[j];
            b.tile_cnt[tbase + j] = c;
            if (resolve) resolve_tile(b, it, sc, tw, inv_w, j, c, l_delta[j]);
            else b.tile_delta[tbase + j] = l_delta[j];
            tot = tot + U2{c, c > 0 ? 1u : 0u};
        }
        if (!resolve)
            for (uint32_t j = lane; j < tw; j += 64) b.col_bd[cbase + j] = l_col[j];
        tot = wave_sum_u2(tot);
        if (lane == 0) b.path_tot[gp] = make_uint2(tot.x, tot.y * alpha_rows(it));
    }
}

// Group class: one path per block; LDS when the rect fits (max_tiles, max_cols), else global atomics on the
// path's own (first zeroed) tiles.
template <bool EMIT, int THREADS>
__device__ __forceinline__ void bin_group(const BatchDev &b, const BinItem &it, uint32_t *s_cnt, uint32_t *s_delta,
                                          int32_t *s_col, uint32_t *queues, uint32_t max_tiles, uint32_t max_cols) {
    const SceneDev &sc = b.scenes[it.k];
    const int4 rect = it.rect;
    const uint32_t tw = (uint32_t)max(rect.z - rect.x, 0), th = (uint32_t)max(rect.w - rect.y, 0);
    const uint32_t area = tw * th;
    const uint32_t tbase = it.tbase, cbase = it.cbase;
    const uint32_t gp = it.gp;
    const uint32_t c0 = it.c0, c1 = it.c1;
    uint32_t *const queue = queues + WALK_QUEUE * (threadIdx.x >> 6);
    const bool resolve = !EMIT && resolved_here(it);
    const float inv_w = 1.0f / (float)(int)tw;
    // the packed LDS deltas hold sums below 2^15 in magnitude: at most one step per chord
    const bool in_lds = area <= max_tiles && tw <= max_cols && (EMIT || c1 - c0 < (1u << 15));
    if (in_lds) {
        if (EMIT) {
            const uint2 base = b.path_tot[gp];
            block_tile_offsets<THREADS>(b, it, area, U2{base.x, base.y}, s_cnt);
        } else {
            for (uint32_t j = threadIdx.x; j < area; j += THREADS) s_cnt[j] = 0;
            for (uint32_t j = threadIdx.x; j < (area + 1) / 2; j += THREADS) s_delta[j] = 0x80008000u;
            for (uint32_t j = threadIdx.x; j < tw; j += THREADS) s_col[j] = 0;
        }
        __syncthreads();
        walk_chords<EMIT, true, true>(b, sc, rect, tbase, cbase, s_cnt, reinterpret_cast<int32_t *>(s_delta), s_col,
                                      c0, c1, threadIdx.x, THREADS, queue);
        if (!EMIT) {
            __syncthreads();
            typedef uint16_t __attribute__((may_alias)) Half;
            Half *const half = reinterpret_cast<Half *>(s_delta);  // tile j's delta, biased
            if (resolve) {
                resolve_columns<THREADS>(b, it, tw, th, half, 0x8000, s_col, threadIdx.x);
                __syncthreads();
            }
            U2 tot{0, 0};
            for (uint32_t j = threadIdx.x; j < area; j += THREADS) {
                const uint32_t c = s_cnt[j];
                const int32_t d = (int32_t)half[j] - 0x8000;
                b.tile_cnt[tbase + j] = c;
                if (resolve) resolve_tile(b, it, sc, tw, inv_w, j, c, d);
                else b.tile_delta[tbase + j] = d;
                tot = tot + U2{c, c > 0 ? 1u : 0u};
            }
            if (!resolve)
                for (uint32_t j = threadIdx.x; j < tw; j += THREADS) b.col_bd[cbase + j] = s_col[j];
            tot = block_sum_u2<THREADS>(tot, reinterpret_cast<U2 *>(s_col));
            if (threadIdx.x == 0) b.path_tot[gp] = make_uint2(tot.x, tot.y * alpha_rows(it));
        }
    } else {
        if (EMIT) {
            const uint2 base = b.path_tot[gp];
            block_tile_offsets<THREADS>(b, it, area, U2{base.x, base.y}, nullptr);
            __threadfence();  // the offsets reach L2 before any thread reads them back
            __syncthreads();
        }
        if (!EMIT) {
            for (uint32_t j = threadIdx.x; j < area; j += THREADS) {
                b.tile_cnt[tbase + j] = 0;
                b.tile_delta[tbase + j] = 0;
            }
            for (uint32_t j = threadIdx.x; j < tw; j += THREADS) b.col_bd[cbase + j] = 0;
            __threadfence();  // the zeros reach L2 before any thread's atomics
            __syncthreads();
        }
        walk_chords<EMIT, false>(b, sc, rect, tbase, cbase, nullptr, nullptr, nullptr, c0, c1, threadIdx.x, THREADS,
                                 queue);
        if (!EMIT) {
            __threadfence();  // every thread's atomics are done before the counts are summed
            __syncthreads();
            U2 tot{0, 0};
            auto read = [](const auto *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
            if (resolve) {
                for (uint32_t x = threadIdx.x; x < tw; x += THREADS) {  // a thread per column, 8 rows at a time
                    int32_t run = read(&b.col_bd[cbase + x]);
                    for (uint32_t r0 = 0; r0 < th; r0 += 8) {
                        int32_t d[8];
                        uint32_t c[8];
#pragma unroll
                        for (uint32_t i = 0; i < 8; i++) {
                            const uint32_t t = tbase + (r0 + i) * tw + x;
                            d[i] = r0 + i < th ? read(&b.tile_delta[t]) : 0;
                            c[i] = r0 + i < th ? read(&b.tile_cnt[t]) : 0u;
                        }
#pragma unroll
                        for (uint32_t i = 0; i < 8; i++) {
                            if (r0 + i < th) resolve_tile(b, it, sc, tw, inv_w, (r0 + i) * tw + x, c[i], (int8_t)run);
                            run += (int8_t)d[i];
                            tot = tot + U2{c[i], c[i] > 0 ? 1u : 0u};
                        }
                    }
                    if (b.dump) b.col_bd[cbase + x] = run;
                }
            } else {
                for (uint32_t j = threadIdx.x; j < area; j += THREADS) {
                    const uint32_t c = read(&b.tile_cnt[tbase + j]);
                    tot = tot + U2{c, c > 0 ? 1u : 0u};
                }
            }
            tot = block_sum_u2<THREADS>(tot, reinterpret_cast<U2 *>(s_col));  // s_col is unused on this path
            if (threadIdx.x == 0) b.path_tot[gp] = make_uint2(tot.x, tot.y * alpha_rows(it));
        }
    }
}

template <bool EMIT, int THREADS, typename Lds>
__device__ __forceinline__ void bin_group_item(const BatchDev &b, Lds &lds, uint32_t item) {
    const BinItem it = b.bin_items[b.n_bin_wave + item];
    if (b.n_big && is_big(it, b.scenes[it.k])) return;  // uniform over the block
    bin_group<EMIT, THREADS>(b, it, lds.cnt, lds.delta, lds.col, lds.queue[0], BIN_GROUP_TILES, BIN_GROUP_COLS);
}

// The big paths, listed by k_bin_items, a block of 1024 threads each with the LDS that the batch's largest
// takes (max_tiles, max_cols).  Through global atomics, a 2048^2 scene of 400 paths with 50 whole-canvas rects
// (16 384 tiles each) took 80 us to count and 50 to emit; now 22 + 18 and 24 + 20.
template <bool EMIT>
__global__ __launch_bounds__(1024) void k_bin_big(BatchDev b, uint32_t max_tiles, uint32_t max_cols) {
    extern __shared__ uint32_t big_lds[];
    uint32_t *const cnt = big_lds, *const delta = cnt + max_tiles;
    uint32_t *const queue = delta + (EMIT ? 0u : (max_tiles + 1) / 2);
    int32_t *const col = reinterpret_cast<int32_t *>(queue + (1024 / 64) * WALK_QUEUE);
    const uint32_t n = b.counters[C_BIG];
    for (uint32_t i = blockIdx.x; i < n; i += gridDim.x) {  // uniform over the block
        const BinItem it = b.bin_items[b.big_list[i]];
        bin_group<EMIT, 1024>(b, it, cnt, delta, col, queue, max_tiles, max_cols);
        __syncthreads();
    }
}

// Both classes in one launch, the group class's paths first (they last longest).  512 threads: a long
// path's walk is twice as wide as with 256, and 8 wave-class slices (40 KB in the count pass) leave the
// wave class its 32 waves per CU (which the compiler is held to: 83 -> 80 us at 4096^2 against 7 a SIMD).
template <bool EMIT>
__global__ __launch_bounds__(512, 8) void k_bin(BatchDev b) {
    __shared__ BinLds<EMIT, 512> lds;
    if (blockIdx.x < b.n_bin_group) {  // uniform over the block
        bin_group_item<EMIT, 512>(b, lds.g, blockIdx.x);
    } else {
        const uint32_t wave = (blockIdx.x - b.n_bin_group) * 8 + (threadIdx.x >> 6);
        bin_wave<EMIT, 512>(b, lds.w, __builtin_amdgcn_readfirstlane(wave));  // uniform: scalar loads
    }
}

// A class per launch, in blocks of 256: a block's LDS is held by its slowest wave, so with the chip full
// the smaller blocks keep more waves in flight.
template <bool EMIT>
__global__ __launch_bounds__(256) void k_bin_wave(BatchDev b) {
    __shared__ BinSlice<EMIT> lds[4];
    bin_wave<EMIT, 256>(b, lds, __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6)));
}
template <bool EMIT>
__global__ __launch_bounds__(256) void k_bin_group(BatchDev b) {
    __shared__ BinPath<EMIT, 256> lds;
    bin_group_item<EMIT, 256>(b, lds, blockIdx.x);
}

// Item s of a tile sits at LDS word s + s / 16: striped rows (lane-consecutive) and blocked
// runs (16 per thread, threads 17 words apart) are both bank-conflict free.
__device__ __forceinline__ uint32_t scan_pad(uint32_t s) { return s + (s >> 4); }

// A tile's state word: 0 nothing yet, SCAN_SUM | its total, SCAN_PREFIX | the total up to its end.
// Flag and value are one word, so a reader needs no ordering between two.
constexpr unsigned long long SCAN_SUM = 1ull << 32, SCAN_PREFIX = 2ull << 32;
template <typename T> constexpr int SCAN_WORDS = sizeof(T) / 4;  // state words per tile
__device__ __forceinline__ uint32_t scan_part(uint32_t v, int) { return v; }
__device__ __forceinline__ uint32_t scan_part(const U2 &v, int i) { return i ? v.y : v.x; }
__device__ __forceinline__ void scan_set(uint32_t &v, int, uint32_t x) { v = x; }
__device__ __forceinline__ void scan_set(U2 &v, int i, uint32_t x) { (i ? v.y : v.x) = x; }

// Sum of the tiles before tile t (> 0), by one wave, which publishes its own total first and the
// total up to its end afterwards: 64 predecessors at a time are read from the nearest back to the
// nearest one that knows its prefix.  Tile numbers are handed out in the order workgroups start
// (k_scan's ticket), so every predecessor has started and none waits for a later one: its words
// arrive.  Components are looked up one after the other.
template <typename T>
__device__ T scan_look_back(unsigned long long *state, uint32_t t, T total) {
    constexpr int W = SCAN_WORDS<T>;
    const uint32_t lane = threadIdx.x & 63;
    if (lane < (uint32_t)W)
        __hip_atomic_store(&state[(uint64_t)t * W + lane], SCAN_SUM | scan_part(total, (int)lane), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    T before{};
#pragma unroll
    for (int c = 0; c < W; c++) {
        uint32_t sum = 0;
        for (int64_t at = (int64_t)t - 1; at >= 0; at -= 64) {  // wave-uniform
            const int64_t i = at - (int64_t)lane;
            unsigned long long w;
            uint64_t known, missing;
            do {
                // before the first tile lies a prefix of 0
                w = i < 0 ? SCAN_PREFIX
                          : __hip_atomic_load(&state[(uint64_t)i * W + c], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                known = __ballot((w & SCAN_PREFIX) != 0);
                missing = __ballot(w == 0);
                if (known) missing &= (known & (0ull - known)) - 1;  // only those nearer than the first prefix matter
            } while (missing);
            const uint64_t use = known ? (known ^ (known - 1)) : ~0ull;  // up to and with the first prefix
            sum += __builtin_amdgcn_readlane(wave_inclusive_sum((use >> lane) & 1ull ? (uint32_t)w : 0u), 63);
            if (known) break;
        }
        scan_set(before, c, sum);
    }
    if (lane < (uint32_t)W)
        __hip_atomic_store(&state[(uint64_t)t * W + lane],
                           SCAN_PREFIX | (scan_part(before, (int)lane) + scan_part(total, (int)lane)), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    return before;
}

// Exclusive scan of n items in one launch of nb tiles of SCAN_TILE items (the store functor also gets
// the total, as item n).  state: a ticket word and SCAN_WORDS words a tile, zeroed before; not used
// with one tile.  Loads and stores are striped (one coalesced row of 256 items at a time) and
// transposed through LDS to the blocked order the per-thread running sum needs.
// Latency-bound: with three launches each (tile sums, their scan, the items) a pass's five scans took
// 61 us on the 512^2 cubic scene, now 29; 79 on the 4096^2 scene, now 48; 89 on the 48-scene
// batch, now 69 (its 4.4 M segments scanned per flattener chunk instead of per segment).
template <typename T, typename Load, typename Store>
__global__ __launch_bounds__(SCAN_THREADS) void k_scan(Load ld, Store st, uint32_t n, uint32_t nb,
                                                       unsigned long long *state) {
    __shared__ T tile[SCAN_TILE + SCAN_TILE / 16];
    __shared__ uint32_t s_ticket;
    __shared__ T s_before;
    const uint32_t tid = threadIdx.x;
    uint32_t t = 0;
    if (nb > 1) {
        if (tid == 0) s_ticket = (uint32_t)atomicAdd(state, 1ull);
        __syncthreads();
        t = s_ticket;
    }
    const uint64_t base = (uint64_t)t * SCAN_TILE;
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; i++) {
        const uint32_t si = (uint32_t)i * SCAN_THREADS + tid;
        const uint64_t j = base + si;
        tile[scan_pad(si)] = j < n ? ld((uint32_t)j) : zero_of<T>();
    }
    __syncthreads();
    T vals[SCAN_ITEMS];
    T s = zero_of<T>();
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; i++) {
        vals[i] = tile[scan_pad(tid * SCAN_ITEMS + (uint32_t)i)];
        s = s + vals[i];
    }
    T total;
    T run = block_exclusive_scan<T>(s, total);  // its barriers order the reads above
    T before = zero_of<T>();
    if (nb > 1) {
        if (tid < 64) {
            const T bf = scan_look_back<T>(state + 1, t, total);
            if (tid == 0) s_before = bf;
        }
        __syncthreads();
        before = s_before;
        run = run + before;
    }
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; i++) {
        tile[scan_pad(tid * SCAN_ITEMS + (uint32_t)i)] = run;
        run = run + vals[i];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; i++) {
        const uint32_t si = (uint32_t)i * SCAN_THREADS + tid;
        const uint64_t j = base + si;
        if (j < n) st((uint32_t)j, tile[scan_pad(si)]);
    }
    if (t == nb - 1 && tid == 0) st(n, before + total);
}

// Scan functors --------------------------------------------------------------

struct LoadU32 {
    const uint32_t *p;
    __device__ uint32_t operator()(uint32_t i) const { return p[i]; }
};
struct StoreU32 {
    uint32_t *p;
    __device__ void operator()(uint32_t i, uint32_t v) const { p[i] = v; }
};
// Tiles: (fill count, has fills) -> fill offsets, alpha indices; totals -> counters.
struct LoadPathTot {
    const uint2 *tot;
    __device__ U2 operator()(uint32_t i) const {
        const uint2 v = tot[i];
        return U2{v.x, v.y};
    }
};
struct StorePathOff {
    uint2 *off;
    uint32_t *fill_end, *alpha_end, *counters;
    uint32_t n;
    __device__ void operator()(uint32_t i, U2 v) const {
        off[i] = make_uint2(v.x, v.y);
        if (i == n) {
            *fill_end = v.x;
            *alpha_end = v.y;
            counters[C_FILLS] = v.x;
            counters[C_ALPHA] = v.y;
        }
    }
};
struct LoadU32Counted {
    const uint32_t *p;
    const uint32_t *n_ptr;
    __device__ uint32_t operator()(uint32_t i) const { return i < *n_ptr ? p[i] : 0u; }
};
struct StoreChunkOff {
    uint32_t *off, *total, *counters;
    uint32_t n;
    __device__ void operator()(uint32_t i, uint32_t v) const {
        off[i] = v;
        if (i == n) {
            *total = v;
            counters[C_LINES] = v;
        }
    }
};
struct StoreEntryOff {
    uint2 *off;
    uint32_t *counters;
    uint32_t n;
    __device__ void operator()(uint32_t i, U2 v) const {
        off[i] = make_uint2(v.x, v.y);
        if (i == n) {
            counters[C_ENTRIES] = v.x;
            counters[C_ALPHA_ENTRIES] = v.y;
        }
    }
};

// ---------------------------------------------------------------------------
// Backdrop propagation down each path column (tiler.cpp:369-439) + z-buffer, for clip paths and what they
// clip (else the count pass does it: resolve_columns)
// ---------------------------------------------------------------------------

// Where a tile of a path column lands in its scene's framebuffer-tile grid.
struct ColumnWalk {
    uint32_t p, rgba, rule, tbase, clip, level;
    bool own_rules;  // clip coverage under each clip path's own fill rule (PFH_CLIP_RULE_OWN)
    int rx, ry;  // the path's rect origin (tiles)
    int w, h, x, fb_row0;  // fb_row0: fb tile index (scene-local) of row 0
    uint32_t fb_base, fb_w;
    // column x of a binned path
    __device__ ColumnWalk(const BatchDev &b, const BinItem &it, uint32_t column) {
        const SceneDev &sc = b.scenes[it.k];
        const int4 r = it.rect;
        p = it.p;
        w = r.z - r.x;
        h = r.w - r.y;
        x = (int)column;
        tbase = it.tbase;
        rgba = it.rgba;
        rule = it.rule & 1u;
        own_rules = (it.rule & RULE_CLIP_OWN) != 0;
        clip = it.clip;
        level = it.level;
        rx = r.x;
        ry = r.y;
        fb_base = sc.fb_base;
        fb_w = (uint32_t)sc.fb_w;
        fb_row0 = (r.y - sc.fb_y0) * sc.fb_w + (r.x + x - sc.fb_x0);
    }
    __device__ uint32_t tile(int row) const { return tbase + (uint32_t)(row * w + x); }
    __device__ uint32_t fb_local(int row) const { return (uint32_t)(fb_row0 + row * (int)fb_w); }
};

// A clip path's tile at given tile coordinates, as resolved by the propagate phase of its clip
// level (an earlier launch): whether it has a coverage mask (its own, or one taken from its own
// clip), whether it covers without one (solid), its backdrop, and its coverage source (the mask
// row whose record holds the chain).
struct ClipTile {
    bool inside, alpha, solid;
    int8_t bd;
    uint32_t src;
};
__device__ __forceinline__ ClipTile clip_tile_at(const BatchDev &b, const BinItem &ci, int tx, int ty) {
    ClipTile r{false, false, false, 0, 0};
    const int4 cr = ci.rect;
    if (tx < cr.x || tx >= cr.z || ty < cr.y || ty >= cr.w) return r;
    const uint32_t ct = ci.tbase + (uint32_t)((ty - cr.y) * (cr.z - cr.x) + (tx - cr.x));
    const uint8_t st = b.tile_st[ct];
    r.inside = true;
    r.alpha = st == TILE_ALPHA || st == TILE_CLIP_MASK;
    r.solid = st == TILE_SOLID;
    r.bd = b.tile_bd[ct];
    r.src = r.alpha ? b.tile_clip_ai[ct] : 0u;
    return r;
}

// What a tile of a path column reads of its clip path: the clip's tile at the same coordinates
// and, for a clip path's tile over a clip mask, the chain record of that mask.  Both were written
// by an earlier propagate phase, so a column loads them for a group of rows before it stores
// anything (no load waits behind a store it might alias).
struct ClipRead {
    ClipTile ct;
    uint4 pr;
};
template <bool LEVELS>
__device__ __forceinline__ ClipRead clip_read(const BatchDev &b, const ColumnWalk &cw, const BinItem &ci, int row) {
    ClipRead r{{false, false, false, 0, 0}, make_uint4(1u, 0u, 0u, 0u)};
    if (cw.clip < CLIP_EMPTY) r.ct = clip_tile_at(b, ci, cw.rx + cw.x, cw.ry + row);
    if (LEVELS && r.ct.alpha && r.ct.src < b.cap_alpha) r.pr = b.clip_rec[r.ct.src];
    return r;
}

// One tile of a path column, its propagated backdrop bd and its fill range [f0, f1) known (ai: its
// mask row when it has fills), with what it reads of its clip path.  LEVELS: the path is a clip path.
// job: the mask combination it asks for, if any.
template <bool LEVELS>
__device__ __forceinline__ void propagate_tile(const BatchDev &b, const ColumnWalk &cw, const ClipRead &cr, int row,
                                               int8_t bd, uint32_t f0, uint32_t f1, uint32_t ai, uint2 &job) {
    const bool clipped = cw.clip < CLIP_EMPTY || cw.clip == CLIP_EMPTY;
    const bool opaque = (cw.rgba >> 24) == 255u;
    const uint32_t t = cw.tile(row);
    const bool alpha = f1 > f0;
    const ClipTile &ct = cr.ct;
    // Whether the tile covers without fills: backdrop != 0, except under the path's own even-odd
    // rule with an even backdrop where clip paths' own rules are taken (PFH_CLIP_RULE_OWN); the
    // reference's clip resolution tests backdrop != 0 alone (tiler.cpp:396-431).
    const bool covers = bd != 0 && !(cw.own_rules && cw.rule && (bd & 1) == 0);
    const uint32_t job_rules = cw.own_rules ? CLIP_JOB_OWN_RULES : 0u;
    if (LEVELS) {
        // A clip path draws nothing itself.  Its fills make two mask rows (ai, ai + 1) that
        // keep |sum + backdrop| under the nonzero and the even-odd rule (under its own rule,
        // both, where clip paths' own rules are taken), for the tiles that take them over; its
        // coverage at the tile is that value, min'd with its own clip's where it is nested and
        // both have masks (a combine job rewrites both rows).
        const bool own = alpha && ai + 1 < b.cap_alpha;
        if (own) {
            const uint32_t r0 = cw.own_rules ? cw.rule : 0u, r1 = cw.own_rules ? cw.rule : 1u;
            b.alpha_rec[ai] = make_uint4(f0, f1, (uint32_t)(uint8_t)bd | (r0 << 8), t);
            b.alpha_rec[ai + 1] = make_uint4(f0, f1, (uint32_t)(uint8_t)bd | (r1 << 8), t);
        }
        uint8_t st = alpha ? TILE_ALPHA : (covers ? TILE_SOLID : TILE_EMPTY);
        int8_t out_bd = bd;
        uint32_t src = ai;
        uint4 rec = make_uint4(1u, 0u, 0u, 0u);  // the chain: this row alone
        if (clipped) {
            if (!ct.inside || (!ct.alpha && !ct.solid)) {
                st = TILE_EMPTY;
                out_bd = 0;
            } else if (ct.alpha && alpha) {
                out_bd = 0;
                const uint4 pr = cr.pr;
                rec = make_uint4(1u + min(pr.x, MAX_CLIP_LEVELS - 1u), ct.src, pr.y, pr.z);
                job = make_uint2(ai | CLIP_JOB_CLIP | job_rules, ai);
            } else if (ct.alpha && covers) {
                st = TILE_CLIP_MASK;  // its own clip's coverage, unchanged
                out_bd = ct.bd;
                src = ct.src;
            }
        }
        if (st == TILE_ALPHA && own) b.clip_rec[ai] = rec;
        if (st == TILE_ALPHA || st == TILE_CLIP_MASK) b.tile_clip_ai[t] = src;
        b.tile_st[t] = st;
        b.tile_bd[t] = out_bd;
        return;
    }
    if (clipped) {
        if (alpha && ai < b.cap_alpha)
            b.alpha_rec[ai] = make_uint4(f0, f1, (uint32_t)(uint8_t)bd | (cw.rule << 8), t);
        uint8_t st;
        int8_t out_bd = 0;
        if (!ct.inside || (!ct.alpha && !ct.solid)) {
            st = TILE_EMPTY;  // outside the clip's rect or over a blank clip tile: culled
        } else if (ct.alpha && alpha) {
            // both masks: min(|own + backdrop|, clip coverage) replaces the mask; backdrop 0
            st = TILE_ALPHA;
            job = make_uint2(ai | job_rules, ct.src);
        } else if (ct.alpha && covers) {
            st = TILE_CLIP_MASK;  // solid over a clip mask: the clip's mask and backdrop
            out_bd = ct.bd;
            b.tile_clip_ai[t] = ct.src + cw.rule;
        } else {
            // unchanged: an alpha tile, or a solid tile over a solid clip tile
            const bool even = cw.rule && (bd & 1) == 0;
            st = alpha ? TILE_ALPHA : (bd == 0 ? TILE_EMPTY : (even ? TILE_CLEAR : TILE_SOLID));
            out_bd = bd;
            if (st == TILE_SOLID && opaque) atomicMax(&b.zbuf[cw.fb_base + cw.fb_local(row)], cw.p);
        }
        b.tile_st[t] = st;
        if (b.dump) b.tile_bd[t] = out_bd;
        return;
    }
    const bool even = cw.rule && (bd & 1) == 0;
    b.tile_st[t] = alpha ? TILE_ALPHA : (bd == 0 ? TILE_EMPTY : (even ? TILE_CLEAR : TILE_SOLID));
    if (b.dump) b.tile_bd[t] = bd;
    if (alpha) {
        if (ai < b.cap_alpha) b.alpha_rec[ai] = make_uint4(f0, f1, (uint32_t)(uint8_t)bd | (cw.rule << 8), t);
    } else if (opaque && bd != 0 && !even) {
        atomicMax(&b.zbuf[cw.fb_base + cw.fb_local(row)], cw.p);
    }
}

// Walk down a path's tiles (core/d3d9/tiler.cpp:369-439): backdrops, tile status, alpha
// records, z-buffer, and clip resolution (tiler.cpp:385-431) against the clip path's resolved
// tile at the same coordinates: outside its rect or over a blank tile -> culled; both with masks ->
// a combine job (the tile's backdrop moves into it); a solid tile over a mask -> it takes that
// mask; otherwise unchanged (a solid clip tile passes the tile through).
// A launch per clip level, 1..MAX_CLIP_LEVELS: the clip paths of that level, a clip path nested in
// another being resolved against it like a draw path (the level structure of
// core/d3d11/scene_builder.cpp:92-133, shaders/d3d11/propagate.comp:133-176); then one for the clipped
// draw paths.  Each reads only tiles of earlier launches.
// Columns [xa, xb) of a path, at most PROP_COLS, by a block: a thread per column and stretch of rows; each
// sums its stretch's deltas, starts from the sums of the stretches above it and takes its rows PROP_ROWS
// at a time, every load of a group issued before the first is used.
// Latency-bound (dependent loads per group, a few wide clip rects per level), so the work is strips of
// columns, listed by k_bin_items and dealt to as many blocks as the chip holds, with stretches a few
// groups long.  The 4096^2 scene of 2 500 paths under clips nested 4 deep: with a thread per column, tall
// columns listed for 16 or 64 lanes each in two more launches and every launch over all columns, 156 us in
// 15 launches; with a block per path, 148 in 5; now 62 in 5.
constexpr int PROP_ROWS = 4;
constexpr uint32_t NO_JOB = 0xffffffffu;  // not a mask row with its flags
constexpr int PROP_THREADS = 512;

template <bool LEVELS>
__device__ __forceinline__ void propagate_strip(const BatchDev &b, const BinItem &it, uint32_t xa, int32_t *part) {
    const uint32_t t = threadIdx.x;
    const uint32_t tw = (uint32_t)max(it.rect.z - it.rect.x, 0), cols = min(PROP_COLS, tw - xa);
    const int th = max(it.rect.w - it.rect.y, 0);
    const uint32_t bits = cols > 1 ? 32u - (uint32_t)__clz((int)(cols - 1)) : 0u;
    const int parts = max(min(PROP_THREADS >> bits, th), 1);
    const int rows = (th + parts - 1) / parts;
    const int p = (int)(t >> bits);
    const uint32_t x = t & ((1u << bits) - 1u);  // from xa
    const int ra = min(p * rows, th), rb = min(ra + rows, th);
    const int32_t start = x < cols ? b.col_bd[it.cbase + xa + x] : 0;  // before a stretch stores its column's sum
    int32_t sum = 0;
    if (x < cols) {
        for (int r0 = ra; r0 < rb; r0 += 8) {
            int32_t d[8];
#pragma unroll
            for (int i = 0; i < 8; i++)
                d[i] = r0 + i < rb ? b.tile_delta[it.tbase + (uint32_t)(r0 + i) * tw + xa + x] : 0;
#pragma unroll
            for (int i = 0; i < 8; i++) sum += (int8_t)d[i];
        }
    }
    part[t] = sum;
    __syncthreads();
    if (p < parts && x < cols) {
        BinItem ci;
        if (it.clip < CLIP_EMPTY) ci = b.bin_items[it.clip];
        const ColumnWalk cw(b, it, xa + x);
        int32_t running = start;
        for (int q = 0; q < p; q++) running += part[((uint32_t)q << bits) + x];
        for (int row0 = ra; row0 < rb; row0 += PROP_ROWS) {
            int32_t delta[PROP_ROWS];
            uint32_t f0[PROP_ROWS], f1[PROP_ROWS], ai[PROP_ROWS];
            ClipRead cr[PROP_ROWS];
#pragma unroll
            for (int i = 0; i < PROP_ROWS; i++) {
                delta[i] = 0;
                f0[i] = f1[i] = ai[i] = 0;
                cr[i] = ClipRead{{false, false, false, 0, 0}, make_uint4(1u, 0u, 0u, 0u)};
                if (row0 + i < rb) {
                    const uint32_t tile = cw.tile(row0 + i);
                    delta[i] = b.tile_delta[tile];
                    f0[i] = b.tile_fill_off[tile];
                    f1[i] = b.tile_fill_off[tile + 1];
                    ai[i] = b.tile_alpha_idx[tile];
                    cr[i] = clip_read<LEVELS>(b, cw, ci, row0 + i);
                }
            }
            uint2 job[PROP_ROWS];
            uint32_t n_jobs = 0, at[PROP_ROWS];
#pragma unroll
            for (int i = 0; i < PROP_ROWS; i++) {
                job[i] = make_uint2(NO_JOB, 0u);
                if (row0 + i < rb) {
                    propagate_tile<LEVELS>(b, cw, cr[i], row0 + i, (int8_t)running, f0[i], f1[i], ai[i], job[i]);
                    running += (int8_t)delta[i];
                }
                const uint64_t m = __ballot(job[i].x != NO_JOB);
                at[i] = n_jobs + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
                n_jobs += (uint32_t)__popcll(m);
            }
            if (n_jobs == 0) continue;  // of the wave's active lanes: uniform
            // one add for the wave's rows: the counter takes one every 4-5 ns
            uint32_t first = 0;
            if ((threadIdx.x & 63) == (uint32_t)__builtin_ctzll(__ballot(true)))
                first = atomicAdd(&b.counters[C_CLIP_JOBS], n_jobs);
            first = __builtin_amdgcn_readfirstlane(first);
#pragma unroll
            for (int i = 0; i < PROP_ROWS; i++)
                if (job[i].x != NO_JOB && first + at[i] < b.cap_alpha) b.clip_jobs[first + at[i]] = job[i];
        }
        if (b.dump && rb == th && (ra < th || th == 0)) b.col_bd[it.cbase + xa + x] = running;  // the column's last rows
    }
    __syncthreads();  // the next strip rewrites part
}

// LEVELS: the strips of the clip paths of a level, else those of the clipped draw paths.
template <bool LEVELS>
__global__ __launch_bounds__(PROP_THREADS) void k_propagate(BatchDev b, uint32_t level) {
    __shared__ int32_t part[PROP_THREADS];
    const uint32_t n = b.counters[LEVELS ? C_CLIP_STRIPS : C_DRAW_STRIPS];
    for (uint32_t i = blockIdx.x; i < n; i += gridDim.x) {  // uniform over the block
        const uint2 st = b.prop_strips[LEVELS ? i : b.cap_strips - 1 - i];
        const BinItem it = b.bin_items[st.x];
        if (!LEVELS || it.level == level) propagate_strip<LEVELS>(b, it, st.y, part);
    }
}

// Draw entries: tiles with a mask or a nonzero backdrop that survive the z-cull
// (core/d3d9/scene_builder.cpp:57-79, shaders/d3d9/tile.vert:103-118), per path like the
// bin kernels (a wave per small rect, a block per large one) with the threads striding over
// the rect's tiles in row-major order.  The count pass stores each path's entry count;
// after their scan the write pass numbers the path's entries in row-major order by ballot
// rank, so consecutive threads write consecutive entries.  Entries of a path precede those
// of the next, which is all the sort by framebuffer tile needs to keep draw order: a path
// has at most one tile per framebuffer tile.

struct EntryTile {
    bool keep;
    uint32_t st, fbl, ai;  // ai: the alpha index of an alpha tile (write pass)
};

// e: the entry's index; ea: its index among alpha entries (for an alpha tile).  The alpha
// entries' tiles are listed in that order for the fill kernel, which rasterizes only them.
// With clip paths, the solid tiles of several draw paths can take one clip mask row: the first
// entry to list it claims it in clip_seen, the others list nothing (NO_ALPHA: the fill kernel
// skips the slot), so the row is rasterized once.
template <bool CLIPS>
__device__ __forceinline__ void write_entry(const BatchDev &b, const SceneDev &sc, uint32_t p, uint32_t rgba,
                                            uint32_t paint, uint32_t tbase, uint32_t j, const EntryTile &et,
                                            uint32_t e, uint32_t ea) {
    if (e >= b.cap_entries) return;  // past the capacity: the batch is retried
    const uint32_t ai = (et.st == TILE_ALPHA || et.st == TILE_CLIP_MASK) ? et.ai : NO_ALPHA;
    if (ai != NO_ALPHA && ea < b.cap_vis) {
        uint32_t listed = ai;
        if (CLIPS && et.st == TILE_CLIP_MASK && ai < b.cap_alpha) {
            const uint32_t bit = 1u << (ai & 31u);
            if (atomicOr(&b.clip_seen[ai >> 5], bit) & bit) {
                listed = NO_ALPHA;
                atomicAdd(&b.counters[C_CLIP_DUPS], 1u);
            }
        }
        b.alpha_vis[ea] = listed;
    }
    // even-odd solid tile with an even winding covers nothing: zero alpha
    uint32_t rx = ai, ry = et.st == TILE_CLEAR ? (rgba & 0x00ffffffu) : rgba;
    // a path with a paint record: flagged, its mask row (or none) and its paint; a tile that covers
    // nothing stays a transparent solid entry, unless its paint composites through an op (which
    // sets the alpha of every pixel of the tile, shaders/d3d9/tile.frag:585-598)
    if (paint != PAINT_NONE) {
        if (et.st != TILE_CLEAR) {
            rx = ENTRY_GRADIENT | (ai == NO_ALPHA ? ENTRY_ROW_NONE : min(ai, ENTRY_ROW_EMPTY - 1u));
            ry = paint;
        } else if (sc.paints[paint].op != 0) {
            rx = ENTRY_GRADIENT | ENTRY_ROW_EMPTY;
            ry = paint;
        } else {
            rx = NO_ALPHA;
            ry = 0u;
        }
    }
    b.keys[e] = sc.fb_base + et.fbl;
    b.entry_rec[e] = make_uint2(rx, ry);
    if (b.dump) b.entry_meta[e] = make_uint2(p, et.fbl);
}

// One wave over the tiles [j0, j1) of a path's rect, row-major.  Count pass: returns the
// range's {entries, alpha entries}.  Write pass: numbers them from `first` (entry, alpha entry)
// by ballot rank.
template <bool WRITE, bool CLIPS>
__device__ __forceinline__ uint2 range_entries(const BatchDev &b, const SceneDev &sc, const BinItem &it, uint32_t j0,
                                               uint32_t j1, uint2 first) {
    const uint32_t lane = threadIdx.x & 63;
    const uint64_t lt_mask = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    const uint32_t p = it.p;
    const int4 r = it.rect;
    const int w = max(r.z - r.x, 0);
    const uint32_t tbase = it.tbase;
    const int fb_row0 = (r.y - sc.fb_y0) * sc.fb_w + (r.x - sc.fb_x0);
    const uint32_t rgba = it.rgba;
    const float inv_w = w > 0 ? 1.0f / (float)w : 0.0f;
    uint32_t e = first.x, n_alpha = first.y;
    // tile j's status, its framebuffer tile and that tile's z, loaded one chunk ahead; row = j / w
    // from a float estimate (off by at most one below 2^24 tiles), then corrected
    auto fetch = [&](uint32_t j, uint32_t &st, uint32_t &z, uint32_t &fbl) {
        st = TILE_EMPTY;
        z = 0;
        fbl = 0;
        if (j < j1) {
            uint32_t row = (uint32_t)((float)j * inv_w);
            if (row * (uint32_t)w > j) row--;
            else if ((row + 1) * (uint32_t)w <= j) row++;
            const uint32_t x = j - row * (uint32_t)w;
            fbl = (uint32_t)(fb_row0 + (int)row * sc.fb_w + (int)x);
            st = b.tile_st[tbase + j];
            z = b.zbuf[sc.fb_base + fbl];
        }
    };
    uint32_t n_st, n_z, n_fbl;
    fetch(j0 + lane, n_st, n_z, n_fbl);
    // write pass: a chunk's alpha indices are loaded at the end of the chunk before it
    auto alpha_of = [&](uint32_t st, uint32_t j) {
        if (!CLIPS) return st == TILE_ALPHA ? b.tile_alpha_idx[tbase + j] : NO_ALPHA;
        return st == TILE_ALPHA ? b.tile_alpha_idx[tbase + j] : (st == TILE_CLIP_MASK ? b.tile_clip_ai[tbase + j] : NO_ALPHA);
    };
    uint32_t n_ai = WRITE ? alpha_of(n_st, j0 + lane) : NO_ALPHA;
    for (uint32_t jc = j0; jc < j1; jc += 64) {  // uniform over the wave
        const uint32_t j = jc + lane;
        EntryTile et;
        et.st = n_st;
        et.fbl = n_fbl;
        et.ai = n_ai;
        et.keep = n_st != TILE_EMPTY && (int32_t)p >= (int32_t)n_z;
        fetch(jc + 64 + lane, n_st, n_z, n_fbl);
        const uint64_t m = __ballot(et.keep);
        const uint64_t ma = __ballot(et.keep && (et.st == TILE_ALPHA || (CLIPS && et.st == TILE_CLIP_MASK)));
        if (WRITE && et.keep)
            write_entry<CLIPS>(b, sc, p, rgba, it.paint, tbase, j, et, e + (uint32_t)__popcll(m & lt_mask),
                        n_alpha + (uint32_t)__popcll(ma & lt_mask));
        e += (uint32_t)__popcll(m);
        n_alpha += (uint32_t)__popcll(ma);
        if (WRITE) n_ai = alpha_of(n_st, jc + 64 + lane);
    }
    return make_uint2(e, n_alpha);
}

// One launch for both binning classes, the group class's blocks first.  A block per large path: wave w
// takes the w-th part of the rect's tiles (row-major, in whole 64-tile chunks), so the waves need no
// barrier.  The count pass keeps each part's counts (ent_part) beside the path's total; the
// write pass starts each wave after the parts before it.  Behind them a wave per small path.
// A clip path draws nothing: no entries.
// A wave takes its part's chunks one after the other, so few paths take blocks of 16 waves and many 4 (the
// launch's choice, WAVES): 400 paths, 50 of them of 16 384 tiles, 22 + 32 us with 4 waves, 8 + 15 with 16;
// 48 scenes with 67 000 paths 74 + 190 with 4, 90 + 251 with 8.
template <bool WRITE, bool CLIPS, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void k_entries(BatchDev b) {
    __shared__ uint2 part[WAVES];
    const uint32_t wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (blockIdx.x >= b.n_bin_group) {  // uniform over the block
        const uint32_t item = __builtin_amdgcn_readfirstlane((blockIdx.x - b.n_bin_group) * WAVES + wv);  // uniform
        if (item >= b.n_bin_wave) return;  // whole wave
        const BinItem it = b.bin_items[item];
        const int4 r = it.rect;
        const uint32_t area = CLIPS && it.level != 0 ? 0u : (uint32_t)max(r.z - r.x, 0) * (uint32_t)max(r.w - r.y, 0);
        const uint2 first = WRITE ? b.path_ent[it.gp] : make_uint2(0u, 0u);
        const uint2 n = range_entries<WRITE, CLIPS>(b, b.scenes[it.k], it, 0, area, first);
        if (!WRITE && lane == 0) b.path_ent[it.gp] = n;
        return;
    }
    const uint32_t item = blockIdx.x;
    const BinItem it = b.bin_items[b.n_bin_wave + item];
    const int4 r = it.rect;
    const uint32_t area = CLIPS && it.level != 0 ? 0u : (uint32_t)max(r.z - r.x, 0) * (uint32_t)max(r.w - r.y, 0);
    const uint32_t q = (area + 64 * WAVES - 1) / (64 * WAVES) * 64;  // tiles per part, whole chunks
    const uint32_t j0 = min(wv * q, area), j1 = min(j0 + q, area);
    uint2 first = make_uint2(0u, 0u);
    if (WRITE) {
        first = b.path_ent[it.gp];
        for (uint32_t v = 0; v < wv; v++) {
            const uint2 c = b.ent_part[item * WAVES + v];
            first.x += c.x;
            first.y += c.y;
        }
    }
    const uint2 n = range_entries<WRITE, CLIPS>(b, b.scenes[it.k], it, j0, j1, first);
    if (!WRITE) {
        if (lane == 0) {
            b.ent_part[item * WAVES + wv] = n;
            part[wv] = n;
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            uint2 n_all = part[0];
            for (uint32_t v = 1; v < WAVES; v++) n_all = make_uint2(n_all.x + part[v].x, n_all.y + part[v].y);
            b.path_ent[it.gp] = n_all;
        }
    }
}

// ---------------------------------------------------------------------------
// Draw entries grouped by framebuffer tile, in draw order within a tile
// ---------------------------------------------------------------------------
//
// A scene's entries are contiguous, in draw order, and their keys lie in its own range of framebuffer
// tiles, so each scene is sorted by itself, stably, by scene-local tile.  Two steps: the entries are
// distributed over 256 buckets of consecutive tiles per scene (histogram, its scan, scatter: blocks of
// SORT_TILE entries over the whole chip), then a block per bucket groups its entries by tile and
// writes its tiles' ranges.  The entries' records move along, so that what reads a tile's entries
// reads them in a row.  Where every scene is small (SORT_SMALL), the second step alone does it, a
// block per scene.
// Launch-bound on a single scene: as an LSD radix sort with its block table, a histogram, scan and
// scatter per 8-bit digit and a pass for the ranges (8 launches, 5 for one digit) this took 82 us at
// 4096x4096 with 10^4 paths and 36 us at 256x256; as 4 launches (1) 56 us and 7.
// Bound by the stable ranking (a match per digit bit) and its LDS traffic: 48 scenes of 1024x1024,
// 265 us before, 245 now, which also has the composite read records in a row (391 us, then 357).
// The scatter's loads are all issued before the ranking: 16 us against 21 (48 scenes: 83, 127).

// Scenes of at most 256 framebuffer tiles and this many path tiles are sorted by one block each.
constexpr uint64_t SORT_SMALL = 16384;
// Buckets of this many path tiles on average (a bound of their entries) take blocks of 1024 threads while
// there are at most SORT_WIDE_SCENES scenes.
constexpr uint64_t SORT_WIDE = 4096;
constexpr uint32_t SORT_WIDE_SCENES = 2;
constexpr int SORT_THREADS = 256;
constexpr int SORT_ITEMS = 16;
constexpr int SORT_TILE = SORT_THREADS * SORT_ITEMS;

// Bits of a scene-local tile below its bucket.
__device__ __forceinline__ uint32_t sort_shift(uint32_t n_fb) {
    const uint32_t bits = n_fb > 1 ? 32u - (uint32_t)__clz((int)(n_fb - 1)) : 0u;
    return bits > 8 ? bits - 8 : 0u;
}

// What is sorted: the keys (batch framebuffer tiles) and what goes with them.
struct SortArrays {
    uint32_t *keys;
    uint2 *rec, *meta;  // meta: with dumps only, else null
};

// Blocks of the distribution never straddle scenes: scene k's entries [seg_e[k], seg_e[k + 1]) (clamped
// to the capacity) take blocks [seg_b[k], seg_b[k + 1]), and the histogram is laid out
// [scene][bucket][block of the scene], so that its exclusive scan places every entry inside its scene's
// range, ordered by bucket, then block, then rank.  The histogram pass finds a block's scene by scanning
// the scenes' block counts; its first block leaves them in seg_e and seg_b for the passes after it.
struct SortBlock {
    int k;
    uint32_t lb, nbk, hbase, e0, e1, fb_base, shift;
};
__device__ __forceinline__ void sort_block(const BatchDev &b, const uint32_t *seg_e, const uint32_t *seg_b, int k,
                                           uint32_t e, uint32_t e_next, uint32_t b0, uint32_t b1, SortBlock &sb) {
    sb.k = k;
    sb.lb = blockIdx.x - b0;
    sb.nbk = b1 - b0;
    sb.hbase = 256u * b0;
    sb.e0 = e + sb.lb * SORT_TILE;
    sb.e1 = min(sb.e0 + SORT_TILE, e_next);
    sb.fb_base = b.scenes[k].fb_base;
    sb.shift = sort_shift(b.scenes[k].n_fb);
}

__global__ __launch_bounds__(SORT_THREADS) void k_sort_hist(BatchDev b, uint32_t *seg_e, uint32_t *seg_b, uint32_t *hist) {
    __shared__ uint32_t h[256];
    __shared__ uint32_t s_k, s_e, s_en, s_b0, s_b1;
    const uint32_t tid = threadIdx.x;
    h[tid] = 0;
    if (tid == 0) s_k = 0xffffffffu;
    __syncthreads();
    uint32_t carry = 0;
    for (int k0 = 0; k0 <= b.n_scenes; k0 += SORT_THREADS) {
        const int k = k0 + (int)tid;
        uint32_t e = 0, e_next = 0;
        if (k <= b.n_scenes) {
            const uint32_t total = min(b.counters[C_ENTRIES], b.cap_entries);
            e = k < b.n_scenes ? min(b.path_ent[b.scenes[k].path_base].x, total) : total;
            e_next = k + 1 < b.n_scenes ? min(b.path_ent[b.scenes[k + 1].path_base].x, total) : total;
        }
        const uint32_t nbk = k < b.n_scenes ? (e_next - e + SORT_TILE - 1) / SORT_TILE : 0u;
        uint32_t tot;
        const uint32_t at = carry + block_exclusive_scan<uint32_t>(nbk, tot);
        if (k <= b.n_scenes && blockIdx.x == 0) {
            seg_e[k] = e;
            seg_b[k] = at;
        }
        if (blockIdx.x >= at && blockIdx.x - at < nbk) {
            s_k = (uint32_t)k;
            s_e = e;
            s_en = e_next;
            s_b0 = at;
            s_b1 = at + nbk;
        }
        carry += tot;
    }
    __syncthreads();
    if (s_k == 0xffffffffu) return;  // past the last block: uniform
    SortBlock sb;
    sort_block(b, seg_e, seg_b, (int)s_k, s_e, s_en, s_b0, s_b1, sb);
    // neighbours mostly share a bucket: one add per run of a wave's row, by its first lane
    const uint32_t lane = tid & 63;
#pragma unroll 4
    for (int i = 0; i < SORT_ITEMS; i++) {
        const uint32_t j = sb.e0 + (uint32_t)i * SORT_THREADS + tid;
        const uint32_t d = j < sb.e1 ? (b.keys[j] - sb.fb_base) >> sb.shift : 256u;
        const uint32_t left = __shfl_up(d, 1, 64);  // by every lane
        const bool head = lane == 0 || left != d;
        const uint64_t heads = __ballot(head), above = lane == 63 ? 0ull : heads >> (lane + 1);
        const uint32_t run = above ? 1u + (uint32_t)__builtin_ctzll(above) : 64u - lane;
        if (head && d < 256) atomicAdd(&h[d], run);
    }
    __syncthreads();
    hist[sb.hbase + tid * sb.nbk + sb.lb] = h[tid];
}

// Lanes of a wave's row holding the same digit (multisplit by ballots), among `valid` ones.
template <int BITS>
__device__ __forceinline__ uint64_t digit_peers(uint32_t d, bool valid) {
    uint64_t peers = __ballot(valid);
#pragma unroll
    for (int bit = 0; bit < BITS; bit++) {
        const uint64_t m = __ballot((d >> bit) & 1u);
        peers &= ((d >> bit) & 1u) ? m : ~m;
    }
    return peers;
}

// Distribution over the buckets.  The block's entries are ranked stably by bucket: each wave ranks its
// own contiguous 1024 (16 rows of 64) with wave-local counters, a ballot multisplit giving an entry's
// rank among equal buckets of its row, the counter those of earlier rows; then the waves' counts are
// combined.  Entries come path by path, row-major, and a bucket is a stretch of tiles: neighbouring
// lanes mostly store to neighbouring places, so they store straight from registers (4096^2 scene 26 ->
// 20 us against stores in bucket order through LDS; the 48-scene batch, half of whose canvases have
// buckets of a few tiles, 119 -> 128 of 2900).  offs: the scanned histogram.
__global__ __launch_bounds__(SORT_THREADS) void k_sort_scatter(BatchDev b, SortArrays in, SortArrays out,
                                                               const uint32_t *seg_e, const uint32_t *seg_b,
                                                               const uint32_t *offs) {
    constexpr uint32_t WAVE_ITEMS = SORT_ITEMS * 64;
    __shared__ uint32_t wcnt[SORT_THREADS / 64][256];  // per wave and bucket: counts, then where its first entry goes
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (blockIdx.x >= seg_b[b.n_scenes]) return;  // uniform
    SortBlock sb;
    {
        const int k = find_scene_wave(seg_b, b.n_scenes, blockIdx.x);
        sort_block(b, seg_e, seg_b, k, seg_e[k], seg_e[k + 1], seg_b[k], seg_b[k + 1], sb);
    }
    const uint32_t base = sb.e0, n = sb.e1 - sb.e0;
    const uint32_t place = offs[sb.hbase + tid * sb.nbk + sb.lb];  // of this block's first entry of bucket tid
    for (uint32_t q = tid; q < (SORT_THREADS / 64) * 256; q += SORT_THREADS) (&wcnt[0][0])[q] = 0;
    __syncthreads();
    const uint64_t lt_mask = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    uint32_t *cnt = wcnt[wave];
    uint32_t key[SORT_ITEMS], rank[SORT_ITEMS];
    uint2 rec[SORT_ITEMS];
    const uint32_t w0 = wave * WAVE_ITEMS;
#pragma unroll
    for (int r = 0; r < SORT_ITEMS; r++) {
        const uint32_t li = w0 + (uint32_t)r * 64 + lane;
        key[r] = li < n ? in.keys[base + li] : sb.fb_base;
        if (li < n) rec[r] = in.rec[base + li];
    }
#pragma unroll
    for (int r = 0; r < SORT_ITEMS; r++) {
        const bool valid = w0 + (uint32_t)r * 64 + lane < n;
        const uint32_t d = (key[r] - sb.fb_base) >> sb.shift;
        const uint64_t peers = digit_peers<8>(d, valid);
        const uint32_t rk = (uint32_t)__popcll(peers & lt_mask);
        const uint32_t before = valid ? cnt[d] : 0u;  // entries of bucket d in earlier rows of this wave
        rank[r] = before + rk;
        // the last lane of each group advances the counter (after every lane's read: a wave's LDS
        // operations complete in order)
        if (valid && rk == (uint32_t)__popcll(peers) - 1u) cnt[d] = before + rk + 1u;
    }
    __syncthreads();
    {  // per bucket: after the entries of earlier waves
        uint32_t acc = place;
#pragma unroll
        for (int w = 0; w < SORT_THREADS / 64; w++) {
            const uint32_t c = wcnt[w][tid];
            wcnt[w][tid] = acc;
            acc += c;
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < SORT_ITEMS; r++) {
        const uint32_t li = w0 + (uint32_t)r * 64 + lane;
        if (li < n) {
            const uint32_t g = cnt[(key[r] - sb.fb_base) >> sb.shift] + rank[r];
            out.keys[g] = key[r];
            out.rec[g] = rec[r];
            if (in.meta) out.meta[g] = in.meta[base + li];
        }
    }
}

// A block per bucket (SCENE: per scene, straight from the entry pass): its entries [s0, s1) of `a`
// grouped by tile, stably, and its tiles' ranges.  A digit of 8 bits per pass from the lowest, `passes`
// of them (the same for the whole batch), from a to c and back in turn: a histogram of the bucket
// (where it is more than one chunk), then its entries a chunk at a time, ranked as in the
// distribution and moved through LDS, so that a tile's entries of the chunk are stored together (an
// entry's neighbours belong to other tiles: stored from registers each went to a line of its own).  One
// pass covers 256 tiles, of which a bucket of a canvas up to 4096^2 holds no more: the ranges are the
// digits'.  Above that they are marked at the runs of the sorted keys.
template <int THREADS, bool SCENE>
__global__ __launch_bounds__(THREADS) void k_sort_buckets(BatchDev b, SortArrays a, SortArrays c, const uint32_t *seg_b,
                                                          const uint32_t *offs, uint32_t passes) {
    constexpr int WAVES = THREADS / 64, ITEMS = 8;
    constexpr uint32_t CHUNK = THREADS * ITEMS;
    __shared__ uint32_t hist[256], next[256];   // counts; where the next entry of a digit goes
    __shared__ uint32_t goff[256];              // chunk: that, less the digit's first place in the chunk
    __shared__ uint32_t wcnt[WAVES][256];       // per wave and digit: counts, then places in the chunk
    __shared__ uint2 srec[CHUNK];
    __shared__ uint8_t sdig[CHUNK];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint32_t k = SCENE ? blockIdx.x : blockIdx.x >> 8;
    const SceneDev &sc = b.scenes[k];
    const uint32_t n_fb = sc.n_fb, shift = SCENE ? 8u : sort_shift(n_fb);
    const uint32_t bucket = SCENE ? 0u : blockIdx.x & 255u;
    const uint64_t tile0 = (uint64_t)bucket << shift;
    if (tile0 >= n_fb) return;  // uniform over the block
    const uint32_t tiles = (uint32_t)min((uint64_t)n_fb - tile0, 1ull << shift);
    const uint32_t first = sc.fb_base + (uint32_t)tile0;  // the bucket's first batch tile
    uint32_t s0, s1;
    if (SCENE) {
        const uint32_t total = min(b.counters[C_ENTRIES], b.cap_entries);
        s0 = min(b.path_ent[sc.path_base].x, total);
        s1 = (int)k + 1 < b.n_scenes ? min(b.path_ent[b.scenes[k + 1].path_base].x, total) : total;
    } else {
        const uint32_t nbk = seg_b[k + 1] - seg_b[k], h = 256u * seg_b[k] + bucket * nbk;
        s0 = offs[h];
        s1 = offs[h + nbk];
    }
    if (s0 == s1) {  // uniform
        for (uint32_t t = tid; t < tiles; t += THREADS) b.fb_range[first + t] = make_uint2(s0, s0);
        return;
    }
    const bool one = s1 - s0 <= CHUNK;
    const uint64_t lt_mask = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    for (uint32_t p = 0; p < passes; p++) {
        const SortArrays &in = (p & 1u) ? c : a, &out = (p & 1u) ? a : c;
        const bool ranges = passes == 1;
        uint32_t total;
        if (!one) {
            if (tid < 256) hist[tid] = 0;
            __syncthreads();
            for (uint32_t j = s0 + tid; j < s1; j += THREADS) atomicAdd(&hist[((in.keys[j] - first) >> (8 * p)) & 255u], 1u);
            __syncthreads();
            const uint32_t n = tid < 256 ? hist[tid] : 0u;
            const uint32_t start = s0 + block_exclusive_scan<uint32_t, THREADS>(n, total);
            if (tid < 256) next[tid] = start;
            if (ranges && tid < tiles) b.fb_range[first + tid] = make_uint2(start, start + n);
        }
        for (uint32_t at = s0; at < s1; at += CHUNK) {  // uniform over the block
            for (uint32_t q = tid; q < WAVES * 256; q += THREADS) (&wcnt[0][0])[q] = 0;
            __syncthreads();
            uint32_t *cnt = wcnt[wave];
            uint32_t key[ITEMS], rank[ITEMS];
            uint2 rec[ITEMS];
            const uint32_t w0 = at + wave * (64 * ITEMS);
#pragma unroll
            for (int r = 0; r < ITEMS; r++) {
                const uint32_t j = w0 + (uint32_t)r * 64 + lane;
                key[r] = j < s1 ? in.keys[j] : first;
                if (j < s1) rec[r] = in.rec[j];
            }
#pragma unroll
            for (int r = 0; r < ITEMS; r++) {
                if (w0 + (uint32_t)r * 64 >= s1) break;  // wave-uniform
                const bool valid = w0 + (uint32_t)r * 64 + lane < s1;
                const uint32_t d = ((key[r] - first) >> (8 * p)) & 255u;
                const uint64_t peers = digit_peers<8>(d, valid);
                const uint32_t rk = (uint32_t)__popcll(peers & lt_mask);
                const uint32_t before = valid ? cnt[d] : 0u;
                rank[r] = before + rk;
                if (valid && rk == (uint32_t)__popcll(peers) - 1u) cnt[d] = before + rk + 1u;
            }
            __syncthreads();
            uint32_t n = 0;  // the chunk's entries of digit tid
            if (tid < 256) {
#pragma unroll
                for (int w = 0; w < WAVES; w++) {
                    const uint32_t m = wcnt[w][tid];
                    wcnt[w][tid] = n;
                    n += m;
                }
            }
            const uint32_t local = block_exclusive_scan<uint32_t, THREADS>(n, total);
            if (tid < 256) {
#pragma unroll
                for (int w = 0; w < WAVES; w++) wcnt[w][tid] += local;
                const uint32_t to = one ? s0 + local : next[tid];
                goff[tid] = to - local;
                next[tid] = to + n;
                if (one && ranges && tid < tiles) b.fb_range[first + tid] = make_uint2(to, to + n);
            }
            __syncthreads();
#pragma unroll
            for (int r = 0; r < ITEMS; r++) {
                const uint32_t j = w0 + (uint32_t)r * 64 + lane;
                if (j < s1) {
                    const uint32_t d = ((key[r] - first) >> (8 * p)) & 255u, i = cnt[d] + rank[r];
                    srec[i] = rec[r];
                    sdig[i] = (uint8_t)d;
                    if (!ranges) out.keys[goff[d] + i] = key[r];
                    if (in.meta) out.meta[goff[d] + i] = in.meta[j];
                }
            }
            __syncthreads();
            for (uint32_t i = tid; i < min(CHUNK, s1 - at); i += THREADS) out.rec[goff[sdig[i]] + i] = srec[i];
            __syncthreads();  // the next chunk, or pass, reads and rewrites
        }
    }
    if (passes > 1) {
        const uint32_t *keys = (passes & 1u) ? c.keys : a.keys;
        for (uint32_t t = tid; t < tiles; t += THREADS) b.fb_range[first + t] = make_uint2(s0, s0);
        __syncthreads();
        for (uint32_t j = s0 + tid; j < s1; j += THREADS) {
            const uint32_t key = keys[j];
            if (j == s0 || keys[j - 1] != key) b.fb_range[key].x = j;
            if (j + 1 == s1 || keys[j + 1] != key) b.fb_range[key].y = j + 1;
        }
    }
}

// ---------------------------------------------------------------------------
// Launch helpers (host side)
// ---------------------------------------------------------------------------

static inline uint32_t blocks_for(uint64_t n, uint32_t per) { return (uint32_t)((n + per - 1) / per); }

hipError_t launch_zero_spans(const ZeroSpans &z, hipStream_t st) {
    if (z.n < 0 || z.n > ZERO_SPANS) return hipErrorInvalidValue;
    const uint64_t total = z.n ? z.end[z.n - 1] : 0;
    if (total == 0) return hipSuccess;
    uint32_t nb = (uint32_t)std::min<uint64_t>(blocks_for(total, 256), 8192);
    hipLaunchKernelGGL(k_zero_spans, dim3(nb), dim3(256), 0, st, z);
    return hipGetLastError();
}

// 64-bit state words of a scan of n items of `words` 32-bit components each (none for one tile).
uint64_t scan_state_words(uint64_t n, uint32_t words) {
    const uint64_t nb = blocks_for(n, SCAN_TILE);
    return nb > 1 ? 1 + words * nb : 0;
}

template <typename T, typename Load, typename Store>
static hipError_t scan_impl(Load ld, Store st, uint32_t n, unsigned long long *state, hipStream_t s) {
    const uint32_t nb = std::max(1u, blocks_for(n, SCAN_TILE));
    hipLaunchKernelGGL((k_scan<T, Load, Store>), dim3(nb), dim3(SCAN_THREADS), 0, s, ld, st, n, nb, state);
    return hipGetLastError();
}

// Exclusive scan of in[0..n) into out[0..n] (out[n] = total).  in may equal out.
hipError_t scan_u32(const uint32_t *in, uint32_t *out, uint32_t n, unsigned long long *state, hipStream_t s) {
    return scan_impl<uint32_t>(LoadU32{in}, StoreU32{out}, n, state, s);
}

// Exclusive scan in place of the first min(*n_ptr, cap) of cap items, the others taken as 0.
hipError_t scan_counted(uint32_t *inout, const uint32_t *n_ptr, uint32_t cap, unsigned long long *state, hipStream_t s) {
    return scan_impl<uint32_t>(LoadU32Counted{inout, n_ptr}, StoreU32{inout}, cap, state, s);
}

// Exclusive scan of the flattener's chunk totals in place, the batch's total to the counters and
// behind the segments' offsets.
hipError_t scan_chunks(const BatchDev &b, hipStream_t s) {
    const uint32_t n = blocks_for(b.n_segs, b.seg_chunk);
    return scan_impl<uint32_t>(LoadU32{b.chunk_off}, StoreChunkOff{b.chunk_off, b.seg_cnt + b.n_segs, b.counters, n}, n,
                               b.st_seg, s);
}

// Exclusive scan of the per-path {entries, alpha entries} in place, totals to the counters.
hipError_t scan_entries(const BatchDev &b, hipStream_t s) {
    return scan_impl<U2>(LoadPathTot{b.path_ent}, StoreEntryOff{b.path_ent, b.counters, b.n_paths}, b.n_paths,
                         b.st_entries, s);
}

// Exclusive scan of the per-path {fills, alpha tiles} in place (path_tot[P] = totals), with
// the totals also in the counters and at the end of the tile offset arrays.
hipError_t scan_paths(const BatchDev &b, hipStream_t s) {
    return scan_impl<U2>(LoadPathTot{b.path_tot},
                         StorePathOff{b.path_tot, b.tile_fill_off + b.n_tiles, b.tile_alpha_idx + b.n_tiles, b.counters,
                                      b.n_paths},
                         b.n_paths, b.st_paths, s);
}

// chunk: segments a count-pass wave takes (at most 64: b.seg_chunk, an emit-pass wave's, or a multiple)
hipError_t launch_flatten(const BatchDev &b, bool emit, uint32_t chunk, hipStream_t s) {
    if (b.n_segs == 0) return hipSuccess;
    if (b.seg_chunk < 1 || chunk < b.seg_chunk || chunk > 64 || chunk % b.seg_chunk) return hipErrorInvalidValue;
    if (emit)
        hipLaunchKernelGGL(k_flatten_emit, dim3(blocks_for(blocks_for(b.n_segs, b.seg_chunk), 4)), dim3(256), 0, s, b);
    else
        hipLaunchKernelGGL(k_flatten_count, dim3(blocks_for(blocks_for(b.n_segs, chunk), 4)), dim3(256), 0, s, b, chunk);
    return hipGetLastError();
}

// The bin passes run as one launch of 512-thread blocks up to this many (3.5 for each the chip holds at
// once), as a launch per class beyond: launched one after the other, each class's tail leaves most of
// the chip idle, which counts while a launch is a few rounds of blocks.  A pass, one launch / two: 4
// scenes of 2 587 paths 0.362 / 0.407 ms, the stress scene (2 700) 1.025 / 1.044, the 4096^2 scene (10 000 paths,
// about 3 100 blocks) 0.593 / 0.600, 8 scenes (13 754) 0.582 / 0.589; 4 000 stars (4 000 blocks) 0.713 /
// 0.701, the 4096^2 scene with 20 000 paths 0.968 / 0.936, 32 scenes (66 509) 1.805 / 1.716.
constexpr uint32_t BIN_MERGED_BLOCKS = 3584;

hipError_t launch_bin_items(const BatchDev &b, hipStream_t s) {
    const uint32_t wb = blocks_for(b.n_bin_wave, 256), gb = blocks_for(b.n_bin_group, 256);
    if (wb + gb) hipLaunchKernelGGL(k_bin_items, dim3(wb + gb), dim3(256), 0, s, b, wb);
    return hipGetLastError();
}

// LDS of k_bin_big: counts, packed deltas, walk queues and columns.
template <bool EMIT>
static constexpr size_t bin_big_lds(uint32_t tiles, uint32_t cols) {
    return 4 * ((size_t)tiles + (EMIT ? 0 : (tiles + 1) / 2) + (1024 / 64) * WALK_QUEUE + cols);
}

// Lets k_bin_big take the LDS of the largest rect it is given, on the current device.  Before any launch,
// and always to that one size: the attribute belongs to the process, so one set to a batch's own size could
// fall below another thread's between its call and its launch.
hipError_t init_bin_big() {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&k_bin_big<false>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                             (int)bin_big_lds<false>(BIN_BIG_TILES, BIN_BIG_COLS));
    if (e != hipSuccess) return e;
    return hipFuncSetAttribute(reinterpret_cast<const void *>(&k_bin_big<true>), hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)bin_big_lds<true>(BIN_BIG_TILES, BIN_BIG_COLS));
}

template <bool EMIT>
static void launch_bin_t(const BatchDev &b, hipStream_t s) {
    const uint32_t merged = b.n_bin_group + blocks_for(b.n_bin_wave, 8);
    if (merged == 0) return;
    if (b.n_big) {  // first: they last longest
        const uint32_t cols = std::max(b.big_cols, 64u);  // at least what a block's sums take
        hipLaunchKernelGGL(k_bin_big<EMIT>, dim3(std::min<uint32_t>(b.n_big, 1024)), dim3(1024),
                           bin_big_lds<EMIT>(b.big_tiles, cols), s, b, b.big_tiles, cols);
    }
    if (merged <= BIN_MERGED_BLOCKS) {
        hipLaunchKernelGGL(k_bin<EMIT>, dim3(merged), dim3(512), 0, s, b);
        return;
    }
    if (b.n_bin_wave) hipLaunchKernelGGL(k_bin_wave<EMIT>, dim3(blocks_for(b.n_bin_wave, 4)), dim3(256), 0, s, b);
    if (b.n_bin_group) hipLaunchKernelGGL(k_bin_group<EMIT>, dim3(b.n_bin_group), dim3(256), 0, s, b);
}

hipError_t launch_bin(const BatchDev &b, bool emit, hipStream_t s) {
    if (emit) launch_bin_t<true>(b, s);
    else launch_bin_t<false>(b, s);
    return hipGetLastError();
}

hipError_t launch_propagate(const BatchDev &b, hipStream_t s) {
    if (!b.has_clips || b.n_bin_wave + b.n_bin_group == 0) return hipSuccess;
    const dim3 g(std::min<uint32_t>(b.cap_strips, 1024));
    // clip levels from the outermost in, then the draw paths
    for (uint32_t level = 1; level <= std::min(b.clip_levels, MAX_CLIP_LEVELS); level++)
        hipLaunchKernelGGL(k_propagate<true>, g, dim3(PROP_THREADS), 0, s, b, level);
    hipLaunchKernelGGL(k_propagate<false>, g, dim3(PROP_THREADS), 0, s, b, 0u);
    return hipGetLastError();
}

// Waves of a group-class path in the entry passes: 16 up to this many blocks of them, 4 (the two rounds of
// blocks that the chip then holds) beyond.
constexpr uint32_t ENT_WIDE_BLOCKS = 1024;

uint32_t entry_waves(uint32_t n_bin_group, uint32_t n_bin_wave) {
    return n_bin_group + blocks_for(n_bin_wave, 16) <= ENT_WIDE_BLOCKS ? 16 : 4;
}

template <bool WRITE, bool CLIPS>
static void launch_entries_t(const BatchDev &b, hipStream_t s) {
    const uint32_t waves = entry_waves(b.n_bin_group, b.n_bin_wave);
    const dim3 g(b.n_bin_group + blocks_for(b.n_bin_wave, waves));
    if (g.x == 0) return;
    if (waves == 16) hipLaunchKernelGGL((k_entries<WRITE, CLIPS, 16>), g, dim3(1024), 0, s, b);
    else hipLaunchKernelGGL((k_entries<WRITE, CLIPS, 4>), g, dim3(256), 0, s, b);
}

hipError_t launch_entries(const BatchDev &b, bool write, hipStream_t s) {
    if (b.has_clips) {
        if (write) launch_entries_t<true, true>(b, s);
        else launch_entries_t<false, true>(b, s);
    } else {
        if (write) launch_entries_t<true, false>(b, s);
        else launch_entries_t<false, false>(b, s);
    }
    return hipGetLastError();
}

// Blocks of the sort's distribution for a capacity of `cap` entries over `n_scenes` scenes (one partial
// block each).
static uint32_t sort_max_blocks(uint64_t cap, uint32_t n_scenes) { return blocks_for(cap, SORT_TILE) + n_scenes + 1; }

// max_fb, max_tiles: the largest scene's framebuffer tiles and path tiles (a bound of its entries).
static bool sort_small(uint32_t max_fb, uint64_t max_tiles) { return max_fb <= 256 && max_tiles <= SORT_SMALL; }

size_t sort_temp_elems(uint64_t cap, uint32_t n_scenes, uint32_t max_fb, uint64_t max_tiles) {
    return sort_small(max_fb, max_tiles) ? 0 : 2ull * (n_scenes + 1) + 256ull * sort_max_blocks(cap, n_scenes) + 1;
}

// 64-bit state words of the sort's scan.
uint64_t sort_state_words(uint64_t cap, uint32_t n_scenes, uint32_t max_fb, uint64_t max_tiles) {
    return sort_small(max_fb, max_tiles) ? 0 : scan_state_words(256ull * sort_max_blocks(cap, n_scenes), 1);
}

// Sorts the batch's entries; *sorted_alt: their records are in b.rec_alt (else b.entry_rec).
hipError_t sort_entries(const BatchDev &b, uint32_t max_fb, uint64_t max_tiles, uint32_t *tmp, bool *sorted_alt,
                        hipStream_t s) {
    const uint32_t n_sc = (uint32_t)b.n_scenes;
    const SortArrays x{b.keys, b.entry_rec, b.dump ? b.entry_meta : nullptr};
    const SortArrays y{b.keys_alt, b.rec_alt, b.dump ? b.meta_alt : nullptr};
    if (sort_small(max_fb, max_tiles)) {
        *sorted_alt = true;
        hipLaunchKernelGGL((k_sort_buckets<256, true>), dim3(n_sc), dim3(256), 0, s, b, x, y, nullptr, nullptr, 1u);
        return hipGetLastError();
    }
    const uint32_t nb = sort_max_blocks(b.cap_entries, n_sc), nh = 256 * nb;
    uint32_t *seg_e = tmp, *seg_b = tmp + (n_sc + 1), *hist = tmp + 2 * (n_sc + 1);
    hipLaunchKernelGGL(k_sort_hist, dim3(nb), dim3(SORT_THREADS), 0, s, b, seg_e, seg_b, hist);
    // the scan covers the capacity's blocks; entries past this launch's blocks are never read
    hipError_t e = scan_u32(hist, hist, nh, b.st_sort, s);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_sort_scatter, dim3(nb), dim3(SORT_THREADS), 0, s, b, x, y, seg_e, seg_b, hist);
    uint32_t bits = 0;
    while ((1ull << bits) < max_fb) bits++;
    const uint32_t passes = bits > 16 ? (bits - 1) / 8 : 1;  // digits below a bucket's
    *sorted_alt = passes % 2 == 0;
    if (max_tiles / 256 >= SORT_WIDE && n_sc <= SORT_WIDE_SCENES)
        hipLaunchKernelGGL((k_sort_buckets<1024, false>), dim3(256 * n_sc), dim3(1024), 0, s, b, y, x, seg_b, hist, passes);
    else
        hipLaunchKernelGGL((k_sort_buckets<256, false>), dim3(256 * n_sc), dim3(256), 0, s, b, y, x, seg_b, hist, passes);
    return hipGetLastError();
}

}  // namespace pfh
