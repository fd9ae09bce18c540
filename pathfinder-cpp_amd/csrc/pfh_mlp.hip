// FP32 sizing predictor: MLP 12 -> 64 -> 64 -> 3 (ReLU), trained on (path features ->
// log1p(chord count), log1p(fill count), log1p(alpha tile count)) triples that the
// flatten and bin count passes emit.  It
// replaces the reference's "count, read back, grow to 2^k, retry" sizing
// (core/d3d11/renderer.cpp:537-577, 707-724, 834-845) for batched launches; an
// under-prediction costs a retry, never a wrong pixel.  Tiny matrices: plain FP32
// VALU kernels, no MFMA.
//
// Parameter layout (5187 floats): W1[12][64], b1[64], W2[64][64], b2[64], W3[64][3], b3[3]
// (row-major, W[in][out]).  Hidden activations per sample: h1[64], h2[64].
#include "pfh_internal.h"

namespace pfh {

constexpr int NI = 12, NH = 64, NO = 3;
constexpr int OFF_W1 = 0, OFF_B1 = OFF_W1 + NI * NH, OFF_W2 = OFF_B1 + NH, OFF_B2 = OFF_W2 + NH * NH,
              OFF_W3 = OFF_B2 + NH, OFF_B3 = OFF_W3 + NH * NO, N_PARAMS = OFF_B3 + NO;

int64_t mlp_param_count() { return N_PARAMS; }

__global__ void k_zero(float *p, int64_t n) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0.0f;
}


__global__ __launch_bounds__(256) void k_mlp_forward(const float *__restrict__ P, const float *__restrict__ x,
                                                     int64_t n, float *__restrict__ hidden, float *__restrict__ out) {
    __shared__ float w[N_PARAMS];
    for (int i = threadIdx.x; i < N_PARAMS; i += blockDim.x) w[i] = P[i];
    __syncthreads();
    int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    float xi[NI];
#pragma unroll
    for (int i = 0; i < NI; i++) xi[i] = x[s * NI + i];
    float h1[NH];
#pragma unroll 4
    for (int j = 0; j < NH; j++) {
        float a = w[OFF_B1 + j];
#pragma unroll
        for (int i = 0; i < NI; i++) a += xi[i] * w[OFF_W1 + i * NH + j];
        h1[j] = fmaxf(a, 0.0f);
    }
    float o[NO];
#pragma unroll
    for (int q = 0; q < NO; q++) o[q] = w[OFF_B3 + q];
    for (int j = 0; j < NH; j++) {
        float a = w[OFF_B2 + j];
#pragma unroll 8
        for (int i = 0; i < NH; i++) a += h1[i] * w[OFF_W2 + i * NH + j];
        float h2 = fmaxf(a, 0.0f);
        hidden[s * 2 * NH + NH + j] = h2;
#pragma unroll
        for (int q = 0; q < NO; q++) o[q] += h2 * w[OFF_W3 + j * NO + q];
    }
#pragma unroll 8
    for (int j = 0; j < NH; j++) hidden[s * 2 * NH + j] = h1[j];
#pragma unroll
    for (int q = 0; q < NO; q++) out[s * NO + q] = o[q];
}

// Per-sample output and hidden gradients of the mean squared error
// L = 1/(n*NO) * sum (out - target)^2; writes g[s] = (dout[NO], dh2[64], dh1[64]).
__global__ __launch_bounds__(256) void k_mlp_backward_act(const float *__restrict__ P, int64_t n,
                                                          const float *__restrict__ hidden,
                                                          const float *__restrict__ out,
                                                          const float *__restrict__ target, float *__restrict__ g,
                                                          float *__restrict__ loss) {
    __shared__ float w2[NH * NH];
    __shared__ float w3[NH * NO];
    __shared__ float red[4];
    for (int i = threadIdx.x; i < NH * NH; i += blockDim.x) w2[i] = P[OFF_W2 + i];
    for (int i = threadIdx.x; i < NH * NO; i += blockDim.x) w3[i] = P[OFF_W3 + i];
    __syncthreads();
    int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    float l = 0.0f;
    if (s < n) {
        const float scale = 2.0f / (float)(n * NO);
        float d[NO];
        float *gs = g + s * (NO + 2 * NH);
#pragma unroll
        for (int q = 0; q < NO; q++) {
            float e = out[s * NO + q] - target[s * NO + q];
            l += e * e;
            d[q] = scale * e;
            gs[q] = d[q];
        }
        const float *h = hidden + s * 2 * NH;
        float dh2[NH];
#pragma unroll 8
        for (int j = 0; j < NH; j++) {
            float acc = 0.0f;
#pragma unroll
            for (int q = 0; q < NO; q++) acc += d[q] * w3[j * NO + q];
            float v = h[NH + j] > 0.0f ? acc : 0.0f;
            dh2[j] = v;
            gs[NO + j] = v;
        }
        for (int i = 0; i < NH; i++) {
            float a = 0.0f;
#pragma unroll 8
            for (int j = 0; j < NH; j++) a += w2[i * NH + j] * dh2[j];
            gs[NO + NH + i] = h[i] > 0.0f ? a : 0.0f;
        }
    }
    // block reduction of the loss
    for (int d = 32; d > 0; d >>= 1) l += __shfl_down(l, d, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = l;
    __syncthreads();
    if (threadIdx.x == 0) atomicAdd(loss, (red[0] + red[1] + red[2] + red[3]) / (float)(n * NO));
}

// dW[ka][kb] += sum_s A[s][:ka]^T B[s][:kb]; db[kb] += sum_s B[s][:kb].  A block reduces
// OUTER_SAMPLES samples in LDS tiles of OUTER_TILE, keeps its outputs in registers and
// adds them to the global gradient once.
constexpr int OUTER_TILE = 64;
constexpr int OUTER_SAMPLES = 4096;
constexpr int OUTER_PER_THREAD = (NH * NH + NH + 255) / 256;  // 17
__global__ __launch_bounds__(256) void k_mlp_outer(const float *__restrict__ A, int lda, int ka,
                                                   const float *__restrict__ B, int ldb, int boff, int kb, int64_t n,
                                                   float *__restrict__ dW, float *__restrict__ db) {
    __shared__ float sa[OUTER_TILE][NH + 1];
    __shared__ float sb[OUTER_TILE][NH + 1];
    float acc[OUTER_PER_THREAD];
#pragma unroll
    for (int k = 0; k < OUTER_PER_THREAD; k++) acc[k] = 0.0f;
    const int total = ka * kb;
    int64_t first = (int64_t)blockIdx.x * OUTER_SAMPLES;
    int64_t last = min<int64_t>(n, first + OUTER_SAMPLES);
    for (int64_t s0 = first; s0 < last; s0 += OUTER_TILE) {
        int cnt = (int)min<int64_t>(OUTER_TILE, last - s0);
        __syncthreads();
        for (int i = threadIdx.x; i < cnt * ka; i += blockDim.x) sa[i / ka][i % ka] = A[(s0 + i / ka) * lda + i % ka];
        for (int i = threadIdx.x; i < cnt * kb; i += blockDim.x)
            sb[i / kb][i % kb] = B[(s0 + i / kb) * ldb + boff + i % kb];
        __syncthreads();
#pragma unroll
        for (int k = 0; k < OUTER_PER_THREAD; k++) {
            int o = threadIdx.x + k * 256;
            if (o < total) {
                int i = o / kb, j = o % kb;
                float a = 0.0f;
                for (int s = 0; s < cnt; s++) a += sa[s][i] * sb[s][j];
                acc[k] += a;
            } else if (o < total + kb) {
                int j = o - total;
                float a = 0.0f;
                for (int s = 0; s < cnt; s++) a += sb[s][j];
                acc[k] += a;
            }
        }
    }
#pragma unroll
    for (int k = 0; k < OUTER_PER_THREAD; k++) {
        int o = threadIdx.x + k * 256;
        if (o < total) atomicAdd(&dW[o], acc[k]);
        else if (o < total + kb) atomicAdd(&db[o - total], acc[k]);
    }
}


// ---------------------------------------------------------------------------
// Per-path features (the network's inputs), a wave per path
// ---------------------------------------------------------------------------
//
// The bounding box over the canvas' longer side, log1p of the control polygon's length, of its turning
// (the angles between its consecutive edges of non-zero length, in segment order), of the
// line, quad and cubic counts and of the tile rect's area, log of the side, and the fill rule.
// Lanes take consecutive segments; a segment's first edge turns from the last edge of the
// nearest earlier segment that has one, found by ballot.  On the host this took 32 us per thousand
// segments (an arc cosine per edge): 0.32 ms of a 900^2 scene's upload, 1.6 ms of 400 dashed
// strokes'; 12 and 42 us here.
__global__ __launch_bounds__(256) void k_path_features(const float2 *pts, const uint2 *segs, const uint32_t *seg_off,
                                                       const int4 *rects, const uint8_t *rules, uint32_t n_paths,
                                                       float side, float *out) {
#pragma clang fp contract(off)
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t p = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
    if (p >= n_paths) return;  // whole wave
    const uint32_t s0 = seg_off[p], s1 = seg_off[p + 1];
    float poly = 0.0f, turn = 0.0f, bx0 = 1e30f, by0 = 1e30f, bx1 = -1e30f, by1 = -1e30f;
    uint32_t kinds[3] = {0, 0, 0};
    float cx = 0.0f, cy = 0.0f;  // direction of the last edge before this round (wave-uniform)
    bool have = false;
    // no contraction: an arc cosine near 1 turns the last bit of its argument into 3e-4
    auto angle = [](float ax, float ay, float bx, float by) {
#pragma clang fp contract(off)
        return acosf(fmaxf(-1.0f, fminf(1.0f, ax * bx + ay * by)));
    };
    for (uint32_t base = s0; base < s1; base += 64) {  // uniform over the wave
        const uint32_t i = base + lane;
        float fx = 0.0f, fy = 0.0f, lx = 0.0f, ly = 0.0f;  // this segment's first and last edge
        bool any = false;
        if (i < s1) {
            const uint2 sg = segs[i];
            const uint32_t kind = sg.y >> SEG_ORIGINAL_SHIFT;
            kinds[0] += kind == SEG_LINE ? 1u : 0u;
            kinds[1] += kind == SEG_QUAD ? 1u : 0u;
            kinds[2] += kind == SEG_CUBIC ? 1u : 0u;
            const uint32_t np = kind == SEG_LINE ? 2u : (kind == SEG_QUAD ? 3u : 4u);
            float2 a = {};
            for (uint32_t q = 0; q < np; q++) {
                const float2 c = pts[sg.x + q];
                bx0 = c.x < bx0 ? c.x : bx0;
                by0 = c.y < by0 ? c.y : by0;
                bx1 = bx1 < c.x ? c.x : bx1;
                by1 = by1 < c.y ? c.y : by1;
                if (q > 0) {
                    const float dx = c.x - a.x, dy = c.y - a.y, len = sqrtf(dx * dx + dy * dy);
                    poly += len;
                    if (len > 0.0f) {
                        const float ux = dx / len, uy = dy / len;
                        if (any) turn += angle(ux, uy, lx, ly);
                        else {
                            fx = ux;
                            fy = uy;
                        }
                        lx = ux;
                        ly = uy;
                        any = true;
                    }
                }
                a = c;
            }
        }
        const uint64_t m = __ballot(any);
        const uint64_t before = m & ((1ull << lane) - 1ull);
        const int from = before ? 63 - __clzll(before) : 0;
        float px = __shfl(lx, from, 64), py = __shfl(ly, from, 64);
        if (!before) {
            px = cx;
            py = cy;
        }
        if (any && (before || have)) turn += angle(fx, fy, px, py);
        if (m) {
            const int last = 63 - __clzll(m);
            cx = __shfl(lx, last, 64);
            cy = __shfl(ly, last, 64);
            have = true;
        }
    }
    for (int d = 32; d > 0; d >>= 1) {
        poly += __shfl_xor(poly, d, 64);
        turn += __shfl_xor(turn, d, 64);
        const float x0 = __shfl_xor(bx0, d, 64), y0 = __shfl_xor(by0, d, 64), x1 = __shfl_xor(bx1, d, 64),
                    y1 = __shfl_xor(by1, d, 64);
        bx0 = x0 < bx0 ? x0 : bx0;
        by0 = y0 < by0 ? y0 : by0;
        bx1 = bx1 < x1 ? x1 : bx1;
        by1 = by1 < y1 ? y1 : by1;
        for (int k = 0; k < 3; k++) kinds[k] += __shfl_xor(kinds[k], d, 64);
    }
    if (bx0 > bx1) bx0 = by0 = bx1 = by1 = 0.0f;
    if (lane == 0) {
        const int4 r = rects[p];
        float *f = out + (int64_t)p * NI;
        f[0] = bx0 / side;
        f[1] = by0 / side;
        f[2] = bx1 / side;
        f[3] = by1 / side;
        f[4] = log1pf(poly);
        f[5] = log1pf(turn);
        f[6] = log1pf((float)kinds[0]);
        f[7] = log1pf((float)kinds[1]);
        f[8] = log1pf((float)kinds[2]);
        f[9] = log1pf((float)max(0, r.z - r.x) * (float)max(0, r.w - r.y));
        f[10] = logf(side);
        f[11] = (float)rules[p];
    }
}

hipError_t path_features(const float2 *pts, const uint2 *segs, const uint32_t *seg_off, const int4 *rects,
                         const uint8_t *rules, uint32_t n_paths, float side, float *out, hipStream_t s) {
    if (n_paths == 0) return hipSuccess;
    hipLaunchKernelGGL(k_path_features, dim3((n_paths + 3) / 4), dim3(256), 0, s, pts, segs, seg_off, rects, rules, n_paths,
                       side, out);
    return hipGetLastError();
}

// Sizing inference: per path forward pass, expm1 of the (log1p) outputs clamped at 0, summed over
// the paths into sums[NO] (float atomics per block).  A wave per path, a lane per hidden unit with its
// columns of the weights in registers; the first layer's units reach the others as scalars (lane
// reads).  A scene has hundreds to thousands of paths, so a thread per path left a few waves with
// 5 000 dependent multiply-adds each: 304 paths took 100 us, now 4.
constexpr unsigned PREDICT_BLOCKS = 256;  // at most one per CU: 3 adds per block on the same addresses
__global__ __launch_bounds__(256) void k_mlp_predict_sum(const float *__restrict__ P, const float *__restrict__ x,
                                                         int64_t n, float *__restrict__ sums) {
    static_assert(NH == 64, "a lane per hidden unit");
    __shared__ float red[4][NO];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    float w1[NI], w2[NH], w3[NO];
#pragma unroll
    for (int i = 0; i < NI; i++) w1[i] = P[OFF_W1 + i * NH + lane];
#pragma unroll
    for (int i = 0; i < NH; i++) w2[i] = P[OFF_W2 + i * NH + lane];
#pragma unroll
    for (int q = 0; q < NO; q++) w3[q] = P[OFF_W3 + lane * NO + q];
    const float b1 = P[OFF_B1 + lane], b2 = P[OFF_B2 + lane];
    float sum[NO];
#pragma unroll
    for (int q = 0; q < NO; q++) sum[q] = 0.0f;
    const int64_t first = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + wv);
    for (int64_t s = first; s < n; s += (int64_t)gridDim.x * 4) {  // wave-uniform
        float a = b1;
#pragma unroll
        for (int i = 0; i < NI; i++) a += x[s * NI + i] * w1[i];
        const float h1 = fmaxf(a, 0.0f);
        a = b2;
#pragma unroll
        for (int i = 0; i < NH; i++) a += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(h1), i)) * w2[i];
        const float h2 = fmaxf(a, 0.0f);
#pragma unroll
        for (int q = 0; q < NO; q++) {
            float v = h2 * w3[q];
            for (int d = 32; d > 0; d >>= 1) v += __shfl_xor(v, d, 64);
            sum[q] += expm1f(fmaxf(v + P[OFF_B3 + q], 0.0f));
        }
    }
    if (lane == 0) {
#pragma unroll
        for (int q = 0; q < NO; q++) red[wv][q] = sum[q];
    }
    __syncthreads();
    if (threadIdx.x < NO) atomicAdd(&sums[threadIdx.x], red[0][threadIdx.x] + red[1][threadIdx.x] +
                                                            red[2][threadIdx.x] + red[3][threadIdx.x]);
}

hipError_t mlp_predict_sum(const float *params, const float *x, int64_t n, float *sums, hipStream_t s) {
    hipLaunchKernelGGL(k_zero, dim3(1), dim3(32), 0, s, sums, (int64_t)NO);
    if (n > 0)
        hipLaunchKernelGGL(k_mlp_predict_sum, dim3((unsigned)std::min<int64_t>((n + 3) / 4, PREDICT_BLOCKS)), dim3(256), 0,
                           s, params, x, n, sums);
    return hipGetLastError();
}

hipError_t mlp_forward(const float *params, const float *x, int64_t n, float *hidden, float *out, hipStream_t s) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_mlp_forward, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, params, x, n, hidden, out);
    return hipGetLastError();
}

// grad: N_PARAMS floats (overwritten); loss: 1 float (overwritten); scratch: n * (NO + 2 NH) floats.
hipError_t mlp_backward(const float *params, const float *x, int64_t n, const float *hidden, const float *out,
                        const float *target, float *grad, float *loss, float *scratch, hipStream_t s) {
    hipLaunchKernelGGL(k_zero, dim3((N_PARAMS + 255) / 256), dim3(256), 0, s, grad, (int64_t)N_PARAMS);
    hipLaunchKernelGGL(k_zero, dim3(1), dim3(32), 0, s, loss, (int64_t)1);
    if (n == 0) return hipGetLastError();
    unsigned nb = (unsigned)((n + 255) / 256);
    hipLaunchKernelGGL(k_mlp_backward_act, dim3(nb), dim3(256), 0, s, params, n, hidden, out, target, scratch, loss);
    unsigned nc = (unsigned)((n + OUTER_SAMPLES - 1) / OUTER_SAMPLES);
    const int LG = NO + 2 * NH;
    // layer 3: A = h2, B = dout
    hipLaunchKernelGGL(k_mlp_outer, dim3(nc), dim3(256), 0, s, hidden + NH, 2 * NH, NH, scratch, LG, 0, NO, n,
                       grad + OFF_W3, grad + OFF_B3);
    // layer 2: A = h1, B = dh2
    hipLaunchKernelGGL(k_mlp_outer, dim3(nc), dim3(256), 0, s, hidden, 2 * NH, NH, scratch, LG, NO, NH, n,
                       grad + OFF_W2, grad + OFF_B2);
    // layer 1: A = x, B = dh1
    hipLaunchKernelGGL(k_mlp_outer, dim3(nc), dim3(256), 0, s, x, NI, NI, scratch, LG, NO + NH, NH, n, grad + OFF_W1,
                       grad + OFF_B1);
    return hipGetLastError();
}

__global__ void k_adam(float *p, float *m, float *v, const float *g, int64_t n, float lr, float c1, float c2) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    float gi = g[i];
    float mi = b1 * m[i] + (1.0f - b1) * gi;
    float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

hipError_t mlp_adam(float *params, float *m, float *v, const float *grad, int64_t n, float lr, int step,
                    hipStream_t s) {
    float c1 = 1.0f - powf(0.9f, (float)step), c2 = 1.0f - powf(0.999f, (float)step);
    hipLaunchKernelGGL(k_adam, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, params, m, v, grad, n, lr, c1, c2);
    return hipGetLastError();
}

}  // namespace pfh
