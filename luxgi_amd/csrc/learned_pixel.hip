// learned_pixel.hip -- per-pixel learned edge-stopping scales for the reflection a-trous chain,
// with their training kernels, for gfx950. No counterpart in the reference.
//
// A 12 -> 32 -> 32 -> 5 ReLU MLP with FP16 weights maps per-pixel features to one scale per
// a-trous pass, s_i = exp(clamp(o_i, -4, 4)). Pass i of the reference's chain
// (Reflection/DenoiseAtrous.comp:63-134, driven by RaytracedReflection.cpp:419-494) then weighs
// each tap by the reference's edge-stopping weight (EdgeStop.glsl:24-40) with the luminance term
// scaled, wL = s_i(p) |l_p - l_q| / phi_p (luxgi_svgf_reflection_atrous_scaled). All-zero output
// weights give s = 1: the reference chain, bit for bit.
//
// Features f of pixel p (the pass-0 input: rgb + variance; the reprojection's moments m1, m2 and
// history length; the G-buffer normal and linear depth):
//   f0, f1  |z(x+1) - z(x-1)| / 2z and the same along y (edge-clamped), at most 1
//   f2..f4  the decoded normal
//   f5      log(1 + l), l the input luminance
//   f6, f7  log(1 + mean) and min(std / (mean + 1e-3), 4) of the 3x3 luminances
//   f8      min(sqrt(variance) / (l + 1e-3), 4)
//   f9, f10 log(1 + m1) and min(sqrt(max(0, m2 - m1^2)) / (m1 + 1e-3), 4)
//   f11     min(history length, 32) / 32
// Parameters (FP32 master copy; the forward rounds the weights, the features and the hidden
// activations to FP16 for the MFMA and accumulates in FP32): W1 [32][12], b1 [32], W2 [32][32],
// b2 [32], W3 [5][32], b3 [5] = 1637 floats.
//
// Inference: one kernel computes the features and runs the three layers on
// v_mfma_f32_16x16x16_f16 / v_mfma_f32_16x16x32_f16 (units x features . features x 16 pixels),
// the activations passed between layers through LDS. Training: the backward of a scaled pass in
// gather form (a centre kernel keeps each filtered pixel's dL/d(out) / sum of weights and its
// luminance factor; a gather kernel adds each pixel's share of its neighbours' taps, no atomics)
// and the MLP's backward on the matrix units with the parameter gradient summed per wave, block
// and grid in a fixed order (deterministic). The weights' dependence on the input
// colour (luminance, the variance behind phi) is held fixed in the backward.
#include <algorithm>

#include "svgf_common.hpp"

namespace luxgi {

constexpr int kLpIn = 12, kLpInPad = 16, kLpHid = 32, kLpOut = 5;
constexpr int kLpW1 = 0, kLpB1 = kLpW1 + kLpHid * kLpIn, kLpW2 = kLpB1 + kLpHid, kLpB2 = kLpW2 + kLpHid * kLpHid,
              kLpW3 = kLpB2 + kLpHid, kLpB3 = kLpW3 + kLpOut * kLpHid, kLpParams = kLpB3 + kLpOut;
static_assert(kLpParams == LUXGI_LEARNED_PIXEL_PARAMS, "parameter count");
constexpr float kLpClamp = 4.0f;

typedef _Float16 lp_half4 __attribute__((ext_vector_type(4)));
typedef _Float16 lp_half8 __attribute__((ext_vector_type(8)));
typedef float lp_float4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void lp_features(int W, int H, int x, int y, const float4* __restrict__ color,
                                            const float4* __restrict__ moments, const float4* __restrict__ normals,
                                            const float4* __restrict__ pbr, float* f) {
    const int xl = max(x - 1, 0), xr = min(x + 1, W - 1), yu = max(y - 1, 0), yd = min(y + 1, H - 1);
    const size_t e = (size_t)y * W + x;
    const float z = load_linear_depth(pbr, e);
    const float iz = 1.0f / fmaxf(z, 1e-4f);
    const float zl = load_linear_depth(pbr, (size_t)y * W + xl), zr = load_linear_depth(pbr, (size_t)y * W + xr);
    const float zu = load_linear_depth(pbr, (size_t)yu * W + x), zd = load_linear_depth(pbr, (size_t)yd * W + x);
    f[0] = fminf(fabsf(zr - zl) * 0.5f * iz, 1.0f);
    f[1] = fminf(fabsf(zd - zu) * 0.5f * iz, 1.0f);
    const f3 n = load_normal(normals, e);
    f[2] = n.x;
    f[3] = n.y;
    f[4] = n.z;
    const float4 c = color[e];
    const float l = luminance(c.x, c.y, c.z);
    f[5] = log1pf(l);
    float s1 = 0.0f, s2 = 0.0f;
    for (int yy = -1; yy <= 1; ++yy)
        for (int xx = -1; xx <= 1; ++xx) {
            const int qx = min(max(x + xx, 0), W - 1), qy = min(max(y + yy, 0), H - 1);
            const float4 q = color[(size_t)qy * W + qx];
            const float lq = luminance(q.x, q.y, q.z);
            s1 += lq;
            s2 += lq * lq;
        }
    const float mu = s1 * (1.0f / 9.0f);
    const float sd = sqrtf(fmaxf(0.0f, s2 * (1.0f / 9.0f) - mu * mu));
    f[6] = log1pf(mu);
    f[7] = fminf(sd / (mu + 1e-3f), 4.0f);
    f[8] = fminf(sqrtf(fmaxf(c.w, 0.0f)) / (l + 1e-3f), 4.0f);
    const float4 m = moments[e];
    const float m1 = fmaxf(m.x, 0.0f);
    f[9] = log1pf(m1);
    f[10] = fminf(sqrtf(fmaxf(0.0f, m.y - m1 * m1)) / (m1 + 1e-3f), 4.0f);
    f[11] = fminf(m.z, 32.0f) * (1.0f / 32.0f);
}

// ---------------------------------------------------------------------------------------------
// Forward: features + MLP (MFMA). 256 pixels per block, one per lane for the features; each wave
// then runs its 64 pixels through the layers 16 at a time. MFMA lane layouts (l = lane, g = l / 16):
//   16x16x16 f16: A[l % 16][4g + j], B[4g + j][l % 16];  16x16x32 f16: A[l % 16][8g + j],
//   B[8g + j][l % 16];  D[4g + v][l % 16].  A = weights (units x inputs), B = inputs x pixels.
// ---------------------------------------------------------------------------------------------
struct LpForwardLds {
    _Float16 f[256][kLpInPad];    // features, FP16
    _Float16 h[4][16][kLpHid];    // per wave: one layer's activations of 16 pixels
};

__global__ __launch_bounds__(256) void lp_forward_kernel(const float* __restrict__ P, int W, int H,
                                                         const float4* __restrict__ color,
                                                         const float4* __restrict__ moments,
                                                         const float4* __restrict__ normals,
                                                         const float4* __restrict__ pbr, float* __restrict__ scales,
                                                         float* __restrict__ featOut) {
    __shared__ LpForwardLds lds;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int col = lane & 15, g = lane >> 4;
    const long long N = (long long)W * H;
    const long long p0 = (long long)blockIdx.x * 256;
    {
        const long long p = p0 + tid;
        float f[kLpIn];
        if (p < N) {
            lp_features(W, H, int(p % W), int(p / W), color, moments, normals, pbr, f);
            if (featOut)
                for (int i = 0; i < kLpIn; ++i) featOut[p * kLpIn + i] = f[i];
        } else {
            for (int i = 0; i < kLpIn; ++i) f[i] = 0.0f;
        }
        for (int i = 0; i < kLpIn; ++i) lds.f[tid][i] = (_Float16)f[i];
        for (int i = kLpIn; i < kLpInPad; ++i) lds.f[tid][i] = (_Float16)0.0f;
    }
    // weight fragments (A operands), rounded to FP16; biases of the rows this lane's D holds
    lp_half4 a1[2];
    lp_half8 a2[2], a3;
    float b1v[2][4], b2v[2][4], b3v[4];
    for (int mt = 0; mt < 2; ++mt) {
        const int u = mt * 16 + col;
        for (int j = 0; j < 4; ++j) {
            const int k = 4 * g + j;
            a1[mt][j] = (_Float16)(k < kLpIn ? P[kLpW1 + u * kLpIn + k] : 0.0f);
        }
        for (int j = 0; j < 8; ++j) a2[mt][j] = (_Float16)P[kLpW2 + u * kLpHid + 8 * g + j];
        for (int v = 0; v < 4; ++v) {
            b1v[mt][v] = P[kLpB1 + mt * 16 + 4 * g + v];
            b2v[mt][v] = P[kLpB2 + mt * 16 + 4 * g + v];
        }
    }
    for (int j = 0; j < 8; ++j) a3[j] = (_Float16)(col < kLpOut ? P[kLpW3 + col * kLpHid + 8 * g + j] : 0.0f);
    for (int v = 0; v < 4; ++v) b3v[v] = 4 * g + v < kLpOut ? P[kLpB3 + 4 * g + v] : 0.0f;
    __syncthreads();
    for (int b = 0; b < 4; ++b) {
        const int pl = wave * 64 + b * 16;  // the batch's first pixel in the block
        // layer 1
        lp_half4 bf;
        for (int j = 0; j < 4; ++j) bf[j] = lds.f[pl + col][4 * g + j];
        for (int mt = 0; mt < 2; ++mt) {
            lp_float4 d = __builtin_amdgcn_mfma_f32_16x16x16f16(a1[mt], bf, lp_float4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
            for (int v = 0; v < 4; ++v) lds.h[wave][col][mt * 16 + 4 * g + v] = (_Float16)fmaxf(d[v] + b1v[mt][v], 0.f);
        }
        __syncthreads();
        // layer 2
        lp_half8 bh;
        for (int j = 0; j < 8; ++j) bh[j] = lds.h[wave][col][8 * g + j];
        __syncthreads();
        for (int mt = 0; mt < 2; ++mt) {
            lp_float4 d = __builtin_amdgcn_mfma_f32_16x16x32_f16(a2[mt], bh, lp_float4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
            for (int v = 0; v < 4; ++v) lds.h[wave][col][mt * 16 + 4 * g + v] = (_Float16)fmaxf(d[v] + b2v[mt][v], 0.f);
        }
        __syncthreads();
        // layer 3
        for (int j = 0; j < 8; ++j) bh[j] = lds.h[wave][col][8 * g + j];
        __syncthreads();
        const lp_float4 d = __builtin_amdgcn_mfma_f32_16x16x32_f16(a3, bh, lp_float4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
        const long long p = p0 + pl + col;
        if (p < N) {
            for (int v = 0; v < 4; ++v) {
                const int o = 4 * g + v;
                if (o < kLpOut) scales[(size_t)o * N + p] = __expf(clampf(d[v] + b3v[v], -kLpClamp, kLpClamp));
            }
        }
    }
}

// ---------------------------------------------------------------------------------------------
// Backward of one scaled reflection a-trous pass (FP32 images).
// ---------------------------------------------------------------------------------------------
struct LpPassArgs {
    int W, H, tilesX, radius, stepSize;
    float phi, phiNormal, sigmaDepth;
    int sqNormal;
};

// mode of a pixel in the pass: 0 the output is the input (copy tile, or roughness outside the
// band), 1 filtered, 2 zero (sky in a filtered tile)
__device__ __forceinline__ int lp_mode(const LpPassArgs& A, const uint8_t* tileMap, const float4* pbr, int x, int y) {
    if (!tileMap[(y >> 3) * A.tilesX + (x >> 3)]) return 0;
    const size_t e = (size_t)y * A.W + x;
    const float cd = load_linear_depth(pbr, e), rough = load_roughness(pbr, e);
    if (cd == 1.0f) return 2;
    return (rough <= 0.05f || rough >= 0.45f) ? 0 : 1;
}

// Both kernels run over 16x16-pixel blocks. Where the footprint radius * step is at most kLpHalo, the block
// stages its images with that halo in LDS, guides decoded once per texel, as the forward passes do
// (TILED); larger steps read every tap from memory. Bound: with every tap read and its normal
// decoded at every use (the centre kernel walks its taps twice), by instructions and L1 requests:
// 32 + 28 us per pass at 960x540 against 17 + 23 staged (the step: 569 -> 480 us).
constexpr int kLpHalo = 8;

struct LpRegion {
    int h, side, ox, oy;
};
__device__ __forceinline__ LpRegion lp_region(const LpPassArgs& A) {
    LpRegion r;
    r.h = max(A.radius * A.stepSize, 1);
    r.side = 16 + 2 * r.h;
    r.ox = (int)blockIdx.x * 16 - r.h;
    r.oy = (int)blockIdx.y * 16 - r.h;
    return r;
}
// stages image texels and guides (decoded normal, linear depth); 0 outside the image
__device__ __forceinline__ void lp_stage(const LpPassArgs& A, const LpRegion& r, const float4* __restrict__ normals,
                                         const float4* __restrict__ pbr, const float4* __restrict__ in, float4* sIn,
                                         float4* sGuide) {
    for (int ly = threadIdx.x >> 4; ly < r.side; ly += 16)
        for (int lx = threadIdx.x & 15; lx < r.side; lx += 16) {
            const int gx = r.ox + lx, gy = r.oy + ly;
            float4 v = make_float4(0.f, 0.f, 0.f, 0.f), g = v;
            if (inside(gx, gy, A.W, A.H)) {
                const size_t q = (size_t)gy * A.W + gx;
                v = in[q];
                const f3 n = load_normal(normals, q);
                g = make_float4(n.x, n.y, n.z, load_linear_depth(pbr, q));
            }
            sIn[ly * r.side + lx] = v;
            sGuide[ly * r.side + lx] = g;
        }
}
// weight of a tap: the reference's exponent 32 in line, others through the general power
__device__ __forceinline__ float lp_weight(const LpPassArgs& A, float cd, float d, float invPhiZ, f3 cn, f3 sn, float cl,
                                           float sl, float invPhiL) {
    return A.sqNormal == 5 ? edge_stop32(cd, d, invPhiZ, cn, sn, cl, sl, invPhiL)
                           : edge_stop(cd, d, invPhiZ, cn, sn, A.phiNormal, A.sqNormal, cl, sl, invPhiL);
}

// record[p] = (dL/d out_p / sw_p (rgb), s_p / phi_p) for filtered centres; mode[p]; dL/ds_p. One walk over
// the taps: with r = dL/d out / sw, dw/ds = -|l_p - l_q| / phi_p w and colours relative to the centre's (d_q =
// x_q - x_p, m = sum w d_q / sw), dL/ds = sum r . (x_q - out) dw/ds = -(1 / phi_p) r . (sum w |dl| d_q - m sum w |dl|).
// Sums of the colours themselves would cancel: a channel of 1000 that varies by 0.05 came out 1e-2 wrong.
template <bool TILED>
__global__ __launch_bounds__(256) void lp_pass_centre_kernel(LpPassArgs A, const float4* __restrict__ normals,
                                                             const float4* __restrict__ pbr,
                                                             const uint8_t* __restrict__ tileMap,
                                                             const float4* __restrict__ in,
                                                             const float* __restrict__ scale,
                                                             const float4* __restrict__ gOut,
                                                             float4* __restrict__ record, uint8_t* __restrict__ mode,
                                                             float* __restrict__ gScale) {
    extern __shared__ float4 lpLds[];
    const LpRegion r = lp_region(A);
    float4* sIn = lpLds;
    float4* sGuide = lpLds + r.side * r.side;
    const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
    const int x = blockIdx.x * 16 + tx, y = blockIdx.y * 16 + ty;
    const bool on = x < A.W && y < A.H;
    const size_t e = (size_t)y * A.W + x;
    const int m = on ? lp_mode(A, tileMap, pbr, x, y) : 0;
    if (TILED) {
        if (__syncthreads_or(m == 1)) {  // uniform over the block
            lp_stage(A, r, normals, pbr, in, sIn, sGuide);
            __syncthreads();
        }
    }
    if (!on) return;
    mode[e] = (uint8_t)m;
    if (m != 1) {
        record[e] = make_float4(0.f, 0.f, 0.f, 0.f);
        gScale[e] = 0.0f;
        return;
    }
    const int lc = (ty + r.h) * r.side + tx + r.h;
    const float kw[3] = {1.0f, 2.0f / 3.0f, 1.0f / 6.0f};
    const float kv[2][2] = {{1.0f / 4.0f, 1.0f / 8.0f}, {1.0f / 8.0f, 1.0f / 16.0f}};
    const float4 c = TILED ? sIn[lc] : in[e];
    float var = 0.0f;
    for (int yy = -1; yy <= 1; ++yy)
        for (int xx = -1; xx <= 1; ++xx)
            var += (TILED ? sIn[lc + yy * r.side + xx].w : fetch4(in, x + xx, y + yy, A.W, A.H).w) * kv[abs(xx)][abs(yy)];
    const float cl = luminance(c.x, c.y, c.z);
    const float phiC = A.phi * sqrtf(fmaxf(0.0f, var)) + 1e-10f;
    const float invPhiC = 1.0f / phiC, invPhiZ = 1.0f / A.sigmaDepth;
    const float invPhiL = invPhiC * scale[e];
    float cd;
    f3 cn;
    if (TILED) {
        const float4 gc = sGuide[lc];
        cd = gc.w;
        cn = mk(gc.x, gc.y, gc.z);
    } else {
        cd = load_linear_depth(pbr, e);
        cn = load_normal(normals, e);
    }
    float sw = 1.0f, sd = 0.0f;
    f3 m1 = mk(0.f, 0.f, 0.f), md = m1;  // sums of w d_q and of w |dl| d_q
    for (int yy = -A.radius; yy <= A.radius; ++yy)
        for (int xx = -A.radius; xx <= A.radius; ++xx) {
            const int px = x + xx * A.stepSize, py = y + yy * A.stepSize;
            if (!inside(px, py, A.W, A.H) || (xx == 0 && yy == 0)) continue;
            float4 sc;
            f3 sn;
            float d;
            if (TILED) {
                const int l = lc + yy * A.stepSize * r.side + xx * A.stepSize;
                sc = sIn[l];
                const float4 g = sGuide[l];
                sn = mk(g.x, g.y, g.z);
                d = g.w;
            } else {
                const size_t q = (size_t)py * A.W + px;
                sc = in[q];
                sn = load_normal(normals, q);
                d = load_linear_depth(pbr, q);
            }
            const float sl = luminance(sc.x, sc.y, sc.z);
            const float w = lp_weight(A, cd, d, invPhiZ, cn, sn, cl, sl, invPhiL) * (kw[abs(xx)] * kw[abs(yy)]);
            const float wd = w * fabsf(cl - sl);
            sw += w;
            sd += wd;
            const f3 dq = mk(sc.x - c.x, sc.y - c.y, sc.z - c.z);
            m1 = m1 + dq * w;
            md = md + dq * wd;
        }
    const float isw = 1.0f / sw;
    const f3 k = md - m1 * (isw * sd);
    const float4 g = gOut[e];
    const f3 rr = mk(g.x * isw, g.y * isw, g.z * isw);
    record[e] = make_float4(rr.x, rr.y, rr.z, invPhiL);
    gScale[e] = -invPhiC * (rr.x * k.x + rr.y * k.y + rr.z * k.z);
}

// dL/d in_q (rgb): its own term plus r_p w_pq for every filtered neighbour p whose tap q is. Tiled, the
// block also stages its neighbours' records; a neighbour that is not filtered has a zero record.
template <bool TILED>
__global__ __launch_bounds__(256) void lp_pass_gather_kernel(LpPassArgs A, const float4* __restrict__ normals,
                                                             const float4* __restrict__ pbr,
                                                             const float4* __restrict__ in,
                                                             const float4* __restrict__ gOut,
                                                             const float4* __restrict__ record,
                                                             const uint8_t* __restrict__ mode,
                                                             float4* __restrict__ gIn) {
    extern __shared__ float4 lpLds[];
    const LpRegion r = lp_region(A);
    float4* sIn = lpLds;
    float4* sGuide = lpLds + r.side * r.side;
    float4* sRec = lpLds + 2 * r.side * r.side;
    const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
    const int x = blockIdx.x * 16 + tx, y = blockIdx.y * 16 + ty;
    const bool on = x < A.W && y < A.H;
    const size_t e = (size_t)y * A.W + x;
    if (TILED) {
        bool any = false;  // a filtered centre in reach
        for (int ly = ty; ly < r.side; ly += 16)
            for (int lx = tx; lx < r.side; lx += 16) {
                const int gx = r.ox + lx, gy = r.oy + ly;
                float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
                if (inside(gx, gy, A.W, A.H)) {
                    const size_t q = (size_t)gy * A.W + gx;
                    any = any || mode[q] == 1;
                    v = record[q];
                }
                sRec[ly * r.side + lx] = v;
            }
        any = __syncthreads_or(any);
        if (any) {
            lp_stage(A, r, normals, pbr, in, sIn, sGuide);
            __syncthreads();
        }
        if (!on) return;
        if (!any) {
            const float4 g = mode[e] == 0 ? gOut[e] : make_float4(0.f, 0.f, 0.f, 0.f);
            gIn[e] = make_float4(g.x, g.y, g.z, 0.0f);
            return;
        }
    }
    if (!on) return;
    const int lc = (ty + r.h) * r.side + tx + r.h;
    const float kw[3] = {1.0f, 2.0f / 3.0f, 1.0f / 6.0f};
    const int m = mode[e];
    float a0 = 0.0f, a1 = 0.0f, a2 = 0.0f;
    if (m == 0) {
        const float4 g = gOut[e];
        a0 = g.x;
        a1 = g.y;
        a2 = g.z;
    } else if (m == 1) {
        const float4 own = TILED ? sRec[lc] : record[e];
        a0 = own.x;
        a1 = own.y;
        a2 = own.z;
    }
    const float4 sc = TILED ? sIn[lc] : in[e];
    const float sl = luminance(sc.x, sc.y, sc.z);
    float d;
    f3 sn;
    if (TILED) {
        const float4 gc = sGuide[lc];
        d = gc.w;
        sn = mk(gc.x, gc.y, gc.z);
    } else {
        d = load_linear_depth(pbr, e);
        sn = load_normal(normals, e);
    }
    const float invPhiZ = 1.0f / A.sigmaDepth;
    for (int yy = -A.radius; yy <= A.radius; ++yy)
        for (int xx = -A.radius; xx <= A.radius; ++xx) {
            const int px = x - xx * A.stepSize, py = y - yy * A.stepSize;  // the centre whose tap (xx, yy) this is
            if (!inside(px, py, A.W, A.H) || (xx == 0 && yy == 0)) continue;
            const size_t p = (size_t)py * A.W + px;
            const int l = lc - yy * A.stepSize * r.side - xx * A.stepSize;
            if (!TILED && mode[p] != 1) continue;
            const float4 rec = TILED ? sRec[l] : record[p];
            // a tiled neighbour without a record (w = s / phi > 0 in every record) is skipped alike
            if (TILED && rec.w == 0.0f && rec.x == 0.0f && rec.y == 0.0f && rec.z == 0.0f) continue;
            const float4 cp = TILED ? sIn[l] : in[p];
            float pd;
            f3 pn;
            if (TILED) {
                const float4 g = sGuide[l];
                pd = g.w;
                pn = mk(g.x, g.y, g.z);
            } else {
                pd = load_linear_depth(pbr, p);
                pn = load_normal(normals, p);
            }
            const float w = lp_weight(A, pd, d, invPhiZ, pn, sn, luminance(cp.x, cp.y, cp.z), sl, rec.w) *
                            (kw[abs(xx)] * kw[abs(yy)]);
            a0 += rec.x * w;
            a1 += rec.y * w;
            a2 += rec.z * w;
        }
    gIn[e] = make_float4(a0, a1, a2, 0.0f);
}

// ---------------------------------------------------------------------------------------------
// Backward of the MLP, on the matrix units, 16 pixels per wave and step. With the lane layouts
// above, D of a layer leaves lane (g, col) with units 4g + v and 16 + 4g + v of pixel col; the next
// contraction over units takes them as they are, with its K slots numbered to match (FP16
// 16x16x32: slot 8g + j is unit 4g + j, or 16 + 4g + j - 4; FP32 16x16x4: step (mt, v) has unit
// 16 mt + 4g + v in slot g), so the activations and the gradients pass from layer to layer in
// registers and only the weight fragments carry the permutation. The forward is recomputed as
// lp_forward_kernel does it (FP16 operands, FP32 sums); everything that holds a gradient is FP32
// (v_mfma_f32_16x16x4f32). The parameter gradients contract over pixels: the wave turns its 16
// pixels' gradients and activations around through its own LDS rows and keeps the 1,637 sums
// in accumulators over all its pixels. A block adds its waves in wave order into
// partial[block]; lp_reduce_kernel adds the blocks, in an order that is fixed too.
//
// Bound: the FP32 matrix rate (56 MFMAs of 32 cycles per 16 pixels: 24 us for 960x540) and the
// LDS turn. One lane per pixel with the per-parameter sums read from LDS (64 of a block's 256
// lanes busy in the layers, a scalar chain per parameter) took 2,553 us at 960x540, and the
// training step there 3.14 ms against 0.60 ms with this form.
// ---------------------------------------------------------------------------------------------
constexpr int kLpBwdBlocks = 240;
constexpr int kLpBwdWaves = 8;     // two waves per SIMD of the block's CU
constexpr int kLpRow = 17;         // LDS row of 16 pixels, padded by one bank

// one wave's 16 pixels, [unit][pixel]
struct LpTurn {
    float f[16][kLpRow];            // 12 features, then 1 (the bias column of layer 1), then 0
    float h1[kLpHid][kLpRow], h2[kLpHid][kLpRow], g1[kLpHid][kLpRow], g2[kLpHid][kLpRow];
    float go[16][kLpRow];           // 5 outputs, then 0
};
union LpBackwardLds {
    LpTurn turn[kLpBwdWaves];
    float sums[kLpBwdWaves][kLpParams];
};

typedef float lp_float4_a4 __attribute__((ext_vector_type(4), aligned(4)));

__device__ __forceinline__ float lp_q(float v) { return (float)(_Float16)v; }
__device__ __forceinline__ lp_float4 lp_mfma4(float a, float b, lp_float4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

__global__ __launch_bounds__(64 * kLpBwdWaves) void lp_mlp_backward_kernel(const float* __restrict__ P, long long N,
                                                                           const float* __restrict__ feat,
                                                                           const float* __restrict__ gScales,
                                                                           const float* __restrict__ scales,
                                                                           float* __restrict__ partial) {
    __shared__ LpBackwardLds lds;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int col = lane & 15, g = lane >> 4;
    // forward weight fragments (FP16), biases of the units this lane's D holds
    lp_half4 a1[2];
    lp_half8 a2[2], a3;
    lp_float4 b1v[2], b2v[2], b3v;
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
        const int u = mt * 16 + col;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int k = 4 * g + j;
            a1[mt][j] = (_Float16)(k < kLpIn ? P[kLpW1 + u * kLpIn + k] : 0.0f);
            a2[mt][j] = (_Float16)P[kLpW2 + u * kLpHid + k];
            a2[mt][4 + j] = (_Float16)P[kLpW2 + u * kLpHid + 16 + k];
            b1v[mt][j] = P[kLpB1 + mt * 16 + k];
            b2v[mt][j] = P[kLpB2 + mt * 16 + k];
        }
    }
    // the transposed weights of the gradient's way back, [unit of the layer below][unit], step (mt, v)
    float t3[2][4], t2[2][2][4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const int k = 4 * g + v;
        a3[v] = (_Float16)(col < kLpOut ? P[kLpW3 + col * kLpHid + k] : 0.0f);
        a3[4 + v] = (_Float16)(col < kLpOut ? P[kLpW3 + col * kLpHid + 16 + k] : 0.0f);
        b3v[v] = k < kLpOut ? P[kLpB3 + k] : 0.0f;
#pragma unroll
        for (int mo = 0; mo < 2; ++mo) {
            t3[mo][v] = k < kLpOut ? lp_q(P[kLpW3 + k * kLpHid + mo * 16 + col]) : 0.0f;
#pragma unroll
            for (int mt = 0; mt < 2; ++mt) t2[mo][mt][v] = lp_q(P[kLpW2 + (mt * 16 + k) * kLpHid + mo * 16 + col]);
        }
    }
    const lp_float4 zero = {0.f, 0.f, 0.f, 0.f};
    lp_float4 w1[2] = {zero, zero}, w2[2][2] = {{zero, zero}, {zero, zero}}, w3[2] = {zero, zero};
    lp_float4 sb2[2] = {zero, zero}, sb3 = zero;
    LpTurn& T = lds.turn[wave];
    const long long tiles = (N + 15) / 16;
    for (long long tile = (long long)blockIdx.x * kLpBwdWaves + wave; tile < tiles;
         tile += (long long)gridDim.x * kLpBwdWaves) {
        const long long p = tile * 16 + col;
        const bool in = p < N;
        lp_float4 f = zero;
        if (in && g < 3) f = *reinterpret_cast<const lp_float4_a4*>(feat + p * kLpIn + 4 * g);
        float gs[4], sc[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const bool on = in && 4 * g + v < kLpOut;
            const size_t e = (size_t)(4 * g + v) * N + p;
            gs[v] = on ? gScales[e] : 0.0f;
            sc[v] = on ? scales[e] : 0.0f;
        }
        lp_half4 bf;
#pragma unroll
        for (int j = 0; j < 4; ++j) bf[j] = (_Float16)f[j];
        lp_half8 q1, q2;
        lp_float4 d1[2], d2[2];
#pragma unroll
        for (int mt = 0; mt < 2; ++mt) {
            d1[mt] = __builtin_amdgcn_mfma_f32_16x16x16f16(a1[mt], bf, b1v[mt], 0, 0, 0);
#pragma unroll
            for (int v = 0; v < 4; ++v) q1[mt * 4 + v] = (_Float16)fmaxf(d1[mt][v], 0.0f);
        }
#pragma unroll
        for (int mt = 0; mt < 2; ++mt) {
            d2[mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a2[mt], q1, b2v[mt], 0, 0, 0);
#pragma unroll
            for (int v = 0; v < 4; ++v) q2[mt * 4 + v] = (_Float16)fmaxf(d2[mt][v], 0.0f);
        }
        const lp_float4 o = __builtin_amdgcn_mfma_f32_16x16x32_f16(a3, q2, b3v, 0, 0, 0);
        lp_float4 go;
#pragma unroll
        for (int v = 0; v < 4; ++v) go[v] = (o[v] > -kLpClamp && o[v] < kLpClamp) ? gs[v] * sc[v] : 0.0f;
        lp_float4 g2[2] = {zero, zero}, g1[2] = {zero, zero};
#pragma unroll
        for (int v = 0; v < 4; ++v)
#pragma unroll
            for (int mo = 0; mo < 2; ++mo) g2[mo] = lp_mfma4(t3[mo][v], go[v], g2[mo]);
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
#pragma unroll
            for (int v = 0; v < 4; ++v) g2[mt][v] = d2[mt][v] > 0.0f ? g2[mt][v] : 0.0f;
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
#pragma unroll
            for (int v = 0; v < 4; ++v)
#pragma unroll
                for (int mo = 0; mo < 2; ++mo) g1[mo] = lp_mfma4(t2[mo][mt][v], g2[mt][v], g1[mo]);
        // turn: [unit][pixel], written by pixel and read by unit (the wave's own rows: no barrier, the
        // LDS serves a wave's accesses in order)
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int u = mt * 16 + 4 * g + v;
                g1[mt][v] = d1[mt][v] > 0.0f ? g1[mt][v] : 0.0f;
                T.g1[u][col] = g1[mt][v];
                T.g2[u][col] = g2[mt][v];
                T.h1[u][col] = (float)q1[mt * 4 + v];
                T.h2[u][col] = (float)q2[mt * 4 + v];
            }
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            T.f[4 * g + v][col] = g < 3 ? (float)bf[v] : (v == 0 ? 1.0f : 0.0f);
            T.go[4 * g + v][col] = go[v];
        }
        sb2[0] += g2[0];
        sb2[1] += g2[1];
        sb3 += go;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int s = 0; s < 4; ++s) {  // pixels 4s + g
            const int px = 4 * s + g;
            const float bF = T.f[col][px], aO = T.go[col][px];
            const float h1a = T.h1[col][px], h1b = T.h1[16 + col][px], h2a = T.h2[col][px], h2b = T.h2[16 + col][px];
#pragma unroll
            for (int mt = 0; mt < 2; ++mt) {
                const float x1 = T.g1[mt * 16 + col][px], x2 = T.g2[mt * 16 + col][px];
                w1[mt] = lp_mfma4(x1, bF, w1[mt]);
                w2[mt][0] = lp_mfma4(x2, h1a, w2[mt][0]);
                w2[mt][1] = lp_mfma4(x2, h1b, w2[mt][1]);
            }
            w3[0] = lp_mfma4(aO, h2a, w3[0]);
            w3[1] = lp_mfma4(aO, h2b, w3[1]);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    }
    __syncthreads();
    // each parameter's sum of this wave; D[4g + v][col]
    float* S = lds.sums[wave];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const int r = 4 * g + v;
#pragma unroll
        for (int mt = 0; mt < 2; ++mt) {
            const int j = mt * 16 + r;
            if (col < kLpIn) S[kLpW1 + j * kLpIn + col] = w1[mt][v];
            if (col == kLpIn) S[kLpB1 + j] = w1[mt][v];
            S[kLpW2 + j * kLpHid + col] = w2[mt][0][v];
            S[kLpW2 + j * kLpHid + 16 + col] = w2[mt][1][v];
            if (r < kLpOut) S[kLpW3 + r * kLpHid + mt * 16 + col] = w3[mt][v];
            float b = sb2[mt][v];  // over the 16 pixel columns
#pragma unroll
            for (int d = 8; d > 0; d >>= 1) b += __shfl_xor(b, d, 16);
            if (col == 0) S[kLpB2 + j] = b;
        }
        float b = sb3[v];
#pragma unroll
        for (int d = 8; d > 0; d >>= 1) b += __shfl_xor(b, d, 16);
        if (col == 0 && r < kLpOut) S[kLpB3 + r] = b;
    }
    __syncthreads();
    for (int k = tid; k < kLpParams; k += 64 * kLpBwdWaves) {
        float s = 0.0f;
#pragma unroll
        for (int w = 0; w < kLpBwdWaves; ++w) s += lds.sums[w][k];
        partial[(size_t)blockIdx.x * kLpParams + k] = s;
    }
}

// grad += the blocks' partial sums: 16 parameters per block of 256, 16 lanes per parameter with every
// 16th block each, added in lane order. (One lane per parameter was a chain of 240 loads: 59 us.)
__global__ __launch_bounds__(256) void lp_reduce_kernel(const float* __restrict__ partial, int blocks,
                                                        float* __restrict__ grad) {
    __shared__ float part[16][17];
    const int kl = threadIdx.x & 15, j = threadIdx.x >> 4, k = blockIdx.x * 16 + kl;
    float s = 0.0f;
    if (k < kLpParams)
#pragma unroll 5
        for (int b = j; b < blocks; b += 16) s += partial[(size_t)b * kLpParams + k];
    part[j][kl] = s;
    __syncthreads();
    if (j == 0 && k < kLpParams) {
        s = 0.0f;
        for (int q = 0; q < 16; ++q) s += part[q][kl];
        grad[k] += s;
    }
}

}  // namespace luxgi

using namespace luxgi;

static bool lp_gbuf_ok(const LuxgiGBuffer* g) { return g && g->normals && g->pbr; }

extern "C" int luxgi_learned_pixel_scales(const float* params, int32_t W, int32_t H, const LuxgiGBuffer* cur,
                                          const float* color, const float* moments, float* scales, float* features,
                                          void* stream) {
    if (!params || W <= 0 || H <= 0 || !lp_gbuf_ok(cur) || !color || !moments || !scales)
        return LUXGI_ERR_INVALID_ARGUMENT;
    const long long N = (long long)W * H;
    if (N > (1ll << 30)) return LUXGI_ERR_UNSUPPORTED;
    hipLaunchKernelGGL(lp_forward_kernel, dim3((unsigned)((N + 255) / 256)), dim3(256), 0, as_stream(stream), params,
                       W, H, reinterpret_cast<const float4*>(color), reinterpret_cast<const float4*>(moments),
                       reinterpret_cast<const float4*>(cur->normals), reinterpret_cast<const float4*>(cur->pbr),
                       scales, features);
    LUXGI_LAUNCH_CHECK();
    return LUXGI_OK;
}

extern "C" size_t luxgi_learned_pixel_pass_backward_workspace_size(int32_t W, int32_t H) {
    if (W <= 0 || H <= 0) return 0;
    const size_t n = (size_t)W * H;
    return ((n * sizeof(float4) + 255) & ~size_t(255)) + n;
}

extern "C" int luxgi_learned_pixel_pass_backward(const LuxgiReflectionAtrousParams* p, int32_t W, int32_t H,
                                                 const LuxgiGBuffer* cur, const uint8_t* tileMap, const float* input,
                                                 const float* lumScale, const float* gradOut, float* gradIn,
                                                 float* gradScale, void* workspace, size_t workspaceBytes,
                                                 void* stream) {
    if (!p || W <= 0 || H <= 0 || !lp_gbuf_ok(cur) || !tileMap || !input || !lumScale || !gradOut || !gradIn ||
        !gradScale)
        return LUXGI_ERR_INVALID_ARGUMENT;
    if (p->radius < 0 || p->radius > 2) return LUXGI_ERR_UNSUPPORTED;
    if (p->stepSize < 1 || p->stepSize > (1 << 16)) return LUXGI_ERR_INVALID_ARGUMENT;
    if (gradIn == input || gradIn == gradOut) return LUXGI_ERR_INVALID_ARGUMENT;  // the gather reads both
    const size_t need = luxgi_learned_pixel_pass_backward_workspace_size(W, H);
    if (!workspace || workspaceBytes < need) return LUXGI_ERR_WORKSPACE_TOO_SMALL;
    const size_t n = (size_t)W * H;
    float4* record = static_cast<float4*>(workspace);
    uint8_t* mode = static_cast<uint8_t*>(workspace) + ((n * sizeof(float4) + 255) & ~size_t(255));
    LpPassArgs A{W, H, (W + 7) / 8, p->radius, p->stepSize, p->phiColor, p->phiNormal, p->sigmaDepth,
                 normal_squarings(p->phiNormal)};
    const dim3 grid((W + 15) / 16, (H + 15) / 16);
    hipStream_t st = as_stream(stream);
    const float4* nrm = reinterpret_cast<const float4*>(cur->normals);
    const float4* pbr = reinterpret_cast<const float4*>(cur->pbr);
    const float4* img = reinterpret_cast<const float4*>(input);
    const float4* go = reinterpret_cast<const float4*>(gradOut);
    const bool tiled = (long long)p->radius * p->stepSize <= kLpHalo;
    const int side = 16 + 2 * std::max(p->radius * std::min(p->stepSize, kLpHalo), 1);
    const size_t lds = tiled ? (size_t)side * side * sizeof(float4) : 0;
    hipLaunchKernelGGL(tiled ? lp_pass_centre_kernel<true> : lp_pass_centre_kernel<false>, grid, dim3(256), 2 * lds, st, A,
                       nrm, pbr, tileMap, img, lumScale, go, record, mode, gradScale);
    LUXGI_LAUNCH_CHECK();
    hipLaunchKernelGGL(tiled ? lp_pass_gather_kernel<true> : lp_pass_gather_kernel<false>, grid, dim3(256), 3 * lds, st, A,
                       nrm, pbr, img, go, record, mode, reinterpret_cast<float4*>(gradIn));
    LUXGI_LAUNCH_CHECK();
    return LUXGI_OK;
}

extern "C" size_t luxgi_learned_pixel_mlp_backward_workspace_size(void) {
    return (size_t)kLpBwdBlocks * kLpParams * sizeof(float);
}

extern "C" int luxgi_learned_pixel_mlp_backward(const float* params, int32_t W, int32_t H, const float* features,
                                                const float* scales, const float* gradScales, float* gradParams,
                                                void* workspace, size_t workspaceBytes, void* stream) {
    if (!params || W <= 0 || H <= 0 || !features || !scales || !gradScales || !gradParams)
        return LUXGI_ERR_INVALID_ARGUMENT;
    if (!workspace || workspaceBytes < luxgi_learned_pixel_mlp_backward_workspace_size())
        return LUXGI_ERR_WORKSPACE_TOO_SMALL;
    const long long N = (long long)W * H;
    hipStream_t st = as_stream(stream);
    float* partial = static_cast<float*>(workspace);
    hipLaunchKernelGGL(lp_mlp_backward_kernel, dim3(kLpBwdBlocks), dim3(64 * kLpBwdWaves), 0, st, params, N, features,
                       gradScales, scales, partial);
    LUXGI_LAUNCH_CHECK();
    hipLaunchKernelGGL(lp_reduce_kernel, dim3((kLpParams + 15) / 16), dim3(256), 0, st, partial, kLpBwdBlocks,
                       gradParams);
    LUXGI_LAUNCH_CHECK();
    return LUXGI_OK;
}
