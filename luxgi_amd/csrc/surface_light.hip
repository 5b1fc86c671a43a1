// surface_light.hip -- surface-cache lighting of the global surface atlas, for gfx950.
//
// Reference passes, all drawn as one quad per atlas tile (GlobalSurfaceAtlas.cpp:554-574)
// into the light cache and blended there (GlobalSurfaceAtlas.cpp:886-1085):
//   CopyEmissive.frag:22-27          light = emissive                       (blend none)
//   SDFDeferredLight.frag:79-130     light += direct(light l), per light l   (blend add)
//   SDFAtlasIndirectLight.frag:44-68 light += DDGI bounce                   (blend add)
// Here one kernel evaluates the sum per texel: two blocks per tile draw, each over its
// half of the tile in chunks of 512 texels. The quad covers the tile's full
// rect X..X+Wt-1 while the tile UV maps onto the rect minus its one-texel padding
// (extends.zw = (Wt - 1) / res, GlobalSurfaceAtlas.cpp:272-276), so texel p
// samples the G-buffer bilinearly at ((p + 0.5 - X) / Wt) * extends.zw + extends.xy,
// as the reference's fragments do. The direct term traces a shadow ray through
// the global SDF (tracyGlobalSDF with cascadeTraceStartBias 2,
// SDFDeferredLight.frag:104-112); the bounce is sampleIrradiance of the probe
// atlases (DDGICommon.glsl:163-233).
#include "probe_common.hpp"
#include "sdf_trace.hpp"

namespace luxgi {

constexpr int kMaxLights = 32;  // MAX_LIGHTS, Common/Light.glsl:30

struct SurfaceArgs {
    LuxgiSurfaceLightParams p;
    LuxgiGlobalSDFData g;
    LuxgiDDGIUniform u;
    AtlasGeom irrG, depG;
    ProbeReloc rl;
    int res;       // atlas resolution
    int sdfRes, mipRes, maxSteps;
    int indirect;  // probe atlases bound and the indirect pass requested
    int outHalf;
};

// bilinear, repeat addressing, all four channels (texture() with the default sampler)
template <class S>
__device__ __forceinline__ float4 bilinear_rgba(const S* __restrict__ img, int W, int H, float u, float v) {
    const float x = u * float(W) - 0.5f, y = v * float(H) - 0.5f;
    const float fx = floorf(x), fy = floorf(y);
    const float ax = x - fx, ay = y - fy;
    const int x0 = wrap_index(int(fx), W), x1 = wrap_index(int(fx) + 1, W);
    const int y0 = wrap_index(int(fy), H), y1 = wrap_index(int(fy) + 1, H);
    const float4 a = Texel<S>::ld4(img, (size_t)y0 * W + x0), b = Texel<S>::ld4(img, (size_t)y0 * W + x1);
    const float4 c = Texel<S>::ld4(img, (size_t)y1 * W + x0), d = Texel<S>::ld4(img, (size_t)y1 * W + x1);
    auto lerp2 = [&](float p, float q, float r, float s) {
        return (p * (1.0f - ax) + q * ax) * (1.0f - ay) + (r * (1.0f - ax) + s * ax) * ay;
    };
    return make_float4(lerp2(a.x, b.x, c.x, d.x), lerp2(a.y, b.y, c.y, d.y), lerp2(a.z, b.z, c.z, d.z),
                       lerp2(a.w, b.w, c.w, d.w));
}

// a . b with the fused products named. Near a mirror the BRDF divides by the square of cosLh^2 (a^2 - 1) + 1,
// which turns the last bit of the half vector's length into percents of the highlight: left to the compiler,
// the product that is rounded first, and with it the texel, depends on the code around the call.
__device__ __forceinline__ float dot_named(f3 a, f3 b) {
    return __builtin_fmaf(a.z, b.z, __builtin_fmaf(a.x, b.x, a.y * b.y));
}

// BRDF (Raytraced/BRDF.glsl:12-79, the 7-argument form, the half vector worked out here)
__device__ __forceinline__ f3 brdf_ggx(f3 albedo, f3 n, float rough, float metal, f3 view, f3 l) {
    const f3 s = l + view;
    const float len = sqrtf(dot_named(s, s));
    const f3 h = mk(s.x / len, s.y / len, s.z / len);
    const f3 F0 = mk(mixf(0.04f, albedo.x, metal), mixf(0.04f, albedo.y, metal), mixf(0.04f, albedo.z, metal));
    const float cosLi = fmaxf(0.0f, dot_named(n, l)), cosLh = fmaxf(0.0f, dot_named(n, h));
    const float NdotV = fmaxf(0.0f, dot_named(n, view));
    const float c = clampf(1.0f - fmaxf(dot_named(h, view), 0.0f), 0.0f, 1.0f);
    const float c5 = c * c * c * c * c;
    const f3 F = mk(F0.x + (1.0f - F0.x) * c5, F0.y + (1.0f - F0.y) * c5, F0.z + (1.0f - F0.z) * c5);
    const float alpha = rough * rough, a2 = alpha * alpha;
    const float denom = __builtin_fmaf(cosLh * cosLh, a2 - 1.0f, 1.0f);
    const float D = a2 / (kPiF * denom * denom);
    const float r = rough + 1.0f, k = r * r * 0.125f;
    const float G = cosLi / (cosLi * (1.0f - k) + k) * (NdotV / (NdotV * (1.0f - k) + k));
    const float spec = D * G / fmaxf(0.00001f, 4.0f * cosLi * NdotV);
    const float km = (1.0f - metal) * (1.0f / kPiF);
    return mk((1.0f - F.x) * km * albedo.x + F.x * spec, (1.0f - F.y) * km * albedo.y + F.y * spec,
              (1.0f - F.z) * km * albedo.z + F.z * spec);
}

// fetchLight (SDFDeferredLight.frag:41-76): types 0 directional, 1 spot, 2 point (Light.glsl:13-15)
__device__ __forceinline__ void fetch_light(const LuxgiLight& L, f3 wp, f3& Wi, float& tmax, float& atten) {
    Wi = mk(0.f, 0.f, 0.f);
    tmax = kGlobalSdfWorldSize;
    atten = 1.0f;
    const f3 lp = mk(L.position[0], L.position[1], L.position[2]);
    const f3 ld = mk(L.direction[0], L.direction[1], L.direction[2]);
    if (L.type == 0.0f) {
        Wi = mk(-ld.x, -ld.y, -ld.z);
    } else if (L.type == 2.0f) {
        const f3 dv = lp - wp;
        const float dist = len3(dv);
        Wi = normalize3(dv);
        atten = L.radius / (dist * dist + 1.0f);
        tmax = dist;
    } else if (L.type == 1.0f) {
        const f3 dv = lp - wp;
        const float cutoff = 1.0f - L.angle;
        Wi = normalize3(dv);
        const float dist = len3(dv);
        const float theta = dot3(Wi, ld);
        const float e = cutoff - cutoff * 0.9f;
        atten = (theta - cutoff) / e * (L.radius / (dist * dist + 1.0f));
        atten = clampf(atten, 0.0f, 1.0f);
        tmax = dist;
    }
}

// A chunk of a tile: up to kChunkTexels texels, one block. The shadow rays of the chunk's texels are
// gathered into a list first and marched 64 to a wave: with a ray per texel and light in its own lane,
// the lanes facing away from the light (about half of them) idle through their neighbours' march and
// each wave runs to the longest ray of every light in turn.
constexpr int kChunkTexels = 512;
constexpr int kRayLights = 4;  // lights whose rays fit the list together

struct SurfaceLds {
    LuxgiLight lights[kMaxLights];
    float wp[3][kChunkTexels], n[3][kChunkTexels];
    uint32_t visible[kChunkTexels];                // bit l: light l reaches the texel
    uint32_t rays[kChunkTexels * kRayLights];      // texel | light << 16
    uint32_t count;
};

// Shadow-ray march bound: the latency of its dependent lookups, so registers are held to 4 waves per
// SIMD (131 without the limit: 3 waves). 1,800 tiles of 40x40 texels, two lights and the bounce:
// 644 us with one lane per texel and light, 530 us with the list (4 waves without the list: 619).
template <class SS, int FL, class SA>
__global__ __launch_bounds__(256, 4) void surface_light_kernel(SurfaceArgs A, const LuxgiLight* __restrict__ lights,
                                                               const LuxgiAtlasTile* __restrict__ tiles, int numTiles,
                                                               const LuxgiSurfaceDraw* __restrict__ draws,
                                                               const __half* __restrict__ gbColor,
                                                               const __half* __restrict__ gbNormal,
                                                               const Unorm8* __restrict__ gbPbr,
                                                               const __half* __restrict__ gbEmissive, SdfView<SS> sdf,
                                                               const SA* __restrict__ irr, const SA* __restrict__ dep,
                                                               void* __restrict__ out) {
    __shared__ SurfaceLds sm;
    const LuxgiSurfaceDraw dr = draws[blockIdx.x];
    if (dr.tile >= (uint32_t)numTiles) return;  // uniform over the block
    const LuxgiAtlasTile& t = tiles[dr.tile];
    const float res = float(A.res);
    const int X = int(rintf(t.extends[0] * res)), Y = int(rintf(t.extends[1] * res));
    const int Wt = int(rintf(t.extends[2] * res)) + 1, Ht = int(rintf(t.extends[3] * res)) + 1;
    const int texels = Wt * Ht;
    const int chunks = (texels + kChunkTexels - 1) / kChunkTexels;
    if ((int)blockIdx.y >= chunks) return;  // uniform over the block
    const int per = ((texels + chunks - 1) / chunks + 63) & ~63;  // equal chunks of whole waves
    const int nl = (A.p.passes & LUXGI_SURFACE_DIRECT) ? A.p.numLights : 0;
    for (int i = threadIdx.x; i < nl; i += blockDim.x) sm.lights[i] = lights[i];
    const f3 cam = mk(A.p.cameraPosition[0], A.p.cameraPosition[1], A.p.cameraPosition[2]);
    const float sb = A.p.cameraPosition[3];
    // texel k of the tile: its atlas coordinate, and its place in the atlas
    auto place = [&](int k, int& px, int& py, float& au, float& av) {
        px = X + k % Wt;
        py = Y + k / Wt;
        au = ((float(px) + 0.5f - float(X)) / float(Wt)) * t.extends[2] + t.extends[0];
        av = ((float(py) + 0.5f - float(Y)) / float(Ht)) * t.extends[3] + t.extends[1];
        return px >= 0 && py >= 0 && px < A.res && py < A.res;
    };
    for (int c = blockIdx.y; c < chunks; c += gridDim.y) {
        const int k0 = c * per, cnt = min(per, texels - k0);
        __syncthreads();  // the previous chunk's LDS reads are done (and the lights are staged)
        for (int i = threadIdx.x; i < cnt && nl > 0; i += 256) {
            int px, py;
            float au, av;
            const bool on = place(k0 + i, px, py, au, av);
            f3 wp = mk(0.f, 0.f, 0.f), n = wp;
            if (on) {
                const float4 cc = bilinear_rgba<__half>(gbColor, A.res, A.res, au, av);
                const float4 nt = bilinear_rgba<__half>(gbNormal, A.res, A.res, au, av);
                n = oct_decode(nt.x, nt.y);
                wp = mk(cc.w, nt.z, nt.w);
            }
            sm.wp[0][i] = wp.x; sm.wp[1][i] = wp.y; sm.wp[2][i] = wp.z;
            sm.n[0][i] = n.x; sm.n[1][i] = n.y; sm.n[2][i] = n.z;
            sm.visible[i] = 0;
        }
        for (int l0 = 0; l0 < nl; l0 += kRayLights) {
            if (threadIdx.x == 0) sm.count = 0;
            __syncthreads();
            for (int i0 = 0; i0 < cnt; i0 += 256) {  // every lane takes part in the ballots
                const int i = i0 + threadIdx.x;
                for (int l = l0; l < min(nl, l0 + kRayLights); ++l) {
                    if (!((dr.lightMask >> l) & 1u)) continue;  // uniform over the block
                    bool ray = false;
                    if (i < cnt) {
                        f3 L;
                        float dist, atten;
                        fetch_light(sm.lights[l], mk(sm.wp[0][i], sm.wp[1][i], sm.wp[2][i]), L, dist, atten);
                        const float NoL = dot3(mk(sm.n[0][i], sm.n[1][i], sm.n[2][i]), L);
                        ray = NoL > 0.0f && atten > 0.0f;
                        if (NoL > 0.0f && !ray) sm.visible[i] |= 1u << l;  // this lane's own texel
                    }
                    const unsigned long long b = __ballot(ray);
                    uint32_t base = 0;
                    if ((threadIdx.x & 63) == 0 && b) base = atomicAdd(&sm.count, (uint32_t)__popcll(b));
                    base = (uint32_t)__shfl((int)base, 0);
                    if (ray)
                        sm.rays[base + __popcll(b & ((1ull << (threadIdx.x & 63)) - 1ull))] = (uint32_t)i | (uint32_t)l << 16;
                }
            }
            __syncthreads();
            const int rays = (int)sm.count;
            for (int r = threadIdx.x; r < rays; r += 256) {
                const uint32_t e = sm.rays[r];
                const int i = e & 0xffffu, l = e >> 16;
                const f3 wp = mk(sm.wp[0][i], sm.wp[1][i], sm.wp[2][i]), n = mk(sm.n[0][i], sm.n[1][i], sm.n[2][i]);
                f3 L;
                float dist, atten;
                fetch_light(sm.lights[l], wp, L, dist, atten);
                const float bias = 2.0f * sb * clampf(1.0f - dot3(n, L), 0.0f, 1.0f) + sb;
                const SdfHitTime h = trace_global_sdf<SS, FL>(sdf, A.g, wp + n * sb, L, dist - bias, 2.0f, A.maxSteps);
                if (!(h.time >= 0.0f)) atomicOr(&sm.visible[i], 1u << l);
            }
            __syncthreads();
        }
        for (int i = threadIdx.x; i < cnt; i += 256) {
            int px, py;
            float au, av;
            if (!place(k0 + i, px, py, au, av)) continue;
            f3 acc = mk(0.f, 0.f, 0.f);
            if (A.p.passes & LUXGI_SURFACE_EMISSIVE) {
                const float4 e = bilinear_rgba<__half>(gbEmissive, A.res, A.res, au, av);
                acc = mk(e.x, e.y, e.z);
            }
            if (nl > 0 || A.indirect) {
                const float4 cc = bilinear_rgba<__half>(gbColor, A.res, A.res, au, av);
                const float4 pbr = bilinear_rgba<Unorm8>(gbPbr, A.res, A.res, au, av);
                f3 n, wp;
                if (nl > 0) {
                    wp = mk(sm.wp[0][i], sm.wp[1][i], sm.wp[2][i]);
                    n = mk(sm.n[0][i], sm.n[1][i], sm.n[2][i]);
                } else {
                    const float4 nt = bilinear_rgba<__half>(gbNormal, A.res, A.res, au, av);
                    n = oct_decode(nt.x, nt.y);
                    wp = mk(cc.w, nt.z, nt.w);
                }
                const f3 view = normalize3(cam - wp);
                for (int l = 0; l < nl; ++l) {
                    if (!((dr.lightMask >> l) & 1u)) continue;
                    f3 L;
                    float dist, atten;
                    fetch_light(sm.lights[l], wp, L, dist, atten);
                    const float shadow = (sm.visible[i] >> l) & 1u ? 1.0f : 0.0f;
                    const float inten = __powf(sm.lights[l].intensity, 1.4f) + 0.1f;
                    const float* lc = sm.lights[l].color;
                    const f3 Lrad = mk(lc[0] * inten, lc[1] * inten, lc[2] * inten);
                    const float cosLi = fmaxf(0.0f, dot3(n, L));
                    const f3 b = brdf_ggx(mk(cc.x, cc.y, cc.z), n, pbr.y, pbr.x, view, L);
                    const float s = cosLi * shadow * atten;
                    acc = acc + mk(b.x * Lrad.x * s, b.y * Lrad.y * s, b.z * Lrad.z * s);
                }
                if (A.indirect) {
                    const float m = pbr.x;
                    const f3 alb = mk(fminf(cc.x, 0.9f), fminf(cc.y, 0.9f), fminf(cc.z, 0.9f));
                    const f3 diff = mk((alb.x - alb.x * m) / kPiF, (alb.y - alb.y * m) / kPiF, (alb.z - alb.z * m) / kPiF);
                    const f3 ir = sample_irradiance<SA>(A.u, A.irrG, A.depG, wp, n, view, irr, dep, A.rl);
                    acc = acc + mk(A.p.indirectIntensity * diff.x * ir.x, A.p.indirectIntensity * diff.y * ir.y,
                                   A.p.indirectIntensity * diff.z * ir.z);
                }
            }
            const size_t e = (size_t)py * A.res + px;
            const float4 o = make_float4(acc.x, acc.y, acc.z, 1.0f);
            if (A.outHalf) Texel<__half>::st4(static_cast<__half*>(out), e, o);
            else Texel<float>::st4(static_cast<float*>(out), e, o);
        }
    }
}

}  // namespace luxgi

using namespace luxgi;

template <class SS, int FL, class SA>
static void launch_surface(const SurfaceArgs& A, const LuxgiLight* lights, const LuxgiAtlasTile* tiles,
                           int numTiles, const LuxgiSurfaceDraw* draws, int numDraws, const LuxgiSurfaceGBuffer* gb,
                           const LuxgiSDFVolume* vol, const LuxgiProbeAtlas* probes, void* out, hipStream_t st) {
    const SdfView<SS> v = sdf_view<SS>(vol);
    // two blocks per tile share its chunks; one of them leaves at once when there is a single chunk
    hipLaunchKernelGGL((surface_light_kernel<SS, FL, SA>), dim3(numDraws, 2), dim3(256), 0, st, A, lights, tiles,
                       numTiles, draws, static_cast<const __half*>(gb->color), static_cast<const __half*>(gb->normal),
                       static_cast<const Unorm8*>(gb->pbr), static_cast<const __half*>(gb->emissive), v,
                       probes ? static_cast<const SA*>(probes->irradiance) : nullptr,
                       probes ? static_cast<const SA*>(probes->depth) : nullptr, out);
}

template <class SS, int FL>
static void launch_surface_sa(const SurfaceArgs& A, const LuxgiLight* lights, const LuxgiAtlasTile* tiles,
                              int numTiles, const LuxgiSurfaceDraw* draws, int numDraws, const LuxgiSurfaceGBuffer* gb,
                              const LuxgiSDFVolume* vol, const LuxgiProbeAtlas* probes, void* out, hipStream_t st) {
    if (probes && probes->storage == LUXGI_STORAGE_FP16)
        launch_surface<SS, FL, __half>(A, lights, tiles, numTiles, draws, numDraws, gb, vol, probes, out, st);
    else
        launch_surface<SS, FL, float>(A, lights, tiles, numTiles, draws, numDraws, gb, vol, probes, out, st);
}

extern "C" int luxgi_surface_light(const LuxgiSurfaceLightParams* params, const LuxgiLight* lights,
                                   const LuxgiAtlasTile* tiles, int32_t numTiles, const LuxgiSurfaceDraw* draws,
                                   int32_t numDraws,
                                   const LuxgiSurfaceGBuffer* gb, const LuxgiGlobalSDFData* sdfData,
                                   const LuxgiSDFVolume* vol, const LuxgiDDGIUniform* ddgi,
                                   const LuxgiProbeAtlas* probes, int32_t outStorage, void* lightCache,
                                   void* stream) {
    if (!params || !gb || !lightCache || numDraws < 0) return LUXGI_ERR_INVALID_ARGUMENT;
    if (params->passes & ~(LUXGI_SURFACE_EMISSIVE | LUXGI_SURFACE_DIRECT | LUXGI_SURFACE_INDIRECT))
        return LUXGI_ERR_INVALID_ARGUMENT;
    if (outStorage != LUXGI_STORAGE_FP32 && outStorage != LUXGI_STORAGE_FP16) return LUXGI_ERR_UNSUPPORTED;
    if (gb->resolution <= 0 || (size_t)gb->resolution * gb->resolution >= (1ull << 31)) return LUXGI_ERR_INVALID_ARGUMENT;
    if (numDraws == 0) return LUXGI_OK;
    if (!tiles || !draws || numTiles <= 0) return LUXGI_ERR_INVALID_ARGUMENT;
    const bool direct = (params->passes & LUXGI_SURFACE_DIRECT) && params->numLights > 0;
    const bool indirect = (params->passes & LUXGI_SURFACE_INDIRECT) != 0;
    if ((params->passes & LUXGI_SURFACE_EMISSIVE) && !gb->emissive) return LUXGI_ERR_INVALID_ARGUMENT;
    if ((direct || indirect) && (!gb->color || !gb->normal || !gb->pbr)) return LUXGI_ERR_INVALID_ARGUMENT;
    if (params->numLights < 0 || params->numLights > LUXGI_MAX_LIGHTS) return LUXGI_ERR_INVALID_ARGUMENT;
    if (direct) {
        if (!lights) return LUXGI_ERR_INVALID_ARGUMENT;
        const int st = sdf_volume_status(sdfData, vol);
        if (st != LUXGI_OK) return st;
        if (vol->storage == LUXGI_STORAGE_BF16) return LUXGI_ERR_UNSUPPORTED;  // BF16: the probe-ray trace only
    }
    if (indirect) {
        if (!ddgi || !probes || !probes->irradiance || !probes->depth) return LUXGI_ERR_INVALID_ARGUMENT;
        if (probes->storage != LUXGI_STORAGE_FP32 && probes->storage != LUXGI_STORAGE_FP16)
            return LUXGI_ERR_UNSUPPORTED;
        if (!probe_atlas_geometry_valid(*ddgi)) return LUXGI_ERR_INVALID_ARGUMENT;
    }
    SurfaceArgs A{};
    A.p = *params;
    if (!direct) A.p.numLights = 0;
    if (direct) A.g = *sdfData;
    if (indirect) {
        A.u = *ddgi;
        A.irrG = atlas_geom(ddgi->irradianceTextureWidth, ddgi->irradianceTextureHeight, ddgi->irradianceProbeSideLength);
        A.depG = atlas_geom(ddgi->depthTextureWidth, ddgi->depthTextureHeight, ddgi->depthProbeSideLength);
    }
    A.res = gb->resolution;
    A.maxSteps = params->maxSteps > 0 ? params->maxSteps : 250;
    A.indirect = indirect ? 1 : 0;
    A.outHalf = outStorage == LUXGI_STORAGE_FP16 ? 1 : 0;
    hipStream_t st = as_stream(stream);
    const LuxgiSDFVolume* v = direct ? vol : nullptr;
    const LuxgiProbeAtlas* pr = indirect ? probes : nullptr;
    A.rl = probe_reloc(pr);
    const bool half = v && v->storage == LUXGI_STORAGE_FP16;
    const int layout = v ? v->layout : LUXGI_LAYOUT_LINEAR;
#define LUXGI_SURFACE_LAUNCH(SS_, FL_) \
    launch_surface_sa<SS_, FL_>(A, lights, tiles, numTiles, draws, numDraws, gb, v, pr, lightCache, st)
    if (layout == LUXGI_LAYOUT_BRICK4) {
        if (half) LUXGI_SURFACE_LAUNCH(__half, LUXGI_LAYOUT_BRICK4);
        else LUXGI_SURFACE_LAUNCH(float, LUXGI_LAYOUT_BRICK4);
    } else if (layout == LUXGI_LAYOUT_CELL8) {
        if (half) LUXGI_SURFACE_LAUNCH(__half, LUXGI_LAYOUT_CELL8);
        else LUXGI_SURFACE_LAUNCH(float, LUXGI_LAYOUT_CELL8);
    } else {
        if (half) LUXGI_SURFACE_LAUNCH(__half, LUXGI_LAYOUT_LINEAR);
        else LUXGI_SURFACE_LAUNCH(float, LUXGI_LAYOUT_LINEAR);
    }
#undef LUXGI_SURFACE_LAUNCH
    LUXGI_LAUNCH_CHECK();
    return LUXGI_OK;
}
