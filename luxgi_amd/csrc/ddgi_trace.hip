// ddgi_trace.hip -- DDGI probe rays through the global SDF with surface-atlas
// radiance at the hits, for gfx950.
//
// Reference: Shaders/DDGI/GISDFRays.comp:63-128 (ray generation and encode),
// Shaders/SDF/SDFCommon.glsl:98-194 (tracyGlobalSDF), :64-71 (cascade UV),
// :84-95 (lineHitAABB), :196-199 (surface threshold),
// Shaders/SDF/AtlasCommon.glsl:50-157 (surface-atlas lookup);
// host dispatch Engine/DDGI/DDGIRenderer.cpp:304-321.
//
// One lane per ray; the 64 lanes of a wave trace 64 rays of the same probe, so
// early march steps of a wave read neighbouring voxels. The reference inverts
// each candidate object's transform per hit (AtlasCommon.glsl:134); here the
// inverses are computed once per call into the workspace (trace_prepare_kernel).
// The march (march_kernel) and the per-hit work (shade_kernel) are separate
// launches, so the march loop carries only the registers it needs. The march
// stores everything that needs no atlas lookup: the final results of misses and
// inside hits, and the direction and distance of the front hits. The shade adds
// the front hits' radiance.
#include "atlas_sample.hpp"
#include "sdf_trace.hpp"

#include <algorithm>
#include <type_traits>

namespace luxgi {

constexpr float kWorldSize = 60000.0f;  // GLOBAL_SDF_WORLD_SIZE, SDFCommon.glsl:6

// Everything a trace reads about its scene: the global SDF (clipmap data, fine volume, coarse mip and
// their options), the surface atlas with its object/tile/chunk buffers, and the sky. A single call
// (or a batch over one scene) carries one in TraceArgs; a batch over several scenes indexes an
// array of them in device memory (LuxgiTraceScene, the same fields).
struct TraceScene {
    LuxgiGlobalSDFData g;
    LuxgiSurfaceAtlasData ad;
    const void* sdf;
    const void* mip;
    const float* guard;       // optional brick guard (FP32 volumes)
    const float* brickScale;  // optional per-brick scale of a BRICK4 fine volume
    const float* refine;      // optional FP32 fine volume re-evaluated at hits
    const uint32_t* chunks;
    const uint32_t* culled;
    const LuxgiAtlasObject* objects;
    const LuxgiAtlasTile* tiles;
    const void* color;
    const float* atlasDepth;
    const float* skyFaces;
    long long objectStart;    // the scene's first object in the inverse-transform workspace
    int objectCapacity;       // entries of `objects`
    float sky[3];
    float invCascades;        // 1 / cascadesCount
    int res, mipRes, skySize, refineLayout;
};

struct TraceArgs {
    TraceScene scene;              // the scene of a single call or of a one-scene batch
    const TraceScene* scenes;      // a several-scene batch: per-volume scenes (device memory)
    int maxSteps, P, R, rayWidth;
    float hitEps;
    int fineLayout;                // LuxgiLayout of the fine volume (the kernels' template argument)
    int waveRays;                  // rays per wave: 64, or 16 where few rays leave the chip idle
    LuxgiTraceVolume vol;          // the volume of a single-volume call
    const LuxgiTraceVolume* vols;  // the volumes of a batched call (device memory), their count
    int nVols;                     // and the total of their rays
    long long totalRays;
};

// ---------------------------------------------------------------------------
// March (tracyGlobalSDF, SDFCommon.glsl:98-194): one lane per ray, the 64 lanes
// of a wave on 64 rays of one probe, in trace_block's order. A front hit's record (hitTime, texture
// UV of the hit step; cascade) goes to the workspace for shade_kernel.
// ---------------------------------------------------------------------------

__device__ __forceinline__ void ray_setup(const TraceArgs& A, const LuxgiTraceVolume& v, int probe, int ray,
                                          f3& origin, f3& dir) {
    // probeLocation (DDGICommon.glsl:106-114) + GISDFRays.comp:72-73
    const LuxgiDDGIUniform& u = v.uniform;
    const int px = u.probeCounts[0], pxy = u.probeCounts[0] * u.probeCounts[1];
    const int gx = probe % px, gy = (probe % pxy) / px, gz = probe / pxy;
    origin = mk(u.step[0] * float(gx) + u.startPosition[0], u.step[1] * float(gy) + u.startPosition[1],
                u.step[2] * float(gz) + u.startPosition[2]);
    if (v.probeOffsets) {
        const float4 o = reinterpret_cast<const float4*>(v.probeOffsets)[probe];
        origin = origin + mk(o.x, o.y, o.z);
    }
    const f3 sf = spherical_fibonacci(float(ray), float(u.raysPerProbe));
    const float* rot = v.deviceOrientation ? v.deviceOrientation : v.orientation;  // column-major 4x4
    float m[9];
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int r = 0; r < 3; ++r) m[c * 3 + r] = rot[c * 4 + r];
    dir = normalize3(mk(m[0] * sf.x + m[3] * sf.y + m[6] * sf.z, m[1] * sf.x + m[4] * sf.y + m[7] * sf.z,
                        m[2] * sf.x + m[5] * sf.y + m[8] * sf.z));
}

// the volume of flat ray `gid` in a batch: the last whose rayStart <= gid
__device__ __forceinline__ int trace_volume_of(const LuxgiTraceVolume* __restrict__ vols, int n, long long gid) {
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (vols[mid].rayStart <= gid) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// fine-volume lookup in the volume's layout (FL: LuxgiLayout)
template <class SS, int FL>
__device__ __forceinline__ float fine_lookup(const SS* __restrict__ sdf, const float* __restrict__ scale, int W, int H,
                                             int D, float u, float v, float w) {
    if constexpr (FL == LUXGI_LAYOUT_BRICK4) return sample3d_brick4<SS>(sdf, W, H, D, u, v, w, scale);
    else if constexpr (FL == LUXGI_LAYOUT_CELL8) return sample3d_cell8<SS>(sdf, W, H, D, u, v, w);
    else return sample_volume<SS>(sdf, W, H, D, u, v, w);
}

// coarse-mip lookup: CELL8 records with a CELL8 volume, linear otherwise
template <class SS, int FL>
__device__ __forceinline__ float mip_lookup(const SS* __restrict__ mip, int W, int H, int D, float u, float v,
                                            float w) {
    if constexpr (FL == LUXGI_LAYOUT_CELL8) return sample3d_cell8<SS>(mip, W, H, D, u, v, w);
    else return sample_volume<SS>(mip, W, H, D, u, v, w);
}

// the FP32 re-evaluation volume, in its own layout
__device__ __forceinline__ float refine_lookup(const TraceArgs& A, const TraceScene& S, int W, int H, int D, float u, float v, float w) {
    if (S.refineLayout == LUXGI_LAYOUT_BRICK4) return sample3d_brick4<float>(S.refine, W, H, D, u, v, w);
    if (S.refineLayout == LUXGI_LAYOUT_CELL8) return sample3d_cell8<float>(S.refine, W, H, D, u, v, w);
    return sample_volume<float>(S.refine, W, H, D, u, v, w);
}

// Result of a ray without an atlas lookup (GISDFRays.comp:93-96,121-124): an inside hit stores
// zero radiance, a miss the sky in its direction; both store the world distance.
template <class SR>
__device__ __forceinline__ void store_nonhit(const TraceArgs& A, const TraceScene& S, const float* __restrict__ skyFaces,
                                             SR* __restrict__ outRad, SR* __restrict__ outDD,
                                             uint8_t* __restrict__ flags, size_t e, f3 dir, bool inside) {
    float4 rad = make_float4(0.f, 0.f, 0.f, 0.f);
    if (!inside) {
        const float3 s = skyFaces ? sample_cube(skyFaces, S.skySize, dir) : make_float3(S.sky[0], S.sky[1], S.sky[2]);
        rad = make_float4(s.x, s.y, s.z, 0.f);
    }
    Texel<SR>::st4(outRad, e, rad);
    Texel<SR>::st4(outDD, e, make_float4(dir.x, dir.y, dir.z, kWorldSize));
    if (flags) flags[e] = inside ? 2 : 0;
}

// State of one ray's sphere trace (SDFCommon.glsl:98-171), advanced one step at a time.
struct MarchRay {
    f3 o, d, traceEnd;
    f3 cpos;             // the current cascade's centre
    float half, voxel;   // and its half extent and voxel size
    float invExtent, invVoxel;  // 1 / (2 half) and 1 / voxel (see march_step)
    float stepTime, iy, nextStart;
    int cas, step;
};

// lineHitAABB (SDFCommon.glsl:84-95) and the entry into cascade r.cas (:121-141)
__device__ __forceinline__ void march_enter(const TraceArgs& A, const TraceScene& S, MarchRay& r, float traceMax) {
    const int cas = r.cas;
    r.cpos = mk(S.g.cascadePosDistance[cas][0], S.g.cascadePosDistance[cas][1], S.g.cascadePosDistance[cas][2]);
    r.half = S.g.cascadePosDistance[cas][3];
    r.voxel = S.g.cascadeVoxelSize[cas];
    r.invExtent = 1.0f / (r.half * 2.0f);
    r.invVoxel = 1.0f / r.voxel;
    const float half = r.half;
    const f3 dl = r.traceEnd - r.o;
    const f3 inv = mk(1.0f / dl.x, 1.0f / dl.y, 1.0f / dl.z);
    const f3 en = (r.cpos - mk(half, half, half) - r.o) * inv;
    const f3 ex = (r.cpos + mk(half, half, half) - r.o) * inv;
    float ix = fmaxf(fminf(en.x, ex.x), fmaxf(fminf(en.y, ex.y), fminf(en.z, ex.z)));
    float iy = fminf(fmaxf(en.x, ex.x), fminf(fmaxf(en.y, ex.y), fmaxf(en.z, ex.z)));
    ix = clampf(ix, 0.0f, 1.0f) * traceMax;
    iy = clampf(iy, 0.0f, 1.0f) * traceMax;
    ix = fmaxf(ix, r.nextStart);
    r.stepTime = ix;
    if (ix >= iy) r.stepTime = iy;
    else r.nextStart = iy;
    r.iy = iy;
    r.step = 0;
}

__device__ __forceinline__ void march_begin(const TraceArgs& A, const TraceScene& S, const LuxgiTraceVolume& v, int probe, int ray,
                                            float traceMax, MarchRay& r) {
    ray_setup(A, v, probe, ray, r.o, r.d);
    r.traceEnd = r.o + r.d * traceMax;
    r.nextStart = 0.0f;
    r.cas = 0;
    march_enter(A, S, r, traceMax);
}

// One step of cascade r.cas (the body of SDFCommon.glsl:143-170). Returns true on a hit and fills
// the hit record; otherwise advances stepTime.
template <class SS, int FL, bool COUNT>
__device__ __forceinline__ bool march_step(const TraceArgs& A, const TraceScene& S, const SS* __restrict__ sdf, const SS* __restrict__ mip,
                                           const float* __restrict__ guard, MarchRay& r, float4& ra, float2& rb,
                                           unsigned long long& cMip, unsigned long long& cFine) {
    const int C = (int)S.g.cascadesCount;
    const float chunkSizeDistance = 32.0f / S.g.resolution;
    const float chunkMarginDistance = 4.0f / S.g.resolution;
    const int texW = S.res * C, mipW = S.mipRes * C;
    // The cascade UV (SDFCommon.glsl:64-71) divides by the cascade extent and the cascade count, and
    // the hit thickness (:166-167) by the voxel size; those divisors are fixed per cascade, so the
    // divisions are multiplications by their reciprocals: identical results when the divisor is a
    // power of two (extents of 2^k, one, two or four cascades), within one ulp otherwise (GLSL's
    // own division is within 2.5 ulp).
    const float cmax = r.half * 2.0f;
    const float stepTime = r.stepTime;
    const f3 p = r.o + r.d * stepTime;
    const float ux = clampf((p.x - r.cpos.x) * r.invExtent + 0.5f, 0.0f, 1.0f);
    const float uy = clampf((p.y - r.cpos.y) * r.invExtent + 0.5f, 0.0f, 1.0f);
    const float uz = clampf((p.z - r.cpos.z) * r.invExtent + 0.5f, 0.0f, 1.0f);
    const float tx = (float(r.cas) + ux) * S.invCascades;
    // The fine sample is used only where the mip distance is below the chunk size and the fine
    // distance below twice the chunk margin (SDFCommon.glsl:150-162). A brick guard >= that margin
    // proves the second test fails for every voxel of the footprint (trilinear filtering is a
    // convex combination), so the fine lookup is skipped; the factor 1 + 1e-5 covers fp32
    // rounding of the filter.
    bool needFine = true;
    if (guard) {
        const int gx = clampi(int(floorf(tx * float(texW) - 0.5f)), 0, texW - 1);
        const int gy = clampi(int(floorf(uy * float(S.res) - 0.5f)), 0, S.res - 1);
        const int gz = clampi(int(floorf(uz * float(S.res) - 0.5f)), 0, S.res - 1);
        const float gv = guard[((size_t)(gz >> 2) * (S.res >> 2) + (gy >> 2)) * (texW >> 2) + (gx >> 2)];
        needFine = !(gv >= chunkMarginDistance * 2.0f * (1.0f + 1e-5f));
    }
    const float sm = mip_lookup<SS, FL>(mip, mipW, S.mipRes, S.mipRes, tx, uy, uz);
    float sd = sm;
    float st = 1.0f;
    if (needFine) st = fine_lookup<SS, FL>(sdf, S.brickScale, texW, S.res, S.res, tx, uy, uz);
    if (COUNT) cMip++;
    if (sd < chunkSizeDistance) {
        if (COUNT) cFine++;
        if (needFine && st < chunkMarginDistance * 2.0f) sd = st;
    } else {
        sd = chunkSizeDistance;
    }
    sd *= cmax;
    const float voxel = r.voxel;
    const float thick = A.hitEps > 0.0f ? A.hitEps : voxel * 0.5f * clampf(stepTime * r.invVoxel, 0.0f, 1.0f);
    if (sd < thick) {
        if (S.refine) {  // FP32 re-evaluation of the hit step, same selection rule
            const float f32 = refine_lookup(A, S, texW, S.res, S.res, tx, uy, uz);
            const float s32 = sm < chunkSizeDistance ? (f32 < chunkMarginDistance * 2.0f ? f32 : sm)
                                                     : chunkSizeDistance;
            sd = s32 * cmax;
        }
        ra = make_float4(fmaxf(stepTime + sd - thick, 0.0f), tx, uy, uz);
        rb = make_float2(sd, float(r.cas));
        return true;
    }
    r.stepTime = stepTime + fmaxf(sd, voxel);
    return false;
}

// What a finished ray leaves: a front hit its direction, distance and flag (GISDFRays.comp:121-127) and
// its record for the shade; any other ray its final result and a record without a hit. `end` is the
// end of the march: (hit time or < 0, texture UV), `rb` (distance, cascade).
template <class SR>
__device__ __forceinline__ void march_finish(const TraceArgs& A, const TraceScene& S, const LuxgiTraceVolume& v,
                                             const MarchRay& r, float4 end, float2 rb, int probe, int ray, size_t rid,
                                             float4* __restrict__ recA, uint8_t* __restrict__ recC) {
    SR* outRad = static_cast<SR*>(v.rays.radiance);
    SR* outDD = static_cast<SR*>(v.rays.directionDistance);
    const size_t e = (size_t)probe * v.rays.width + ray;
    const bool inside = end.x >= 0.0f && rb.x <= 0.0f && end.x <= S.g.cascadeVoxelSize[0];
    if (end.x >= 0.0f && !inside) {
        const int cas = int(rb.y);
        const float dist = fmaxf(end.x + S.g.cascadeVoxelSize[cas] * 0.5f, 0.0f);
        Texel<SR>::st4(outDD, e, make_float4(r.d.x, r.d.y, r.d.z, dist));
        if (v.rayFlags) v.rayFlags[e] = 1;
        recC[rid] = (uint8_t)cas;
    } else {
        store_nonhit<SR>(A, S, S.skyFaces, outRad, outDD, v.rayFlags, e, r.d, inside);
        end.x = -1.0f;
    }
    recA[rid] = end;
}

__device__ __forceinline__ float trace_max_distance(const TraceArgs& A, const TraceScene& S) {
    return fminf(kWorldSize, S.g.cascadePosDistance[(int)S.g.cascadesCount - 1][3] * 2.0f);
}

// The sphere trace of one ray (SDFCommon.glsl:98-171) through its cascades.
template <class SS, class SR, bool COUNT, int FL>
__device__ __forceinline__ void march_ray(const TraceArgs& A, const TraceScene& S, const LuxgiTraceVolume& v,
                                          int probe, int ray, size_t rid, float4* __restrict__ recA,
                                          uint8_t* __restrict__ recC, unsigned long long& cMip,
                                          unsigned long long& cFine, unsigned long long& cSteps,
                                          unsigned long long& cHits) {
    const SS* sdf = static_cast<const SS*>(S.sdf);
    const SS* mip = static_cast<const SS*>(S.mip);
    const int C = (int)S.g.cascadesCount;
    const float traceMax = trace_max_distance(A, S);
    MarchRay r;
    march_begin(A, S, v, probe, ray, traceMax, r);
    float4 ra = make_float4(-1.0f, 0.f, 0.f, 0.f);
    float2 rb = make_float2(0.f, 0.f);
    for (;;) {
        int step = 0;
        bool hit = false;
        for (; step < A.maxSteps && r.stepTime < r.iy; ++step)
            if (march_step<SS, FL, COUNT>(A, S, sdf, mip, S.guard, r, ra, rb, cMip, cFine)) {
                hit = true;
                break;
            }
        if (COUNT) cSteps += step;
        if (hit || ++r.cas >= C) break;
        march_enter(A, S, r, traceMax);
    }
    if (COUNT && ra.x >= 0.0f) cHits++;
    march_finish<SR>(A, S, v, r, ra, rb, probe, ray, rid, recA, recC);
}

// The volume of flat ray `gid` of a batch (MODE 1: one scene, MODE 2: a scene per volume). In MODE
// 2 the volumes' ray ranges start at multiples of 64 (luxgi_ddgi_trace_scenes_prepare), so a wave
// lies in one volume: the search runs on the wave's first ray and the volume and scene
// descriptors are read as wave-uniform data.
template <int MODE>
__device__ __forceinline__ int batch_volume(const TraceArgs& A, long long gid) {
    if constexpr (MODE == 2) {
        const int w0 = __builtin_amdgcn_readfirstlane((int)(gid & ~63ll));
        return __builtin_amdgcn_readfirstlane(trace_volume_of(A.vols, A.nVols, w0));
    } else {
        return trace_volume_of(A.vols, A.nVols, gid);
    }
}

__device__ __forceinline__ long long volume_rays(const LuxgiTraceVolume& v) {
    return (long long)v.uniform.probeCounts[0] * v.uniform.probeCounts[1] * v.uniform.probeCounts[2] *
           v.uniform.raysPerProbe;
}

// The ray of flat lane `gid`: false past the rays. MODE 0 (one volume): 64 rays of one probe per wave
// (rays padded to a multiple of 64 per probe). MODE 1 and 2 (batches over one scene / a scene per
// volume): the flat ray list of all volumes, each ray finding its volume by rayStart; a ray past its
// volume's rays (padding, or a stale totalRays) does nothing.
template <int MODE>
__device__ __forceinline__ bool find_ray(const TraceArgs& A, long long gid, const LuxgiTraceVolume*& v, int& probe,
                                         int& ray, size_t& rid) {
    if constexpr (MODE == 0) {
        const int Rp = (A.R + 63) & ~63;
        v = &A.vol;
        probe = int(gid / Rp);
        ray = int(gid % Rp);
        rid = (size_t)probe * A.R + ray;
        return probe < A.P && ray < A.R;
    } else {
        v = &A.vols[batch_volume<MODE>(A, gid)];
        const int R = v->uniform.raysPerProbe;
        const long long local = gid - v->rayStart;
        probe = int(local / R);
        ray = int(local % R);
        rid = (size_t)gid;
        return gid < A.totalRays && local >= 0 && local < volume_rays(*v);
    }
}

// The block of rays of a launched block. The dispatcher deals blocks to the 8 XCDs in turn (block b runs on
// XCD b % 8). Each XCD takes kXcdRun blocks in a row (65,536 rays; 256 probes of 256 rays), whose SDF lines
// stay in its L2, and the next run lies 8 runs on, so at any time the XCDs walk neighbouring probes and share
// what they read from the memory side. With one eighth of the volume per XCD they walk eight distant slabs
// and end unevenly: 32x16x32 probes x 256 rays 1,518 us against 1,350 (runs of 8, 32, 128, 512, 1,024 blocks:
// 1,445, 1,455, 1,482, 1,355, 1,394; probes in 4^3 or 8^3 cubes: 1,444, 1,369). The blocks after the last
// whole turn go in eighths, and so does a launch below two turns (1,048,576 rays): 32x8x16x144 in FP16, one turn
// and a half, 124 us in eighths against 130, 13x7x11x100 68 against 70 undealt; from two turns on runs are the
// faster, 16x16x16x256 441 -> 420, 17x9x31x256 linear FP16 366 -> 346, 32x32x32x64 linear 675 -> 609.
constexpr int kXcdRun = 256;
__device__ __forceinline__ long long trace_block() {
    constexpr uint32_t turn = kXcds * kXcdRun;
    const uint32_t b = blockIdx.x, whole = gridDim.x < 2 * turn ? 0 : gridDim.x / turn * turn;
    if (b >= whole) return whole + xcd_block(b - whole, gridDim.x - whole);
    const uint32_t r = b % turn;
    return b - r + r % kXcds * kXcdRun + r / kXcds;
}

// Flat lane of this thread's ray: each wave has A.waveRays of them, one per lane from lane 0.
__device__ __forceinline__ bool lane_traces(const TraceArgs& A) { return (int)(threadIdx.x & 63) < A.waveRays; }
__device__ __forceinline__ long long wave_ray(const TraceArgs& A) {
    const int lane = threadIdx.x & 63;
    return (trace_block() * 4 + (threadIdx.x >> 6)) * A.waveRays + min(lane, A.waveRays - 1);
}

// Sphere trace of one ray per lane.
template <class SS, class SR, bool COUNT, int FL, int MODE>
__global__ __launch_bounds__(256) void march_kernel(TraceArgs A, float4* __restrict__ recA, uint8_t* __restrict__ recC,
                                                    unsigned long long* __restrict__ counters) {
    const long long gid = wave_ray(A);
    unsigned long long cMip = 0, cFine = 0, cSteps = 0, cHits = 0;
    const LuxgiTraceVolume* v;
    int probe, ray;
    size_t rid;
    if (find_ray<MODE>(A, gid, v, probe, ray, rid) && lane_traces(A))
        march_ray<SS, SR, COUNT, FL>(A, MODE == 2 ? A.scenes[v->scene] : A.scene, *v, probe, ray, rid, recA, recC, cMip,
                                     cFine, cSteps, cHits);
    if (COUNT) {  // lanes without a count stay away from the LDS atomics, which serialise
        __shared__ unsigned long long sc[4];
        if (threadIdx.x < 4) sc[threadIdx.x] = 0;
        __syncthreads();
        if (cMip) atomicAdd(&sc[0], cMip);
        if (cFine) atomicAdd(&sc[1], cFine);
        if (cSteps) atomicAdd(&sc[2], cSteps);
        if (cHits) atomicAdd(&sc[3], cHits);
        __syncthreads();
        if (threadIdx.x == 0) {
            atomicAdd(&counters[0], sc[0]);
            atomicAdd(&counters[1], sc[1]);
            atomicAdd(&counters[6], sc[2]);
            atomicAdd(&counters[7], sc[3]);
        }
    }
}

// Radiance of the front hits (SDFCommon.glsl:172-184, GISDFRays.comp:89-119). A wave takes the 64 rays the
// march's wave traced: first one ray per lane, the hit point, the normal and the chunk's object list,
// then eight lanes per hit, eight hits at a time (sample_atlas_wave).
// One lane per hit, with the hits counting-sorted by chunk so that a wave's lists agree, took
// 479 us for the 2.4 M hits of a 32x16x32x256 volume and 300 us more for the sort: its keys, a
// histogram with an atomic per chunk of each wave, a scan, a scatter, and records and outputs at
// scattered addresses. The whole trace took 1,652 us so and 1,513 in this form (shade 487), before
// trace_block's runs made it 1,350; a 13x7x11x100 volume in FP16 102 and 68, an 8x8x8x64 one 120 and 90, before
// kFewRays made the last 67. Bound at the large size: L2 misses (19.6 M lines in 487 us, 5.1 TB/s), a third
// of them the normals'.
template <class SS, class SC, class SR, bool COUNT, int MODE>
__global__ __launch_bounds__(256) void shade_kernel(TraceArgs A, const float* __restrict__ objInvBase,
                                                    const float4* __restrict__ recA, const uint8_t* __restrict__ recC,
                                                    unsigned long long* __restrict__ counters) {
    __shared__ AtlasQueryLds lds[4];
    const long long gid = wave_ray(A);
    Counts c{};
    const LuxgiTraceVolume* v;
    int probe, ray;
    size_t rid;
    const bool valid = find_ray<MODE>(A, gid, v, probe, ray, rid) && lane_traces(A);
    const TraceScene& S = MODE == 2 ? A.scenes[v->scene] : A.scene;
    float4 ra = make_float4(-1.f, 0.f, 0.f, 0.f);
    if (valid) ra = recA[rid];
    const bool hit = ra.x >= 0.0f;
    uint32_t list = 0, count = 0;
    f3 hp = mk(0.f, 0.f, 0.f), n = hp;
    float thr = 0.0f;
    if (hit) {
        f3 origin, dir;
        ray_setup(A, *v, probe, ray, origin, dir);
        hp = origin + dir * ra.x;
        atlas_list(S.ad, S.chunks, S.culled, hp, list, count);
        thr = S.g.cascadeVoxelSize[recC[rid]] * 1.05f;
        const SS* sdf = static_cast<const SS*>(S.sdf);
        const int texW = S.res * (int)S.g.cascadesCount;
        const float o = 1.0f / S.g.resolution;
        const float tx = ra.y, uy = ra.z, uz = ra.w;
        auto nl = [&](float u_, float v_, float w_) {
            if (S.refine) return refine_lookup(A, S, texW, S.res, S.res, u_, v_, w_);
            if (A.fineLayout == LUXGI_LAYOUT_BRICK4)
                return sample3d_brick4<SS>(sdf, texW, S.res, S.res, u_, v_, w_, S.brickScale);
            if (A.fineLayout == LUXGI_LAYOUT_CELL8) return sample3d_cell8<SS>(sdf, texW, S.res, S.res, u_, v_, w_);
            return sample_volume<SS>(sdf, texW, S.res, S.res, u_, v_, w_);
        };
        const float xp = nl(tx + o, uy, uz), xn = nl(tx - o, uy, uz);
        const float yp = nl(tx, uy + o, uz), yn = nl(tx, uy - o, uz);
        const float zp = nl(tx, uy, uz + o), zn = nl(tx, uy, uz - o);
        n = normalize3(mk(xp - xn, yp - yn, zp - zn));
        if (COUNT) c.normals++;
    }
    const float4 s = sample_atlas_wave<SC, COUNT>(S.ad, S.culled, S.objects, objInvBase + S.objectStart * 16, S.tiles,
                                                  static_cast<const SC*>(S.color), S.atlasDepth, lds[threadIdx.x >> 6],
                                                  hp, n, thr, list, count, c);
    if (hit)
        Texel<SR>::st4(static_cast<SR*>(v->rays.radiance), (size_t)probe * v->rays.width + ray,
                       make_float4(s.x, s.y, s.z, 0.f));
    if (COUNT) {
        __shared__ unsigned long long sc[4];
        if (threadIdx.x < 4) sc[threadIdx.x] = 0;
        __syncthreads();
        if (c.normals) atomicAdd(&sc[0], c.normals);
        if (c.objects) atomicAdd(&sc[1], c.objects);
        if (c.tiles) atomicAdd(&sc[2], c.tiles);
        if (valid) atomicAdd(&sc[3], 1ull);
        __syncthreads();
        if (threadIdx.x < 4) atomicAdd(&counters[2 + threadIdx.x], sc[threadIdx.x]);
    }
}

// per-object inverse transforms, once per call
__global__ void trace_prepare_kernel(const LuxgiAtlasObject* __restrict__ objects, int n, float* __restrict__ inv) {
    object_inverse_kernel_body(objects, n, inv);
}

// the same for every scene of a several-scene batch: scene blockIdx.y, its objects from its objectStart
__global__ void trace_prepare_scenes_kernel(const TraceScene* __restrict__ scenes, float* __restrict__ inv) {
    const TraceScene& S = scenes[blockIdx.y];
    object_inverse_kernel_body(S.objects, S.objectCapacity, inv + S.objectStart * 16);
}

}  // namespace luxgi

using namespace luxgi;

static size_t align256(size_t v) { return (v + 255) & ~size_t(255); }

struct TraceWorkspace {
    float* inv;     // per-object inverse transforms
    float4* recA;   // per-ray hit records
    uint8_t* recC;  // and their cascades
};

static size_t trace_workspace_layout(size_t rays, int64_t objects, char* base, TraceWorkspace* w) {
    size_t off = 0;
    if (w) w->inv = reinterpret_cast<float*>(base + off);
    off += align256((size_t)(objects > 0 ? objects : 0) * 16 * sizeof(float));
    if (w) w->recA = reinterpret_cast<float4*>(base + off);
    off += align256(rays * sizeof(float4));
    if (w) w->recC = reinterpret_cast<uint8_t*>(base + off);
    off += align256(rays);
    return off;
}

extern "C" size_t luxgi_ddgi_trace_workspace_size(const LuxgiDDGIUniform* u, int32_t objectCapacity) {
    if (!u) return 0;
    const size_t P = (size_t)u->probeCounts[0] * u->probeCounts[1] * u->probeCounts[2];
    const size_t R = (size_t)(u->raysPerProbe > 0 ? u->raysPerProbe : 0);
    return trace_workspace_layout(P * R, objectCapacity, nullptr, nullptr);
}

// Up to this many rays (counted as lanes: a single volume's rays per probe padded to a multiple of 64) a wave
// takes 16 of them. A small trace is the chain of its longest rays and of its waves' hits, eight at a time,
// with most of the chip idle: shorter waves spread the hits over four times as many. Full waves -> short ones, us,
// for 32,768 lanes (8x8x8x64) and 65,536 (16x8x8x64), then 76,800, 98,304 (12x8x16x64) and 131,072
// (16x8x16x64), 300 objects:
//   linear FP32 256^3  83 -> 75, 86 -> 80, 102 -> 90, 109 -> 99, 119 -> 126   64^3  50 -> 44, 50 -> 50, 51 -> 55
//   cells FP32 256^3   63 -> 57, 63 -> 61, 64 -> 62, 68 -> 68, 74 -> 87       64^3  47 -> 38, 51 -> 47, 53 -> 49
//   bricks FP32 128^3  60 -> 55, 63 -> 63, 69 -> 66, 74 -> 75, 74 -> 94
//   linear FP16 128^3  57 -> 49, 59 -> 59, 77 -> 68, 79 -> 72, 82 -> 88
//   cells FP16 128^3   54 -> 49, 55 -> 55, 58 -> 60, 60 -> 64, 63 -> 79
//   bricks FP16 128^3  56 -> 50, 61 -> 59, 65 -> 64, 67 -> 69, 69 -> 86
// Batches of three volumes, update included: 33,028 rays 98 -> 92, 57,344 93 -> 91, 81,920 97 -> 95,
// 100,352 102 -> 118; over two scenes 98 -> 91, 89 -> 88, 99 -> 94, 102 -> 110. Up to 65,536 none loses more
// than 1%, past it the forms part.
constexpr long long kFewRays = 65536;

// The kernels of one trace: object inverses, march, shade. MODE 0: one volume, 1: a batch over A.scene,
// 2: a batch over per-volume scenes (A.scenes, nScenes of them, at most maxObjects objects each).
template <class SS, class SC, class SR, bool COUNT, int MODE>
static int launch_trace(TraceArgs A, int nScenes, int maxObjects, const TraceWorkspace& w,
                        unsigned long long* counters, hipStream_t st) {
    const long long lanes = MODE != 0 ? A.totalRays : (long long)A.P * ((A.R + 63) & ~63);
    A.waveRays = !COUNT && lanes <= kFewRays ? 16 : 64;
    if (MODE == 2) {
        if (maxObjects > 0) {
            hipLaunchKernelGGL(trace_prepare_scenes_kernel, dim3((maxObjects + 255) / 256, nScenes), dim3(256), 0, st,
                               A.scenes, w.inv);
            LUXGI_LAUNCH_CHECK();
        }
    } else {
        hipLaunchKernelGGL(trace_prepare_kernel, dim3(std::max(1, (A.scene.objectCapacity + 255) / 256)), dim3(256), 0,
                           st, A.scene.objects, A.scene.objectCapacity, w.inv);
        LUXGI_LAUNCH_CHECK();
    }
    const dim3 grid((int)((lanes + 4 * A.waveRays - 1) / (4 * A.waveRays)));
    if (A.fineLayout == LUXGI_LAYOUT_BRICK4)
        hipLaunchKernelGGL((march_kernel<SS, SR, COUNT, LUXGI_LAYOUT_BRICK4, MODE>), grid, dim3(256), 0, st, A, w.recA,
                           w.recC, counters);
    else if (A.fineLayout == LUXGI_LAYOUT_CELL8)
        hipLaunchKernelGGL((march_kernel<SS, SR, COUNT, LUXGI_LAYOUT_CELL8, MODE>), grid, dim3(256), 0, st, A, w.recA,
                           w.recC, counters);
    else
        hipLaunchKernelGGL((march_kernel<SS, SR, COUNT, LUXGI_LAYOUT_LINEAR, MODE>), grid, dim3(256), 0, st, A, w.recA,
                           w.recC, counters);
    LUXGI_LAUNCH_CHECK();
    hipLaunchKernelGGL((shade_kernel<SS, SC, SR, COUNT, MODE>), grid, dim3(256), 0, st, A, w.inv, w.recA, w.recC,
                       counters);
    LUXGI_LAUNCH_CHECK();
    return LUXGI_OK;
}

template <class SS, class SR, bool COUNT, int MODE>
static int dispatch_color(const TraceArgs& A, int atlasLayout, int colorStorage, int nScenes, int maxObjects,
                          const TraceWorkspace& w, unsigned long long* cnt, hipStream_t st) {
    if (atlasLayout == LUXGI_LAYOUT_BRICK4)
        return launch_trace<SS, PackedAtlas, SR, COUNT, MODE>(A, nScenes, maxObjects, w, cnt, st);
    switch (colorStorage) {
        case LUXGI_STORAGE_FP32: return launch_trace<SS, float, SR, COUNT, MODE>(A, nScenes, maxObjects, w, cnt, st);
        case LUXGI_STORAGE_FP16: return launch_trace<SS, __half, SR, COUNT, MODE>(A, nScenes, maxObjects, w, cnt, st);
        case LUXGI_STORAGE_UNORM8: return launch_trace<SS, Unorm8, SR, COUNT, MODE>(A, nScenes, maxObjects, w, cnt, st);
        default: return LUXGI_ERR_UNSUPPORTED;
    }
}

// Checks one scene (SDF + atlas + sky) and writes its kernel-side descriptor.
static int trace_scene_descriptor(const LuxgiGlobalSDFData* g, const LuxgiSDFVolume* vol, const LuxgiSurfaceAtlas* at,
                                  const LuxgiSkybox* sky, const float* skyColor, TraceScene& S) {
    if (!g || !vol || !at) return LUXGI_ERR_INVALID_ARGUMENT;
    const int rc = sdf_volume_status(g, vol);
    if (rc != LUXGI_OK) return rc;
    if (!at->chunks || !at->culledObjects || !at->objects || !at->tiles || !at->color) return LUXGI_ERR_INVALID_ARGUMENT;
    if (at->layout == LUXGI_LAYOUT_LINEAR) {
        if (!at->depth) return LUXGI_ERR_INVALID_ARGUMENT;
    } else if (at->layout == LUXGI_LAYOUT_BRICK4) {
        if (at->colorStorage != LUXGI_STORAGE_UNORM8 || (at->data.resolution & 3u)) return LUXGI_ERR_INVALID_ARGUMENT;
    } else {
        return LUXGI_ERR_INVALID_ARGUMENT;
    }
    if (at->data.resolution == 0 || at->objectCapacity < 0) return LUXGI_ERR_INVALID_ARGUMENT;
    if (sky && sky->faces && sky->size <= 0) return LUXGI_ERR_INVALID_ARGUMENT;
    S = TraceScene{};
    S.g = *g;
    S.ad = at->data;
    S.sdf = vol->sdf;
    S.mip = vol->mip;
    S.guard = vol->guard;
    S.brickScale = vol->brickScale;
    S.refine = vol->refine;
    S.chunks = at->chunks;
    S.culled = at->culledObjects;
    S.objects = at->objects;
    S.tiles = at->tiles;
    S.color = at->color;
    S.atlasDepth = at->depth;
    S.skyFaces = sky && sky->faces ? sky->faces : nullptr;
    S.objectStart = 0;
    S.objectCapacity = at->objectCapacity;
    for (int i = 0; i < 3; ++i) S.sky[i] = skyColor[i];
    S.invCascades = 1.0f / float(g->cascadesCount);
    S.res = vol->resolution;
    S.mipRes = vol->mipResolution;
    S.skySize = sky ? sky->size : 0;
    S.refineLayout = vol->refineLayout;
    return LUXGI_OK;
}

// The scene arguments shared by the single and batched traces: checks them and fills A's scene
// and the call's settings.
static int trace_scene_args(const LuxgiGlobalSDFData* g, const LuxgiSDFVolume* vol, const LuxgiSurfaceAtlas* at,
                            const LuxgiSkybox* sky, const LuxgiTraceParams* p, TraceArgs& A) {
    if (!p) return LUXGI_ERR_INVALID_ARGUMENT;
    const int rc = trace_scene_descriptor(g, vol, at, sky, p->skyColor, A.scene);
    if (rc != LUXGI_OK) return rc;
    A.scenes = nullptr;
    A.maxSteps = p->maxSteps > 0 ? p->maxSteps : 250;
    A.hitEps = p->hitEpsilon;
    A.fineLayout = vol->layout;
    if (p->shadeOrder != 0 && p->shadeOrder != 1) return LUXGI_ERR_INVALID_ARGUMENT;
    A.vols = nullptr;
    A.nVols = 0;
    A.totalRays = 0;
    return LUXGI_OK;
}

template <bool COUNT, int MODE>
static int trace_launch(const TraceArgs& A, int sdfStorage, int atlasLayout, int colorStorage, int rayStorage,
                        size_t rays, int64_t objects, int nScenes, int maxObjects, void* workspace,
                        size_t workspaceBytes, unsigned long long* counters, hipStream_t st) {
    const size_t need = trace_workspace_layout(rays, objects, nullptr, nullptr);
    if (!workspace || workspaceBytes < need) return LUXGI_ERR_WORKSPACE_TOO_SMALL;
    TraceWorkspace w;
    trace_workspace_layout(rays, objects, static_cast<char*>(workspace), &w);
    const bool r32 = rayStorage == LUXGI_STORAGE_FP32;
    if (rayStorage != LUXGI_STORAGE_FP32 && rayStorage != LUXGI_STORAGE_FP16) return LUXGI_ERR_UNSUPPORTED;
    switch (sdfStorage) {
        case LUXGI_STORAGE_FP32:
            return r32 ? dispatch_color<float, float, COUNT, MODE>(A, atlasLayout, colorStorage, nScenes, maxObjects, w,
                                                                   counters, st)
                       : dispatch_color<float, __half, COUNT, MODE>(A, atlasLayout, colorStorage, nScenes, maxObjects,
                                                                    w, counters, st);
        case LUXGI_STORAGE_FP16:
            return r32 ? dispatch_color<__half, float, COUNT, MODE>(A, atlasLayout, colorStorage, nScenes, maxObjects,
                                                                    w, counters, st)
                       : dispatch_color<__half, __half, COUNT, MODE>(A, atlasLayout, colorStorage, nScenes, maxObjects,
                                                                     w, counters, st);
        case LUXGI_STORAGE_BF16:
            return r32 ? dispatch_color<__bf16, float, COUNT, MODE>(A, atlasLayout, colorStorage, nScenes, maxObjects,
                                                                    w, counters, st)
                       : dispatch_color<__bf16, __half, COUNT, MODE>(A, atlasLayout, colorStorage, nScenes, maxObjects,
                                                                     w, counters, st);
        default: return LUXGI_ERR_UNSUPPORTED;
    }
}

// checks one volume's own arguments (grid and ray buffers)
static int trace_volume_ok(const LuxgiDDGIUniform* u, const LuxgiRayBuffers* rays) {
    if (!u || !rays || !rays->radiance || !rays->directionDistance) return LUXGI_ERR_INVALID_ARGUMENT;
    const long long P = (long long)u->probeCounts[0] * u->probeCounts[1] * u->probeCounts[2];
    if (u->probeCounts[0] <= 0 || u->probeCounts[1] <= 0 || u->probeCounts[2] <= 0) return LUXGI_ERR_INVALID_ARGUMENT;
    if (u->raysPerProbe <= 0 || u->raysPerProbe > rays->width || rays->height < P) return LUXGI_ERR_INVALID_ARGUMENT;
    if (P * u->raysPerProbe >= (1ll << 31)) return LUXGI_ERR_UNSUPPORTED;
    if (rays->storage != LUXGI_STORAGE_FP32 && rays->storage != LUXGI_STORAGE_FP16) return LUXGI_ERR_UNSUPPORTED;
    return LUXGI_OK;
}

template <bool COUNT>
static int trace_entry(const LuxgiDDGIUniform* u, const LuxgiGlobalSDFData* g, const LuxgiSDFVolume* vol,
                       const LuxgiSurfaceAtlas* at, const LuxgiSkybox* sky, const LuxgiTraceParams* p,
                       const float* probeOffsets, const LuxgiRayBuffers* rays, uint8_t* rayFlags, void* workspace,
                       size_t workspaceBytes, unsigned long long* counters, void* stream) {
    int rc = trace_volume_ok(u, rays);
    if (rc != LUXGI_OK) return rc;
    TraceArgs A;
    rc = trace_scene_args(g, vol, at, sky, p, A);
    if (rc != LUXGI_OK) return rc;
    A.P = u->probeCounts[0] * u->probeCounts[1] * u->probeCounts[2];
    A.R = u->raysPerProbe;
    A.rayWidth = rays->width;
    A.vol.uniform = *u;
    for (int i = 0; i < 16; ++i) A.vol.orientation[i] = p->randomOrientation[i];
    A.vol.deviceOrientation = p->deviceOrientation;
    A.vol.probeOffsets = probeOffsets;
    A.vol.rays = *rays;
    A.vol.rayFlags = rayFlags;
    A.vol.rayStart = 0;
    A.vol.scene = 0;
    return trace_launch<COUNT, 0>(A, vol->storage, at->layout, at->colorStorage, rays->storage, (size_t)A.P * A.R,
                                  at->objectCapacity, 1, at->objectCapacity, workspace, workspaceBytes, counters,
                                  as_stream(stream));
}

extern "C" int luxgi_ddgi_trace_batch_prepare(LuxgiTraceVolume* volumes, int32_t count, int32_t rayStorage,
                                              int64_t* totalRays) {
    if (!volumes || !totalRays || count <= 0 || count > LUXGI_MAX_TRACE_BATCH) return LUXGI_ERR_INVALID_ARGUMENT;
    if (rayStorage != LUXGI_STORAGE_FP32 && rayStorage != LUXGI_STORAGE_FP16) return LUXGI_ERR_UNSUPPORTED;
    long long total = 0;
    for (int k = 0; k < count; ++k) {
        LuxgiTraceVolume& v = volumes[k];
        const int rc = trace_volume_ok(&v.uniform, &v.rays);
        if (rc != LUXGI_OK) return rc;
        if (v.rays.storage != rayStorage) return LUXGI_ERR_INVALID_ARGUMENT;
        v.rayStart = total;
        total += (long long)v.uniform.probeCounts[0] * v.uniform.probeCounts[1] * v.uniform.probeCounts[2] *
                 v.uniform.raysPerProbe;
        if (total >= (1ll << 31)) return LUXGI_ERR_UNSUPPORTED;
    }
    *totalRays = total;
    return LUXGI_OK;
}

extern "C" size_t luxgi_ddgi_trace_batch_workspace_size(int64_t totalRays, int32_t objectCapacity) {
    if (totalRays <= 0 || totalRays >= (1ll << 31)) return 0;
    return trace_workspace_layout((size_t)totalRays, objectCapacity, nullptr, nullptr);
}

extern "C" int luxgi_ddgi_trace_sdf_batched(const LuxgiTraceVolume* volumes, int32_t count, int64_t totalRays,
                                            int32_t rayStorage, const LuxgiGlobalSDFData* g,
                                            const LuxgiSDFVolume* vol, const LuxgiSurfaceAtlas* at,
                                            const LuxgiSkybox* sky, const LuxgiTraceParams* p, void* workspace,
                                            size_t workspaceBytes, void* stream) {
    if (!volumes || count <= 0 || count > LUXGI_MAX_TRACE_BATCH || totalRays <= 0 || totalRays >= (1ll << 31))
        return LUXGI_ERR_INVALID_ARGUMENT;
    TraceArgs A;
    const int rc = trace_scene_args(g, vol, at, sky, p, A);
    if (rc != LUXGI_OK) return rc;
    A.P = A.R = A.rayWidth = 0;
    A.vols = volumes;
    A.nVols = count;
    A.totalRays = totalRays;
    return trace_launch<false, 1>(A, vol->storage, at->layout, at->colorStorage, rayStorage, (size_t)totalRays,
                                  at->objectCapacity, 1, at->objectCapacity, workspace, workspaceBytes, nullptr,
                                  as_stream(stream));
}

// ------------------------------------------------------------------------- several scenes

extern "C" size_t luxgi_ddgi_trace_scenes_descriptor_bytes(int32_t sceneCount) {
    if (sceneCount <= 0 || sceneCount > LUXGI_MAX_TRACE_BATCH) return 0;
    return (size_t)sceneCount * sizeof(TraceScene);
}

extern "C" int luxgi_ddgi_trace_scenes_prepare(const LuxgiTraceScene* scenes, int32_t sceneCount,
                                               LuxgiTraceVolume* volumes, int32_t volumeCount, int32_t rayStorage,
                                               void* descriptors, LuxgiTraceSceneBatch* batch) {
    if (!scenes || !volumes || !descriptors || !batch || sceneCount <= 0 || sceneCount > LUXGI_MAX_TRACE_BATCH ||
        volumeCount <= 0 || volumeCount > LUXGI_MAX_TRACE_BATCH)
        return LUXGI_ERR_INVALID_ARGUMENT;
    if (rayStorage != LUXGI_STORAGE_FP32 && rayStorage != LUXGI_STORAGE_FP16) return LUXGI_ERR_UNSUPPORTED;
    TraceScene* out = static_cast<TraceScene*>(descriptors);
    long long objects = 0;
    int maxObjects = 0;
    for (int k = 0; k < sceneCount; ++k) {
        const LuxgiTraceScene& sc = scenes[k];
        TraceScene S;
        const int rc = trace_scene_descriptor(&sc.sdfData, &sc.volume, &sc.atlas, &sc.skybox, sc.skyColor, S);
        if (rc != LUXGI_OK) return rc;
        // one kernel instantiation serves the batch: every scene stores its SDF and atlas alike
        if (sc.volume.storage != scenes[0].volume.storage || sc.volume.layout != scenes[0].volume.layout ||
            sc.atlas.layout != scenes[0].atlas.layout || sc.atlas.colorStorage != scenes[0].atlas.colorStorage)
            return LUXGI_ERR_INVALID_ARGUMENT;
        S.objectStart = objects;
        objects += sc.atlas.objectCapacity;
        maxObjects = std::max(maxObjects, (int)sc.atlas.objectCapacity);
        out[k] = S;
    }
    long long total = 0;
    for (int k = 0; k < volumeCount; ++k) {
        LuxgiTraceVolume& v = volumes[k];
        const int rc = trace_volume_ok(&v.uniform, &v.rays);
        if (rc != LUXGI_OK) return rc;
        if (v.rays.storage != rayStorage || v.scene < 0 || v.scene >= sceneCount) return LUXGI_ERR_INVALID_ARGUMENT;
        total = (total + 63) & ~63ll;  // a wave never spans two volumes
        v.rayStart = total;
        total += (long long)v.uniform.probeCounts[0] * v.uniform.probeCounts[1] * v.uniform.probeCounts[2] *
                 v.uniform.raysPerProbe;
        if (total >= (1ll << 31)) return LUXGI_ERR_UNSUPPORTED;
    }
    batch->totalRays = total;
    batch->totalObjects = objects;
    batch->sceneCount = sceneCount;
    batch->volumeCount = volumeCount;
    batch->maxObjects = maxObjects;
    batch->rayStorage = rayStorage;
    batch->sdfStorage = scenes[0].volume.storage;
    batch->sdfLayout = scenes[0].volume.layout;
    batch->atlasLayout = scenes[0].atlas.layout;
    batch->colorStorage = scenes[0].atlas.colorStorage;
    return LUXGI_OK;
}

extern "C" size_t luxgi_ddgi_trace_scenes_workspace_size(const LuxgiTraceSceneBatch* batch) {
    if (!batch || batch->totalRays <= 0 || batch->totalRays >= (1ll << 31) || batch->totalObjects < 0) return 0;
    return trace_workspace_layout((size_t)batch->totalRays, batch->totalObjects, nullptr, nullptr);
}

extern "C" int luxgi_ddgi_trace_sdf_scenes(const LuxgiTraceSceneBatch* batch, const LuxgiTraceVolume* volumes,
                                           const void* descriptors, const LuxgiTraceParams* p, void* workspace,
                                           size_t workspaceBytes, void* stream) {
    if (!batch || !volumes || !descriptors || !p) return LUXGI_ERR_INVALID_ARGUMENT;
    if (batch->sceneCount <= 0 || batch->sceneCount > LUXGI_MAX_TRACE_BATCH || batch->volumeCount <= 0 ||
        batch->volumeCount > LUXGI_MAX_TRACE_BATCH || batch->totalRays <= 0 || batch->totalRays >= (1ll << 31) ||
        batch->totalObjects < 0 || batch->maxObjects < 0)
        return LUXGI_ERR_INVALID_ARGUMENT;
    TraceArgs A{};
    A.scenes = static_cast<const TraceScene*>(descriptors);
    A.maxSteps = p->maxSteps > 0 ? p->maxSteps : 250;
    A.hitEps = p->hitEpsilon;
    A.fineLayout = batch->sdfLayout;
    A.vols = volumes;
    A.nVols = batch->volumeCount;
    A.totalRays = batch->totalRays;
    return trace_launch<false, 2>(A, batch->sdfStorage, batch->atlasLayout, batch->colorStorage, batch->rayStorage,
                                  (size_t)batch->totalRays, batch->totalObjects, batch->sceneCount, batch->maxObjects,
                                  workspace, workspaceBytes, nullptr, as_stream(stream));
}

extern "C" int luxgi_ddgi_trace_sdf(const LuxgiDDGIUniform* u, const LuxgiGlobalSDFData* g, const LuxgiSDFVolume* vol,
                                    const LuxgiSurfaceAtlas* at, const LuxgiSkybox* sky, const LuxgiTraceParams* p,
                                    const float* probeOffsets, const LuxgiRayBuffers* rays, uint8_t* rayFlags,
                                    void* workspace, size_t workspaceBytes, void* stream) {
    return trace_entry<false>(u, g, vol, at, sky, p, probeOffsets, rays, rayFlags, workspace, workspaceBytes, nullptr,
                              stream);
}

extern "C" int luxgi_ddgi_trace_sdf_count(const LuxgiDDGIUniform* u, const LuxgiGlobalSDFData* g,
                                          const LuxgiSDFVolume* vol, const LuxgiSurfaceAtlas* at,
                                          const LuxgiSkybox* sky, const LuxgiTraceParams* p, const float* probeOffsets,
                                          const LuxgiRayBuffers* rays, uint8_t* rayFlags, void* workspace,
                                          size_t workspaceBytes, unsigned long long* counters, void* stream) {
    if (!counters) return LUXGI_ERR_INVALID_ARGUMENT;
    return trace_entry<true>(u, g, vol, at, sky, p, probeOffsets, rays, rayFlags, workspace, workspaceBytes, counters,
                             stream);
}

namespace luxgi {
__global__ void atlas_pack_kernel(const uint32_t* __restrict__ color, const float* __restrict__ depth, int res,
                                  uint2* __restrict__ packed) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y;
    if (i >= res) return;
    const size_t e = (size_t)j * res + i;
    packed[atlas_block_index(i, j, res)] = make_uint2(color[e], __float_as_uint(depth[e]));
}
}  // namespace luxgi

extern "C" int luxgi_atlas_pack(const uint32_t* color, const float* depth, int32_t res, void* packed, void* stream) {
    if (!color || !depth || !packed || res <= 0 || (res & 3) || (size_t)res * res * 8 >= (1ull << 32))
        return LUXGI_ERR_INVALID_ARGUMENT;
    hipLaunchKernelGGL(atlas_pack_kernel, dim3((res + 255) / 256, res), dim3(256), 0, as_stream(stream), color, depth,
                       res, static_cast<uint2*>(packed));
    LUXGI_LAUNCH_CHECK();
    return LUXGI_OK;
}
