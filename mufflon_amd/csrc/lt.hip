// Light tracer for gfx950: the GPU device of Mufflon's "Lighttracer"
// (GpuLightTracer, gpu_lt.cpp:25-37, gpu_lt.cu:19-101, lt_sample of
// lt_common.hpp:17-78) over the scene, camera and positional lights of a
// path tracer.
//
// A lane owns a light path and runs its iterations one after the other, every
// iteration of a call in one launch (path regeneration, as in the path
// tracer's megakernel; each iteration splats into an image of its own); path i
// of an iteration draws from generator i
// (seeded like the path tracer's) and emits a photon from the light tree
// with index i of numPixels (emit, light_tree_sampling.hpp:81-187: the index
// spreads the photons over the tree's flux intervals), then walks the
// scene on adjoint BSDF samples (walk, random_walk.hpp:38-112). Every
// vertex, the light's own included, is connected to the pinhole camera:
// the direction is projected to its pixel (pinholecam_project,
// pinhole.hpp:86-116), the adjoint BSDF (or the emitter's distribution)
// weights it, a shadow ray checks it, and the contribution is added to the
// pixel's Radiance, Lightness and (when recorded) Density with float
// atomics. The per-iteration splat image then goes into the running means
// (and variances) of the three targets like every target of the output
// handler. The order of the atomic additions is not fixed, so sums agree
// with a sequential evaluation to rounding, not bit for bit.
#include "pt_path.hpp"

namespace mfh {

namespace {

using namespace shade;
using namespace path;

constexpr int kLtThreads = 64;

// Sampler result of a positional light (Emitter, light_sampling.hpp:21-52).
struct LtEmitter {
    V3 position, intensity, normal;
    V3 absorption;  // of the medium the photon leaves into (vacuum around point lights)
    bool area;
};

// sample_light_pos (light_sampling.hpp:80-199) of a light of the tree:
// point, area triangle, quad and sphere.
__device__ LtEmitter light_position(const PtScene& S, uint16_t type, u32 offset, float u0, float u1) {
    const uint8_t* light = S.lightMem + offset;
    LtEmitter e;
    if (type == kLightPoint) {
        const float4 a = ld4(light), b = ld4(light + 16);
        e.position = v3(a.x, a.y, a.z);
        e.intensity = v3(b.x, b.y, b.z);
        e.normal = v3(0, 0, 0);
        e.absorption = v3(0, 0, 0);
        e.area = false;
        return e;
    }
    e.area = true;
    if (type == kLightAreaQuad) {
        V3 pv[4];
        quad_record(light, pv);
        const float4 w0 = ld4(light + 48), w1 = ld4(light + 64);
        const int matIdx = (int)(*reinterpret_cast<const uint16_t*>(light + 80));
        const V3 tangentX = pv[1] + smul(u0, pv[3]);
        const V3 tangentY = pv[2] + smul(u1, pv[3]);
        V3 normal = cross(tangentY, tangentX);
        const float area = len(normal);
        e.normal = normal / area;
        e.position = pv[0] + tangentX * u1 + pv[2] * u0;
        const float lu = w0.x + w0.z * u1 + w1.x * u0 + w1.z * (u0 * u1);
        const float lv = w0.y + w0.w * u1 + w1.y * u0 + w1.w * (u0 * u1);
        const MatParams m = fetch(S, matIdx, lu, lv);
        e.intensity = emission(m, v3(0, 0, 1), v3(0, 0, 1)) * area;
        e.absorption = m.outer.absorption;
        return e;
    }
    if (type == kLightAreaSphere) {
        const float4 q0 = ld4(light);
        const int matIdx = (int)(*reinterpret_cast<const uint16_t*>(light + 16));
        // sample_dir_sphere_uniform (sampling.hpp:101-109)
        const float cosTheta = u0 * 2.0f - 1.0f;
        const float sinTheta = fsqrt((1.0f - cosTheta) * (1.0f + cosTheta));
        const float phi = u1 * 2.0f * kPi;
        const SinCos sc = fsincos(phi);
        const V3 n = v3(sinTheta * sc.s, sinTheta * sc.c, cosTheta);
        // the emitter's uv is (u1, acos(n.z)), the polar angle unnormalized
        // (light_sampling.hpp:181)
        const MatParams m = fetch(S, matIdx, u1, facos(n.z));
        const V3 radiance = emission(m, v3(0, 0, 1), v3(0, 0, 1));
        e.absorption = m.outer.absorption;
        const float area = 4 * kPi * q0.w * q0.w;
        e.position = v3(q0.x, q0.y, q0.z) + n * q0.w;
        e.normal = n;
        e.intensity = radiance * area;
        return e;
    }
    const float4 q0 = ld4(light), q1 = ld4(light + 16), q2 = ld4(light + 32), q3 = ld4(light + 48);
    const V3 p0 = v3(q0.x, q0.y, q0.z), e1 = v3(q0.w, q1.x, q1.y), e2 = v3(q1.z, q1.w, q2.x);
    const int matIdx = (int)(__float_as_uint(q2.y) & 0xFFFFu);
    V3 normal = cross(e1, e2);
    const float area2 = len(normal);
    e.normal = normal / area2;
    const float area = area2 * 0.5f;
    const float s = 1.f - fsqrt(1.f - u0);
    const float t = (1.f - s) * u1;
    e.position = p0 + e1 * s + e2 * t;
    const float lu = q2.z + q3.x * s + q3.z * t;
    const float lv = q2.w + q3.y * s + q3.w * t;
    const MatParams m = fetch(S, matIdx, lu, lv);
    e.intensity = emission(m, v3(0, 0, 1), v3(0, 0, 1)) * area;
    e.absorption = m.outer.absorption;
    return e;
}

// emit (light_tree_sampling.hpp:81-187) for trees of positional lights (the
// host refuses backgrounds that emit): the flux intervals of the tree's
// nodes partition the 64-bit range, which path `index` of numIndices enters
// at seed + index * (2^64-1) / numIndices; the intensity is divided by the
// probability of the chosen light (adjustPdf).
__device__ LtEmitter emit(const PtScene& S, u64 index, u64 numIndices, u64 seed, float u0, float u1) {
    u64 rndChoice = numIndices > 0 ? seed + index * (~0ull / numIndices) : seed;
    if (rndChoice == ~0ull) --rndChoice;
    const float fluxSum = S.bgFlux + S.dirRootFlux + S.posRootFlux;
    const float envProb = S.bgFlux / fluxSum;
    const float dirProb = S.dirRootFlux / fluxSum;
    const float posProb = S.posRootFlux / fluxSum;
    u64 left = percentage_of(~0ull, envProb + dirProb);
    u64 right = ~0ull;
    float lightProb = posProb;
    uint16_t type = (uint16_t)S.posRootType;
    u32 offset = 0;
    for (int guard = 0; type == kLightInternalNode && guard < 64; ++guard) {
        const float4 a = ld4(S.lightMem + offset), b = ld4(S.lightMem + offset + 16);
        const u32 types = __float_as_uint(a.z);
        const float probLeft = a.x / (a.x + b.x);
        const u64 boundary = left + percentage_of(right - left, probLeft);
        if (rndChoice < boundary) {
            type = (uint16_t)(types & 0xFFFFu);
            offset = __float_as_uint(a.y);
            right = boundary;
            lightProb *= probLeft;
        } else {
            type = (uint16_t)(types >> 16);
            offset = __float_as_uint(a.w);
            left = boundary;
            lightProb *= (1.0f - probLeft);
        }
    }
    LtEmitter e = light_position(S, type, offset, u0, u1);
    e.intensity = e.intensity / lightProb;
    return e;
}

// pinholecam_project (pinhole.hpp:86-116): the pixel a direction from the
// camera falls on and the camera's importance w (the pdf of sampling it).
__device__ __forceinline__ bool project(const PtScene& S, V3 dir, int& px, int& py, float& w) {
    const V3 viewDir = v3(S.camDir[0], S.camDir[1], S.camDir[2]);
    const V3 up = v3(S.camUp[0], S.camUp[1], S.camUp[2]);
    const float cosOut = dot(viewDir, dir);
    if (cosOut < 0.0f) return false;
    const V3 xAxis = cross(viewDir, up);
    const float den = cosOut * S.tanVFov;
    float ux = dot(xAxis, dir) / den;
    const float uy = dot(up, dir) / den;
    const float aspect = (float)S.width / (float)S.height;
    ux /= aspect;
    if (!(ux > -1 && ux <= 1 && uy > -1 && uy <= 1)) return false;
    px = (int)floorf((ux * 0.5f + 0.5f) * (float)S.width);
    py = (int)floorf((uy * 0.5f + 0.5f) * (float)S.height);
    if (px >= S.width) px = S.width - 1;
    if (py >= S.height) py = S.height - 1;
    const float pixelArea = (2.0f * S.tanVFov) * (2.0f * S.tanVFov) * aspect;
    w = 1.0f / (pixelArea * cosOut * cosOut * cosOut);
    return true;
}

// Splat image of one iteration: Radiance (3), Lightness, Density per pixel.
constexpr int kLtChannels = 5;

// A connection of a vertex to the camera, splatted when nothing is between.
struct LtSplat {
    V3 a, dir;
    float tmax;
    V3 radiance;
    float lightness, density;
    int pixel;
};

// Connection of the vertex at vpos to the camera (get_connection,
// path_util.hpp:384-399): false when it falls outside the image or carries
// nothing. light: the path's emitter at pathLen 0, vx its vertex after.
__device__ __forceinline__ bool connect_camera(const PtScene& S, V3 vpos, bool atLight, const LtEmitter& light,
                                               const Vertex& vx, V3 throughput, int density, LtSplat& c) {
    const V3 camPos = v3(S.camPos[0], S.camPos[1], S.camPos[2]);
    const V3 conn = vpos - camPos;
    const float distSq = dot(conn, conn);
    const float dist = fsqrt(distSq);
    const float dden = dist + 1e-20f * (dist < 0.0f ? -1.0f : 1.0f);
    const V3 dir = conn / dden;
    int px, py;
    float w;
    if (!project(S, dir, px, py, w)) return false;
    V3 lval;
    float lcos;
    V3 geoN;
    float geomFactor;
    if (atLight) {
        if (light.area) {  // evaluate_area (lights.hpp:286-295)
            const float k = dot(light.normal, neg(dir));
            lval = k <= 0.0f ? v3(0, 0, 0) : light.intensity;
            lcos = k <= 0.0f ? 0.0f : k;
            geoN = light.normal;
            geomFactor = dot(dir, light.normal);
        } else {  // evaluate_point (lights.hpp:262-265)
            lval = light.intensity;
            lcos = 1.0f;
            geoN = v3(0, 0, 0);
            geomFactor = 0.0f;
        }
    } else {
        lval = mat_evaluate_adjoint(vx.ts, vx.mat, vx.incident(), neg(dir), lcos);
        geoN = vx.ts.geoN;
        geomFactor = dot(dir, vx.ts.shadingN);
    }
    V3 bxdfProd = v3(w * lval.x, w * lval.y, w * lval.z);
    const float cosProd = 1.0f * lcos;
    if (!(density || ((bxdfProd.x > 0.0f || bxdfProd.y > 0.0f || bxdfProd.z > 0.0f) && cosProd > 0.0f))) return false;
    // any_intersection (intersection.cu:624-637); the camera has no normal
    c.a = add_epsilon(camPos, dir, v3(0, 0, 0));
    const V3 b = add_epsilon(vpos, neg(dir), geoN);
    const V3 d = b - c.a;
    c.tmax = len(d);
    c.dir = d / c.tmax;
    bxdfProd = bxdfProd / distSq;
    c.radiance = throughput * cosProd * bxdfProd;
    c.lightness = (throughput.x + throughput.y + throughput.z) / 3.0f * cosProd;
    c.density = w * 1.0f / distSq * fabsf(geomFactor);
    c.pixel = px + py * S.width;
    return true;
}

// A turn of the loop is one path segment: the emission, or a closest hit and
// its vertex; then the connection to the camera and the walk to the next
// segment. The connection's shadow ray is traced after the walk, when the
// vertex is no longer live. Against one path per lane and a launch per
// iteration: Cornell box 256x256, 16 iterations 13.9 -> 13.0 ms, 64x87, one
// iteration 1.13 -> 0.87 ms. The splats' atomics are not what bounds it (12.7
// ms without them): it is the traversal's chain, as in the megakernel.
template <int kMode>
__global__ __launch_bounds__(kLtThreads) __attribute__((amdgpu_waves_per_eu(3))) void k_lt_iterate(
    PtScene S, PathWork W, float* __restrict__ splat, int minPathLength, int maxPathLength, int density) {
    __shared__ int sStack[kLdsDepth * kLtThreads];
    int* const lstack = sStack + threadIdx.x;
    const int num = S.width * S.height;
    SlotQueue slots(W);
    bool busy = false;
    int idx = 0, done = 0, pathLen = -1;  // -1: the light emits next
    u64 rng = 0;
    V3 throughput = v3(1.0f, 1.0f, 1.0f), rayOrigin = throughput, dir = throughput, absorption = throughput;
    while (true) {
        const int slot = slots.take(W, busy);
        if (slot >= 0) {
            busy = true;
            idx = slot;
            done = 0;
            pathLen = -1;
            rng = S.rngs[idx];
        }
        if (__ballot(busy) == 0ull && !slots.more) break;
        if (busy) {
            bool ended = false, shadow = false;
            LtEmitter light;
            Vertex vx;
            LtSplat c;
            if (pathLen < 0) {
                throughput = v3(1.0f, 1.0f, 1.0f);
                const u64 xStart = pcg_next(rng);
                const u64 treeSeed = pcg_next(rng);
                light = emit(S, (u64)idx, (u64)num, treeSeed, sample_uniform((u32)xStart),
                             sample_uniform((u32)(xStart >> 32)));
                pcg_next(rng);  // create_camera's RndSet2, unused by the pinhole
            } else {
                const TraceHit hit =
                    trace_mode<kMode, false, kLtThreads, kLdsDepth>(S.trace, rayOrigin, dir, kMaxSceneSize, lstack);
                throughput = throughput * transmission(Medium{1.0f, absorption}, hit.inst == -1 ? kMaxSceneSize : hit.t);
                ended = hit.inst == -1;
                if (!ended)
                    make_vertex(S, rayOrigin, dir, 0.0f, hit.t, hit.inst, hit.prim, hit.w0, hit.w1, vx);
            }
            if (!ended) {
                ++pathLen;
                ended = pathLen > 0 && pathLen >= maxPathLength;
            }
            if (!ended) {
                const bool atLight = pathLen == 0;
                if (pathLen + 1 >= minPathLength && pathLen + 1 <= maxPathLength)
                    shadow = connect_camera(S, atLight ? light.position : vx.position, atLight, light, vx, throughput,
                                            density, c);
                // walk (random_walk.hpp:38-112), adjoint
                const u64 x0 = pcg_next(rng);
                const u64 x1 = pcg_next(rng);
                const float rndRoulette = sample_uniform((u32)pcg_next(rng));
                V3 origin, sThroughput, geoOut;
                if (atLight) {
                    // the light's direction (sample_light_dir_point / _area,
                    // light_sampling.hpp:85-89, 201-211)
                    const float u0 = sample_uniform((u32)x0), u1 = sample_uniform((u32)(x0 >> 32));
                    if (light.area) {
                        const float cosT = fsqrt(u0);
                        const float sinT = fsqrt(1.0f - u0);
                        const float phi = u1 * 2 * kPi;
                        const SinCos sc = fsincos(phi);
                        const float lx = sinT * sc.s, ly = sinT * sc.c;
                        const V3 tx = normalize(perpendicular(light.normal));
                        const V3 ty = cross(light.normal, tx);
                        dir = smul(lx, tx) + smul(ly, ty) + smul(cosT, light.normal);
                        sThroughput = light.intensity * kPi;
                        geoOut = light.normal;
                    } else {
                        const float cosT = u0 * 2.0f - 1.0f;
                        const float sinT = fsqrt((1.0f - cosT) * (1.0f + cosT));
                        const float phi = u1 * 2.0f * kPi;
                        const SinCos sc = fsincos(phi);
                        dir = v3(sinT * sc.s, sinT * sc.c, cosT);
                        sThroughput = light.intensity * 4 * kPi;
                        geoOut = v3(0, 0, 0);
                    }
                    origin = light.position;
                    absorption = light.absorption;
                } else {
                    float pdfF;
                    V3 out;
                    ended = !mat_sample(vx.ts, vx.mat, vx.incident(), sample_uniform((u32)x0),
                                        sample_uniform((u32)(x0 >> 32)), x1, sThroughput, out, pdfF, true);
                    if (!ended) {
                        dir = out;
                        absorption = vx.mat.medium(dot(dir, vx.ts.geoN)).absorption;
                        origin = vx.position;
                        geoOut = vx.ts.geoN;
                    }
                }
                if (!ended) {
                    throughput = throughput * sThroughput;
                    const float cont = mn(mx(mx(throughput.x, throughput.y), throughput.z) + 0.1f, 1.0f);
                    ended = rndRoulette >= cont;
                    if (!ended) {
                        throughput = throughput / cont;
                        rayOrigin = add_epsilon(origin, dir, geoOut);
                    }
                }
            }
            if (shadow &&
                trace_mode<kMode, true, kLtThreads, kLdsDepth>(S.trace, c.a, c.dir, c.tmax, lstack).inst == -1) {
                float* o = splat + (size_t)kLtChannels * ((size_t)num * done + c.pixel);
                atomicAdd(o, c.radiance.x);
                atomicAdd(o + 1, c.radiance.y);
                atomicAdd(o + 2, c.radiance.z);
                atomicAdd(o + 3, c.lightness);
                if (density) atomicAdd(o + 4, c.density);
            }
            if (ended) {
                pathLen = -1;
                if (++done == W.iterations) {
                    S.rngs[idx] = rng;
                    busy = false;
                }
            }
        }
    }
}

__global__ void k_lt_clear(float* p, size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0.0f;
}

// Running mean (and variance) of the splat images of `iterations` iterations
// from index `first` on (UpdateIter, output_handler_variance.hpp:7-31).
__global__ void k_lt_accumulate(const float* __restrict__ splat, float* __restrict__ mean, float* __restrict__ var,
                                size_t n, int first, int iterations) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float m = mean[i], v = var ? var[i] : 0.0f;
    for (int k = 0; k < iterations; ++k) {
        const int iteration = first + k;
        const float iter = splat[n * k + i];
        const float diff = iter - m;
        m = m + diff / mx(1.0f, (float)iteration + 1);
        v += (diff * (iter - m) - v) / mx(1.0f, (float)iteration);
    }
    mean[i] = m;
    if (var) var[i] = v;
}

}  // namespace

void launch_lighttracer(const PtScene& S, int iterations, float* splat, float* mean, float* var, int minPathLength,
                        int maxPathLength, bool density, LaunchQueue& queue, int numCUs, hipStream_t stream) {
    const size_t n = (size_t)kLtChannels * S.width * S.height;
    const size_t all = n * iterations;
    hipLaunchKernelGGL(k_lt_clear, dim3((unsigned)((all + 255) / 256)), dim3(256), 0, stream, splat, all);
    const int mode = trace_mode_of(S.trace);
    auto* const fn = mode == kTraceSingle       ? k_lt_iterate<kTraceSingle>
                     : mode == kTraceMulti      ? k_lt_iterate<kTraceMulti>
                     : mode == kTraceSingleTies ? k_lt_iterate<kTraceSingleTies>
                     : mode == kTraceMultiTies  ? k_lt_iterate<kTraceMultiTies>
                                                : k_lt_iterate<kTraceMixed>;
    PathWork W;
    const int grid =
        path_work(reinterpret_cast<const void*>(fn), S.width * S.height, iterations, queue, numCUs, W);
    hipLaunchKernelGGL(fn, dim3(grid), dim3(kLtThreads), 0, stream, S, W, splat, minPathLength, maxPathLength,
                       density ? 1 : 0);
    MFH_HIP(hipGetLastError());
    queue.next ^= 1;
    hipLaunchKernelGGL(k_lt_accumulate, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, splat, mean, var, n,
                       S.iteration, iterations);
    MFH_HIP(hipGetLastError());
}

}  // namespace mfh
