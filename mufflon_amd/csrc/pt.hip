// Path tracer megakernel for gfx950: the GPU device of Mufflon's pure path
// tracer (GpuPathTracer, gpu_pt.cu:54-152), every iteration of a call in one
// launch.
//
// A lane owns a pixel and runs its iterations one after the other (each
// continues the pixel's generator): pt_sample (pt_common.hpp:75-156) with the
// pinhole camera sample, BSDF sampling with Russian roulette
// (random_walk.hpp:38-112), next-event estimation through the light tree with
// MIS (light_tree_sampling.hpp:195-329, light_sampling.hpp), emission hits
// weighted with light_pdf (:340-412). At the end of each path it folds the
// iteration's targets into the running means of
// output_handler_variance.hpp:7-31 (no separate update pass, no atomics: each
// pixel belongs to one lane). The RNG is Mufflon's PCG64, one 64-bit state per
// pixel, seeded as in gpu_pt.cu:140-152.
//
// Float expressions keep the reference's operand order; transcendental
// functions of the samplers are evaluated in double and rounded once
// (correctly rounded sin/cos), the same definition as the CPU oracle's.
#include <algorithm>

#include "pt_path.hpp"

namespace mfh {

namespace {

using namespace shade;
using namespace path;

constexpr int kPtTile = 8;  // a wave starts on an 8x8 pixel tile
constexpr int kPtThreads = kPtTile * kPtTile;
// Path regeneration. Paths end after very different numbers of segments (2.5
// of 8 on average in the Cornell box), and a wave that runs one path per lane
// works until its longest has ended, a launch per iteration until the longest
// of the image has. So a turn of the loop below is one path segment (closest
// hit, vertex, next-event estimate, walk), and a lane whose path has ended
// starts its pixel's next iteration in the next turn, or takes another pixel
// from the queue once the call's iterations are done. Against one path per
// lane and one launch per iteration: Cornell box 256x256, 16 iterations 22.3
// -> 10.6 ms; terrain of 2.1M triangles and 2048 instances, 1280x720, 4
// iterations 31.5 -> 24.5 ms; one iteration of a 200x151 room 0.82 -> 0.55 ms
// (over binary nodes; 8.7, 19.9 and 0.45 ms over the wide ones).
// What bounds it now is the traversal's chain of dependent loads: in the Cornell
// box the vector units are busy 48 % of the time, with 8 % of the lanes active.
//
// The shadow ray of a vertex is traced after the walk from it (the random
// numbers of both are drawn before, in the order of pt_sample): through that
// traversal the vertex, about 45 registers, is no longer live.
//
// Three waves per SIMD: left to itself the compiler takes 256 VGPRs and more
// (one wave per SIMD), too few waves to hide the traversal's memory latency.
// kMode: traversal specialization (trace_mode_of: one instance, instance
// level, or a scene with quads or spheres).
// kNeeOne: at most one next-event estimate a vertex (several are traced one
// after the other, before the walk).
template <int kMode, bool kNeeOne>
__global__ __launch_bounds__(kPtThreads) __attribute__((amdgpu_waves_per_eu(3))) void k_pt_iterate(PtScene S, PathWork W,
                                                                                                  int tilesX) {
    __shared__ int sStack[kLdsDepth * kPtThreads];
    int* const lstack = sStack + threadIdx.x;
    auto any_hit = [&](const NeeCandidate& c) {
        return trace_mode<kMode, true, kPtThreads, kLdsDepth>(S.trace, c.a, c.dir, c.tmax, lstack).inst != -1;
    };
    SlotQueue slots(W);
    bool busy = false;             // the lane owns a pixel
    int px = 0, py = 0, done = 0;  // its position, its finished iterations
    int pathLen = 0;
    u64 rng = 0;
    Acc acc;
    acc.init(S.targetMask);
    float footA = 0.0f;  // FootprintV0::m_a (footprint.hpp:137-170)
    float pdfF = 1.0f;
    V3 throughput = v3(1.0f, 1.0f, 1.0f), rayOrigin = throughput, dir = throughput, absorption = throughput;
    V3 prevPos = throughput;
    while (true) {
        const int slot = slots.take(W, busy);
        if (slot >= 0) {
            const int tile = slot / kPtThreads, in = slot % kPtThreads;
            px = (tile % tilesX) * kPtTile + in % kPtTile;
            py = (tile / tilesX) * kPtTile + in / kPtTile;
            if (px < S.width && py < S.height) {
                busy = true;
                done = 0;
                pathLen = 0;
                rng = S.rngs[(size_t)px + (size_t)py * S.width];
            }
        }
        if (__ballot(busy) == 0ull && !slots.more) break;
        if (busy) {
            if (pathLen == 0) {  // the camera's sample
                acc.init(S.targetMask);
                footA = 0.0f;
                throughput = v3(1.0f, 1.0f, 1.0f);
                pcg_next(rng);  // create_camera's RndSet2, unused by the pinhole
                const u64 x0 = pcg_next(rng);
                pcg_next(rng);
                pcg_next(rng);  // the roulette always continues at throughput 1
                camera_ray(S, px, py, x0, dir, pdfF);
                rayOrigin = v3(S.camPos[0], S.camPos[1], S.camPos[2]);
                absorption = v3(0.0f, 0.0f, 0.0f);
                prevPos = rayOrigin;
            }
            const TraceHit hit =
                trace_mode<kMode, false, kPtThreads, kLdsDepth>(S.trace, rayOrigin, dir, kMaxSceneSize, lstack);
            throughput = throughput * transmission(Medium{1.0f, absorption}, hit.inst == -1 ? kMaxSceneSize : hit.t);
            footA += 1.0f / fsqrt(pdfF);
            const float guideWeight = 1.f / (1.f + footA * footA / 1.0f);
            Vertex vx;
            make_vertex(S, rayOrigin, dir, pdfF, hit.t, hit.inst, hit.prim, hit.w0, hit.w1, vx);
            ++pathLen;
            vertex_targets(S, vx, pathLen, throughput, guideWeight, acc, prevPos);
            bool ended = vx.isVoid || pathLen >= S.maxPathLength;
            if (!ended) {
                NeeCandidate c;
                bool shadow = false;
                if (pathLen + 1 >= S.minPathLength) {
                    const u64 neeSeed = pcg_next(rng);
                    if constexpr (kNeeOne) {
                        if (S.neeCount > 0)
                            shadow = nee_candidate(S, vx, throughput, guideWeight, 0, neeSeed, pcg_next(rng), c);
                    } else {
                        for (int i = 0; i < S.neeCount; ++i)
                            if (nee_candidate(S, vx, throughput, guideWeight, i, neeSeed, pcg_next(rng), c) &&
                                !any_hit(c))
                                add_nee(c, acc);
                    }
                }
                const u64 x0 = pcg_next(rng);
                const u64 x1 = pcg_next(rng);
                const float rndRoulette = sample_uniform((u32)pcg_next(rng));
                ended = !walk_surface(vx, x0, x1, rndRoulette, throughput, rayOrigin, dir, pdfF, absorption);
                prevPos = vx.position;
                if (shadow && !any_hit(c)) add_nee(c, acc);
            }
            if (ended) {
                const size_t pixel = (size_t)px + (size_t)py * S.width;
                accumulate(S, pixel, S.iteration + done, acc.v, acc.mask);
                if (acc.nans) atomicAdd(S.nanCounter, acc.nans);
                pathLen = 0;
                if (++done == W.iterations) {
                    S.rngs[pixel] = rng;
                    busy = false;
                }
            }
        }
    }
}

// rngs[i] = PCG64(u32(i + seed)) (gpu_pt.cu:140-144, rng.hpp:76-81)
__global__ void k_pt_init_rng(u64* rngs, int num, int seed) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= num) return;
    const u32 s = (u32)(i + seed);
    u64 st = scramble_seed(s);
    pcg_next(st);
    st += s;
    pcg_next(st);
    rngs[i] = st;
}

}  // namespace

void launch_pt_init_rng(u64* rngs, int num, int seed, hipStream_t stream) {
    hipLaunchKernelGGL(k_pt_init_rng, dim3((num + 255) / 256), dim3(256), 0, stream, rngs, num, seed);
    MFH_HIP(hipGetLastError());
}

// Fewest lanes of a wave that take pixels (64 / 32 / 16 / 8: Cornell box 256x256,
// 16 iterations, 11.8 / 10.7 / 8.9 / 8.7 ms, the last with 16 lanes as well by the
// rule below; one iteration of a 200x151 room 0.57 / 0.53 / 0.50 / 0.45 ms. The
// light tracer's Cornell box is fastest at 32: 12.2 / 11.6 / 14.1 / 14.0. The
// terrain image fills the chip and takes 64).
constexpr int kMinLanes = 8;

int path_work(const void* fn, int slots, int iterations, LaunchQueue& queue, int numCUs, PathWork& W) {
    // Lanes of a wave that take slots: all 64, or for launches too small to
    // give every resident wave 64 slots, half as many until they do. More
    // waves of fewer paths each hide one another's memory latency, and the
    // segment of a wave waits for the longest of fewer rays.
    const int resident = queue.blocks_per_cu(fn, 64) * numCUs;
    W.iterations = iterations;
    W.slots = slots;
    W.lanes = 64;
    while (W.lanes > kMinLanes && slots / W.lanes < resident) W.lanes /= 2;
    W.queue = queue.taken();
    W.nextQueue = queue.cleared();
    return std::min((slots + W.lanes - 1) / W.lanes, resident);
}

namespace {

using IterateFn = void (*)(PtScene, PathWork, int);

template <int kMode>
IterateFn iterate_kernel(bool neeOne) {
    return neeOne ? k_pt_iterate<kMode, true> : k_pt_iterate<kMode, false>;
}

}  // namespace

void launch_pt_iterate(const PtScene& S, int iterations, LaunchQueue& queue, int numCUs, hipStream_t stream) {
    const int mode = trace_mode_of(S.trace);
    const bool neeOne = S.neeCount <= 1;
    const IterateFn fn = mode == kTraceSingle       ? iterate_kernel<kTraceSingle>(neeOne)
                         : mode == kTraceMulti      ? iterate_kernel<kTraceMulti>(neeOne)
                         : mode == kTraceSingleTies ? iterate_kernel<kTraceSingleTies>(neeOne)
                         : mode == kTraceMultiTies  ? iterate_kernel<kTraceMultiTies>(neeOne)
                                                    : iterate_kernel<kTraceMixed>(neeOne);
    const int tilesX = (S.width + kPtTile - 1) / kPtTile;
    const int tiles = tilesX * ((S.height + kPtTile - 1) / kPtTile);
    PathWork W;
    const int grid = path_work(reinterpret_cast<const void*>(fn), tiles * kPtThreads, iterations, queue, numCUs, W);
    hipLaunchKernelGGL(fn, dim3(grid), dim3(kPtThreads), 0, stream, S, W, tilesX);
    MFH_HIP(hipGetLastError());
    queue.next ^= 1;
}

}  // namespace mfh
