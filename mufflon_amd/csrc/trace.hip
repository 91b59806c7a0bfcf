// Closest-hit and any-hit trace kernels over ray buffers, built on the
// traversal of traverse.hpp.
#include "traverse.hpp"

namespace mfh {

namespace {

constexpr int kThreads = 64;
constexpr int kCountThreads = 256;

// Persistent waves over the rays (trace_queue). kAny: stop at the first
// accepted hit. kSingle: the scene has one instance (no instance level).
// kMixed: the scene's LoDs hold quads or spheres. kTies: see Trav. Waves per
// SIMD: what the persistent traversal needs itself (up to 96 and 128 VGPRs; one
// wave more a SIMD spills in the loop: 1M-triangle trace with its build 2.48
// instead of 2.13 ms, instanced 1.65 instead of 0.92 ms).
template <bool kAny, bool kSingle, bool kMixed, bool kTies>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(kSingle ? 5 : 4))) void k_trace(
    TraceParams p, const float4* __restrict__ rays, int n, float4* __restrict__ hits, float2* __restrict__ bary,
    int* __restrict__ occluded, int lanes, int chunk, int split, int* queue, int* nextQueue) {
    __shared__ int sStack[kLdsDepth * kThreads];
    using T = Trav<kAny, kSingle, kMixed, kTies, kThreads, kLdsDepth>;
    if (blockIdx.x == 0 && (int)threadIdx.x < kTraceQueueSplit) nextQueue[kQueueStride * (int)threadIdx.x] = 0;
    WaveQueue q(n, lanes, chunk, (int)blockIdx.x, (int)gridDim.x, queue, split);
    trace_queue<T, kSingle ? 1 : 0>(
        q, sStack + threadIdx.x, [&](int) -> const TraceParams& { return p; },
        [&](int i, V3& o, V3& d, float& tmax) {
            const float4 r0 = rays[2 * (size_t)i], r1 = rays[2 * (size_t)i + 1];
            o = v3(r0.x, r0.y, r0.z);
            d = v3(r1.x, r1.y, r1.z);
            tmax = r0.w;
            return true;
        },
        [&](int i, const TraceHit& h) {
            if (kAny) {
                occluded[i] = h.overflow ? -1 : (h.inst != -1 ? 1 : 0);
            } else {
                hits[i] = make_float4(h.t, __int_as_float(h.inst), __int_as_float(h.prim), h.overflow ? 1.0f : 0.0f);
                if (bary) bary[i] = make_float2(h.w0, h.w1);
            }
        });
}

// Closest hits in the reference's order, with per-ray visit counts, one ray a
// lane (1M-triangle mesh, 1M incoherent rays: 1.5 ms; 2.7 ms with the stack in
// private memory and the number of instances found at run time).
template <bool kSingle, bool kMixed>
__global__ __launch_bounds__(kCountThreads) void k_trace_counts(TraceParams p, const float4* __restrict__ rays, int n,
                                                               float4* __restrict__ hits, float2* __restrict__ bary,
                                                               uint2* __restrict__ stats) {
    __shared__ int sStack[kLdsDepth * kCountThreads];
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float4 r0 = rays[2 * (size_t)i], r1 = rays[2 * (size_t)i + 1];
    const TraceHit h = binary_ray<false, true, kSingle ? 1 : 0, kMixed>(
        p, v3(r0.x, r0.y, r0.z), v3(r1.x, r1.y, r1.z), r0.w,
        BinaryStack<kCountThreads, kLdsDepth>{sStack + threadIdx.x, 0, false});
    hits[i] = make_float4(h.t, __int_as_float(h.inst), __int_as_float(h.prim), h.overflow ? 1.0f : 0.0f);
    if (bary) bary[i] = make_float2(h.w0, h.w1);
    stats[i] = make_uint2(h.nodeVisits, h.primTests);
}

using TraceFn = void (*)(TraceParams, const float4*, int, float4*, float2*, int*, int, int, int, int*, int*);

template <bool kAny, bool kSingle>
TraceFn trace_kernel(const TraceParams& p) {
    if (p.mixed) return k_trace<kAny, kSingle, true, !kAny>;
    return !kAny && p.flat ? k_trace<kAny, kSingle, false, !kAny> : k_trace<kAny, kSingle, false, false>;
}
template <bool kAny>
TraceFn trace_kernel(const TraceParams& p) {
    return p.numInstances == 1 ? trace_kernel<kAny, true>(p) : trace_kernel<kAny, false>(p);
}

void launch_trace(TraceFn fn, const TraceParams& p, const float* rays, int n, float4* hits, float2* bary, int* occ,
                  LaunchQueue& queue, int numCUs, hipStream_t stream) {
    const int resident = queue.blocks_per_cu(reinterpret_cast<const void*>(fn), kThreads) * numCUs;
    const int lanes = queue_lanes(n, resident);
    const int waves = std::min(resident, (n + lanes - 1) / lanes);
    // about four chunks a wave, at most 256 rays, so that the waves end together
    const int chunk = std::max(64, std::min(256, n / (4 * resident) / 64 * 64));
    hipLaunchKernelGGL(fn, dim3(waves), dim3(kThreads), 0, stream, p, reinterpret_cast<const float4*>(rays), n, hits,
                       bary, occ, lanes, chunk, std::min(queue.split, waves), queue.taken(), queue.cleared());
    MFH_HIP(hipGetLastError());
    queue.next ^= 1;
}

}  // namespace

int LaunchQueue::blocks_per_cu(const void* fn, int threads) {
    for (const auto& [known, blocks] : occupancy)
        if (known == fn) return blocks;
    int blocks = 0;
    MFH_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, fn, threads, 0));
    occupancy.emplace_back(fn, std::max(blocks, 1));
    return occupancy.back().second;
}

TraceParams trace_params(const Scene& sc) {
    TraceParams p;
    p.numInstances = sc.numInstances;
    p.worldToInst = sc.dWorldToInst.as<float>();
    p.instLod = sc.dInstLod.as<int32_t>();
    p.lods = sc.dLods.as<DevLod>();
    p.tlasNodes = sc.tlasNodes.ptr;
    p.tlasPrimIds = sc.tlasPrimIds.as<int32_t>();
    p.tlasNumInternal = sc.tlasNumInternal;
    p.tlasCoordMax = 0.0f;
    for (int k = 0; k < 6; ++k) p.tlasCoordMax = std::max(p.tlasCoordMax, std::fabs(sc.box[k]));
    p.mixed = sc.mixed ? 1 : 0;
    p.flat = sc.flat ? 1 : 0;
    return p;
}

void launch_trace_closest(const TraceParams& p, const float* rays, int n, float4* hits, float2* bary,
                          LaunchQueue& queue, int numCUs, hipStream_t stream) {
    if (n <= 0) return;
    launch_trace(trace_kernel<false>(p), p, rays, n, hits, bary, nullptr, queue, numCUs, stream);
}

void launch_trace_counts(const TraceParams& p, const float* rays, int n, float4* hits, float2* bary, uint2* stats,
                         hipStream_t stream) {
    if (n <= 0) return;
    auto* const fn = p.numInstances == 1 ? (p.mixed ? k_trace_counts<true, true> : k_trace_counts<true, false>)
                                         : (p.mixed ? k_trace_counts<false, true> : k_trace_counts<false, false>);
    hipLaunchKernelGGL(fn, dim3((n + kCountThreads - 1) / kCountThreads), dim3(kCountThreads), 0, stream, p,
                       reinterpret_cast<const float4*>(rays), n, hits, bary, stats);
    MFH_HIP(hipGetLastError());
}

void launch_trace_any(const TraceParams& p, const float* rays, int n, int32_t* occluded, LaunchQueue& queue,
                      int numCUs, hipStream_t stream) {
    if (n <= 0) return;
    launch_trace(trace_kernel<true>(p), p, rays, n, nullptr, nullptr, occluded, queue, numCUs, stream);
}

}  // namespace mfh
