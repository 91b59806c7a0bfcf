// BVH traversal (closest / any hit) as a device function shared by the trace
// kernels and the path tracer: the GPU device of Mufflon's first_intersection /
// any_intersection (intersection.cu:366-753).
//
// One ray per lane, through two levels: the instances over Mufflon's 64-byte
// collapsed LBVH nodes in the reference's order, the primitives of an object
// over its 4-wide traversal hierarchy (wide_node in lbvh.hip). The primitives of
// a leaf are contiguous 48-byte records in BVH order ({v0, primId}, {v1, kind},
// {v2} for triangles and quads, {center, primId}, {radius, .., kind} for
// spheres). The stack keeps its lowest kLdsDepth entries in LDS (one column
// per lane, so the 64 lanes of a wave touch 64 consecutive dwords) and spills
// deeper entries to a per-lane private array.
//
// A primitive is tested where its leaf's box, in full precision, passes the
// slab test of the reference CPU path (intersection.cu:57-75); the quantized
// boxes above contain that box and are tested with an error margin, so they
// only cull. (A node step replaces two binary ones, with half their dependent
// loads; 44 -> 23.5 steps a ray on a 1M-triangle mesh, 8.3 triangle tests.)
// Closest hit is the lexicographic minimum of (t, instance, primitive), which
// depends on the order inside an object only where surfaces coincide
// (Trav::test_leaf hands such rays to the reference's order); the order of the
// objects, whose entry and exit round the hit distance
// (intersection.cu:321-361), is the reference's.
#pragma once
#include "mfh_device.hpp"
#include "mfh_internal.hpp"

namespace mfh {

constexpr int kSentinel = (int)0xFFFFFFFF;
constexpr int kStackCap = 128;  // entries of the binary traversals
constexpr int kWideCap = 64;    // entries of the wide traversal; fuller stacks take reference_ray
constexpr int kLdsDepth = 16;

// A load of BVH-node or triangle data as a global-memory load: the pointers
// arrive in structs as generic pointers, whose loads would compile to flat
// loads that also wait on the LDS counter.
typedef float GlobalF4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ float4 gload(const float4* p) {
    const GlobalF4 v = *(const __attribute__((address_space(1))) GlobalF4*)p;
    return make_float4(v.x, v.y, v.z, v.w);
}

// An entry of a lane's LDS stack column, addressed as LDS so that a pop,
// which reads either the LDS column or the private spill array, keeps a
// ds_read and a scratch load instead of one flat load through a merged
// pointer.
__device__ __forceinline__ __attribute__((address_space(3))) int& lds_at(int* column, int i) {
    return ((__attribute__((address_space(3))) int*)column)[i];
}
__device__ __forceinline__ int lds_at(const int* column, int i) {
    return ((const __attribute__((address_space(3))) int*)column)[i];
}

// Slab test, reference CPU semantics (intersection.cu:57-75).
__device__ __forceinline__ bool slab(const float* lo, const float* hi, const FastRay& r, float tmax, float& cmin) {
    const float x0 = lo[0] * r.inv.x - r.odiv.x, x1 = hi[0] * r.inv.x - r.odiv.x;
    const float y0 = lo[1] * r.inv.y - r.odiv.y, y1 = hi[1] * r.inv.y - r.odiv.y;
    const float z0 = lo[2] * r.inv.z - r.odiv.z, z1 = hi[2] * r.inv.z - r.odiv.z;
    const float mnx = mn(x0, x1), mxx = mx(x0, x1);
    const float mny = mn(y0, y1), mxy = mx(y0, y1);
    const float mnz = mn(z0, z1), mxz = mx(z0, z1);
    const float cmx = mn(mn(mxx, mxy), mxz);
    cmin = mx(mx(mnx, mny), mnz);
    return (cmx >= 0.0f) && (cmin <= tmax) && (cmin <= cmx);
}

// The same slab test with the hardware min / max (v_min_f32, v_max_f32,
// v_min3_f32, v_max3_f32: about half the instructions of the compare-selects
// above, and no VCC wait states). Where no x0 .. z1 is NaN its accept / reject
// and the order of its entry distances equal slab()'s: the two min / max
// forms then differ at most in the sign of a zero result, and every use of
// cmx, cmin and the entry distances is a value comparison. slab_finite()
// tells a lane where that holds.
__device__ __forceinline__ bool slab_fast(const float* lo, const float* hi, const FastRay& r, float tmax,
                                          float& cmin) {
    const float x0 = lo[0] * r.inv.x - r.odiv.x, x1 = hi[0] * r.inv.x - r.odiv.x;
    const float y0 = lo[1] * r.inv.y - r.odiv.y, y1 = hi[1] * r.inv.y - r.odiv.y;
    const float z0 = lo[2] * r.inv.z - r.odiv.z, z1 = hi[2] * r.inv.z - r.odiv.z;
    const float cmx = __builtin_fminf(__builtin_fminf(__builtin_fmaxf(x0, x1), __builtin_fmaxf(y0, y1)),
                                      __builtin_fmaxf(z0, z1));
    cmin = __builtin_fmaxf(__builtin_fmaxf(__builtin_fminf(x0, x1), __builtin_fminf(y0, y1)),
                           __builtin_fminf(z0, z1));
    return (cmx >= 0.0f) && (cmin <= tmax) && (cmin <= cmx);
}

// True when the slab tests of ray r against boxes whose coordinates are at
// most coordMax in magnitude can produce no NaN: with |1/d| <= 2^64 on every
// axis and |origin|, coordMax <= 2^62 (node boxes are enlarged by 1.0001
// about their centre, so they stay within 2^63) every product is below
// 2^127 and every difference below 2^128, hence finite. A direction with a
// zero component (1/d infinite) or NaN input fails it.
__device__ __forceinline__ bool slab_finite(const FastRay& r, float coordMax) {
    constexpr float kInvMax = 18446744073709551616.0f;   // 2^64
    constexpr float kCoordMax = 4611686018427387904.0f;  // 2^62
    const float inv = __builtin_fmaxf(__builtin_fmaxf(fabsf(r.inv.x), fabsf(r.inv.y)), fabsf(r.inv.z));
    const float org = __builtin_fmaxf(__builtin_fmaxf(fabsf(r.o.x), fabsf(r.o.y)), fabsf(r.o.z));
    // written so that a NaN anywhere makes it false
    return inv <= kInvMax && org <= kCoordMax && coordMax <= kCoordMax && r.inv.x == r.inv.x &&
           r.inv.y == r.inv.y && r.inv.z == r.inv.z && r.o.x == r.o.x && r.o.y == r.o.y && r.o.z == r.o.z;
}

// Both child boxes of a node; fast (wave-uniform) selects slab_fast.
__device__ __forceinline__ void slab_pair(bool fast, const float* lLo, const float* lHi, const float* rLo,
                                          const float* rHi, const FastRay& r, float tmax, bool& t0, bool& t1,
                                          float& c0, float& c1) {
    if (fast) {
        t0 = slab_fast(lLo, lHi, r, tmax, c0);
        t1 = slab_fast(rLo, rHi, r, tmax, c1);
    } else {
        t0 = slab(lLo, lHi, r, tmax, c0);
        t1 = slab(rLo, rHi, r, tmax, c1);
    }
}

// Quad or sphere of a mixed LoD (intersects_primitve, intersection.cu:220-300,
// without alpha testing): the record (a, b, c) at sorted position pos, the
// quad's fourth vertex from quadV3.
struct PrimHit {
    float t, w0, w1;
    int hit;
};
__device__ __forceinline__ PrimHit prim_hit_other(const FastRay& r, float4 a, float4 b, float4 c,
                                                  const float4* quadV3, int pos) {
    PrimHit h;
    h.t = 0.0f;
    h.w0 = 0.0f;
    h.w1 = 0.0f;
    if (__float_as_int(b.w) == kPrimQuad) {
        const float4 d = quadV3[pos];
        h.hit = ray_quad(r, v3(a.x, a.y, a.z), v3(b.x, b.y, b.z), v3(c.x, c.y, c.z), v3(d.x, d.y, d.z), h.t, h.w0,
                         h.w1)
                    ? 1
                    : 0;
    } else {
        h.hit = ray_sphere(r, v3(a.x, a.y, a.z), b.x, h.t) ? 1 : 0;
    }
    return h;
}

// Test of the primitive whose 48-byte record (a, b, c) sits at sorted
// position pos of a LoD: true with t > 0 and the surface parameters (the
// barycentric weights of v0 and v1, or a quad's (u, v)). quadV3() yields the
// LoD's fourth quad vertices; it is only evaluated for a quad. kMixed: the
// scene has LoDs with quads or spheres; without, every record is a triangle
// and the kernels carry no quad or sphere code (the quad test alone would
// raise the single-instance trace kernel from 53 to 70 VGPRs, 8 to 7 waves).
template <bool kMixed, class QuadV3>
__device__ __forceinline__ bool prim_hit(const FastRay& r, float4 a, float4 b, float4 c, int pos, QuadV3 quadV3,
                                         float& t, float& w0, float& w1) {
    if (!kMixed || __float_as_int(b.w) == kPrimTriangle)
        return ray_triangle(r, v3(a.x, a.y, a.z), v3(b.x, b.y, b.z), v3(c.x, c.y, c.z), t, w0, w1) && t > 0.0f;
    const PrimHit h = prim_hit_other(r, a, b, c, __float_as_int(b.w) == kPrimQuad ? quadV3() : nullptr, pos);
    t = h.t;
    w0 = h.w0;
    w1 = h.w1;
    return h.hit != 0;
}

// Accept a hit closer than the current one; at equal distance the lower
// (instance, primitive) pair wins. A hit exactly at the initial tmax (no hit
// yet) is rejected, as the reference's strict t < tmax test does.
__device__ __forceinline__ bool better(float t, int inst, int prim, float hitT, int hInst, int hPrim) {
    if (t < hitT) return true;
    if (t > hitT || hInst == -1) return false;
    if (inst != hInst) return inst < hInst;
    return prim < hPrim;
}

// The instance transition of world_to_object_space (intersection.cu:321-349):
// transform the world ray into the instance, scale tmax, test the object box.
struct ObjectEntry {
    FastRay ray;
    float scale, tmax;
    bool hit;
};
__device__ __forceinline__ ObjectEntry enter_object(const TraceParams& p, int inst, V3 wo, V3 wd, float hitT,
                                                    DevLod& lod) {
    ObjectEntry e;
    const float4* w = reinterpret_cast<const float4*>(p.worldToInst + 12 * (size_t)inst);
    const float4 a = w[0], b = w[1], c = w[2];
    const M34 M{{a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w, c.x, c.y, c.z, c.w}};
    const V3 d = xform_dir(M, wd);
    e.scale = len(d);
    e.ray = make_fast_ray(xform_point(M, wo), d / e.scale);
    e.tmax = hitT * e.scale;
    lod = p.lods[p.instLod[inst]];
    float ot;
    e.hit = slab(lod.box, lod.box + 3, e.ray, e.tmax, ot);
    return e;
}


struct TraceHit {
    float t;
    int inst, prim;
    float w0, w1;
    bool overflow;
    unsigned nodeVisits, primTests;
};

// Stack of the binary traversal: the lowest entries in this lane's LDS column,
// the deeper ones in the private array `spill` of the caller (an array in here
// would keep the scalars beside it in private memory).
template <int kStride, int kLds>
struct BinaryStack {
    static constexpr int kSpill = kStackCap - kLds;
    int* lds;
    int sp;
    bool overflow;
    __device__ __forceinline__ void push(int* spill, int v) {
        if (sp < kLds)
            lds_at(lds, sp * kStride) = v;
        else if (sp < kStackCap)
            spill[sp - kLds] = v;
        if (sp < kStackCap)
            ++sp;
        else
            overflow = true;
    }
    __device__ __forceinline__ int pop(const int* spill) {
        --sp;
        return sp < kLds ? lds_at((const int*)lds, sp * kStride) : spill[sp - kLds];
    }
};

// The leaves of the reference's BVH are cut into parts of at most the traversal
// leaf limit for the wide nodes; a leaf longer than this is walked part by part
// where nothing is counted. (A heightfield's longest leaves hold some 1400
// triangles, a sphere's poles 570.)
constexpr int kLongLeaf = 16;

// True when the ray can hit nothing inside the box before tmax: the slab test
// with a margin for its rounding (make_wide_ray), and on an axis along which the
// ray does not move whether it runs beside the box. NaN makes it false.
__device__ __forceinline__ bool surely_missed(V3 lo, V3 hi, const FastRay& r, float coordMax, float tmax) {
    float enter = 0.0f, leave = tmax;
    bool beside = false;
    auto axis = [&](float l, float h, float o, float inv) {
        const float m = (fabsf(o) + coordMax) * 0x1p-21f;
        beside |= (o < l - m && inv <= 0.0f) || (o > h + m && inv >= 0.0f);
        if (fabsf(inv) <= 18446744073709551616.0f) {
            const float e = m * fabsf(inv), a = (l - o) * inv, b = (h - o) * inv;
            enter = __builtin_fmaxf(enter, __builtin_fminf(a, b) - e);
            leave = __builtin_fminf(leave, __builtin_fmaxf(a, b) + e);
        } else {
            beside |= o < l - m || o > h + m;
        }
    };
    axis(lo.x, hi.x, r.o.x, r.inv.x);
    axis(lo.y, hi.y, r.o.y, r.inv.y);
    axis(lo.z, hi.z, r.o.z, r.inv.z);
    return beside || enter > leave;
}

// Closest or any hit over the reference's BVHs in its order (nearer child
// first with ties to the left, the farther child pushed, leaves pushed as
// (count, index)). kInstances: 1 one instance (no instance level), 0 instance
// level, 2 one of them at run time. kCount: the visit counts (internal nodes
// visited, an object-box test at instance entry among them, and primitives
// tested).
template <bool kAny, bool kCount, int kInstances, bool kMixed, class Stack>
__device__ __forceinline__ TraceHit binary_ray(const TraceParams& p, V3 wo, V3 wd, float tmax, Stack st) {
    int spill[Stack::kSpill];
    st.sp = 0;
    st.overflow = false;
    const bool single = kInstances == 2 ? p.numInstances == 1 : kInstances == 1;
    FastRay cur = make_fast_ray(wo, wd);
    float hitT = tmax;
    int hInst = -1, hPrim = -1;
    float hw0 = 0.0f, hw1 = 0.0f;
    float scale = 1.0f;
    unsigned nodeVisits = 0, primTests = 0;

    // current level: the instance BVH or the BVH of the entered object
    const BvhChild* bvh = (const BvhChild*)p.tlasNodes;
    const float4* tris = nullptr;
    int numInternal = p.tlasNumInternal;
    int objPrims = 0;
    bool inObj = false;
    int curInst = -1;
    int nodeAddr = 0, primCount = 2, primOffset = 0;
    bool done = false;
    // no NaN can reach this lane's slab tests at the current level
    bool finite = slab_finite(cur, p.tlasCoordMax);
    const float4* leafBoxes = nullptr;
    float coordMax = 0.0f;
    int part = 0;  // primitives left of the entered part of a long leaf

    if (single) {
        DevLod lod;
        const ObjectEntry e = enter_object(p, 0, wo, wd, hitT, lod);
        if (kCount) ++nodeVisits;
        if (!e.hit) {
            primCount = 0;
        } else {
            cur = e.ray;
            finite = slab_finite(cur, lod.coordMax);
            scale = e.scale;
            hitT = e.tmax;
            bvh = (const BvhChild*)lod.nodes;
            tris = lod.triVerts;
            leafBoxes = lod.leafBoxes;
            coordMax = lod.coordMax;
            numInternal = lod.numInternal;
            inObj = true;
            curInst = 0;
            if (lod.numPrims == 1) primCount = 1;
        }
    }

    while (true) {
        // descend through internal nodes, nearer child first, farther pushed
        while (nodeAddr < numInternal && primCount > 0) {
            const float4* nd = reinterpret_cast<const float4*>(bvh + 2 * (size_t)nodeAddr);
            const float4 q0 = gload(nd), q1 = gload(nd + 1), q2 = gload(nd + 2), q3 = gload(nd + 3);
            if (kCount) ++nodeVisits;
            const float lLo[3] = {q0.x, q0.y, q0.z}, lHi[3] = {q0.w, q1.x, q1.y};
            const float rLo[3] = {q2.x, q2.y, q2.z}, rHi[3] = {q2.w, q3.x, q3.y};
            const int lIdx = __float_as_int(q1.z), lCnt = __float_as_int(q1.w);
            const int rIdx = __float_as_int(q3.z), rCnt = __float_as_int(q3.w);
            float c0, c1;
            bool t0, t1;
            slab_pair(__all(finite), lLo, lHi, rLo, rHi, cur, hitT, t0, t1, c0, c1);
            if (!t0) c0 = 1e38f;
            if (!t1) c1 = 1e38f;
            if (t0 && t1) {
                const bool farLeft = c1 < c0;
                const int far = farLeft ? lIdx : rIdx;
                if (far >= numInternal) st.push(spill, farLeft ? lCnt : rCnt);
                st.push(spill, far);
            }
            const bool nearLeft = c0 <= c1;
            nodeAddr = nearLeft ? lIdx : rIdx;
            primCount = (nodeAddr >= numInternal) ? (nearLeft ? lCnt : rCnt) : 2;
            primOffset = 0;
            if (!t0 && !t1) primCount = 0;
        }
        if (st.overflow) break;
        // the primitives of a leaf, one after the other
        bool descend = false;
        while (nodeAddr >= numInternal && primCount > 0) {
            if (!kCount && (single || inObj)) {
                if (part == 0 && primCount > kLongLeaf) {
                    const float4* bx = leafBoxes + 2 * (size_t)(nodeAddr - numInternal + primOffset);
                    const float4 b0 = gload(bx), b1 = gload(bx + 1);
                    part = __float_as_int(b1.z);
                    if (surely_missed(v3(b0.x, b0.y, b0.z), v3(b0.w, b1.x, b1.y), cur, coordMax, hitT)) {
                        primOffset += part;
                        primCount -= part;
                        part = 0;
                        continue;
                    }
                }
                if (part > 0) --part;
            }
            const int leafId = nodeAddr - numInternal + primOffset;
            ++primOffset;
            --primCount;
            if (!single && !inObj) {
                // an instance of the top level: enter its object
                const int inst = p.tlasPrimIds[leafId];
                DevLod lod;
                const ObjectEntry e = enter_object(p, inst, wo, wd, hitT, lod);
                if (kCount) ++nodeVisits;
                if (!e.hit) continue;
                if (lod.numPrims == 1) {
                    // single-primitive object: test it and return to the instance level
                    const float4 a = lod.triVerts[0], b = lod.triVerts[1], c = lod.triVerts[2];
                    float t, w0, w1;
                    if (kCount) ++primTests;
                    const float objT = e.tmax;
                    float ht = objT;
                    if (prim_hit<kMixed>(e.ray, a, b, c, 0, [&] { return lod.quadV3; }, t, w0, w1) &&
                        better(t, inst, __float_as_int(a.w), ht, hInst, hPrim)) {
                        ht = t;
                        hInst = inst;
                        hPrim = __float_as_int(a.w);
                        hw0 = w0;
                        hw1 = w1;
                        if (kAny) done = true;
                    }
                    hitT = ht / e.scale;
                    if (done) break;
                    continue;
                }
                if (primCount > 0) {
                    st.push(spill, primCount);
                    st.push(spill, nodeAddr + primOffset);
                }
                st.push(spill, kSentinel);
                cur = e.ray;
                finite = slab_finite(cur, lod.coordMax);
                scale = e.scale;
                hitT = e.tmax;
                bvh = (const BvhChild*)lod.nodes;
                tris = lod.triVerts;
                leafBoxes = lod.leafBoxes;
                coordMax = lod.coordMax;
                numInternal = lod.numInternal;
                objPrims = lod.numPrims;
                inObj = true;
                curInst = inst;
                nodeAddr = 0;
                primCount = objPrims == 1 ? 1 : 2;
                primOffset = 0;
                descend = true;
                break;
            }
            const float4 a = gload(tris + 3 * (size_t)leafId), b = gload(tris + 3 * (size_t)leafId + 1),
                         c = gload(tris + 3 * (size_t)leafId + 2);
            float t, w0, w1;
            const int prim = __float_as_int(a.w);
            if (kCount) ++primTests;
            if (prim_hit<kMixed>(cur, a, b, c, leafId, [&] { return p.lods[p.instLod[single ? 0 : curInst]].quadV3; },
                                 t, w0, w1) &&
                better(t, curInst, prim, hitT, hInst, hPrim)) {
                hitT = t;
                hInst = curInst;
                hPrim = prim;
                hw0 = w0;
                hw1 = w1;
                if (kAny) {
                    done = true;
                    break;
                }
            }
        }
        if (done || st.overflow) break;
        if (descend) continue;
        // pop the next subtree (or return from an object to the instance level)
        if (st.sp == 0) break;
        nodeAddr = st.pop(spill);
        if (!single && nodeAddr == kSentinel) {
            if (st.sp == 0) break;
            cur = make_fast_ray(wo, wd);
            finite = slab_finite(cur, p.tlasCoordMax);
            hitT /= scale;
            scale = 1.0f;
            bvh = (const BvhChild*)p.tlasNodes;
            numInternal = p.tlasNumInternal;
            inObj = false;
            nodeAddr = st.pop(spill);
        }
        primCount = (nodeAddr >= numInternal) ? st.pop(spill) : 2;
        primOffset = 0;
    }
    if (!kAny && inObj) hitT /= scale;  // object_to_world_space
    TraceHit h;
    h.t = hitT;
    h.inst = hInst;
    h.prim = hPrim;
    h.w0 = hw0;
    h.w1 = hw1;
    h.overflow = st.overflow;
    h.nodeVisits = nodeVisits;
    h.primTests = primTests;
    return h;
}

// The same as a call, for the rays that the wide traversals hand over: rays
// whose slab values may be NaN (slab_finite), rays that fill the wide stack and
// rays among coinciding surfaces. Its registers and its stack burden no kernel's
// main path. The call takes the scene's pointers one by one: a reference would
// make the kernels keep their argument block in private memory.
template <bool kAny, bool kMixed, int kInstances>
__device__ __attribute__((noinline, cold)) TraceHit reference_call(int numInstances, const float* worldToInst,
                                                             const int32_t* instLod, const DevLod* lods,
                                                             const void* tlasNodes, const int32_t* tlasPrimIds,
                                                             int tlasNumInternal, float tlasCoordMax, V3 wo, V3 wd,
                                                             float tmax) {
    TraceParams p;
    p.numInstances = numInstances;
    p.worldToInst = worldToInst;
    p.instLod = instLod;
    p.lods = lods;
    p.tlasNodes = tlasNodes;
    p.tlasPrimIds = tlasPrimIds;
    p.tlasNumInternal = tlasNumInternal;
    p.tlasCoordMax = tlasCoordMax;
    return binary_ray<kAny, false, kInstances, kMixed>(p, wo, wd, tmax, BinaryStack<1, 0>{nullptr, 0, false});
}
template <bool kAny, bool kMixed, int kInstances>
__device__ __forceinline__ TraceHit reference_ray(const TraceParams& p, V3 wo, V3 wd, float tmax) {
    return reference_call<kAny, kMixed, kInstances>(p.numInstances, p.worldToInst, p.instLod, p.lods, p.tlasNodes,
                                                    p.tlasPrimIds, p.tlasNumInternal, p.tlasCoordMax, wo, wd, tmax);
}

// A ray in an object's space for the wide nodes: the margin (in distance along
// the ray, per axis) covers the rounding of a quantized plane's distance and of
// the full-precision slab test it stands for. In units of 2^-23 (|origin| +
// |coordinate|) / |direction| the slab test has three roundings, below 1; the
// quantized plane one half each for the node's origin less the ray's, for the fma
// that offsets it, for the last fma, and up to 1 for the scale times a byte (the
// grid spans twice |coordinate| where the node does): 2.5. Together 3.5 of the 4
// that the margin has, so it cannot be halved.
struct WideRay {
    V3 o, inv, eps;
};
__device__ __forceinline__ WideRay make_wide_ray(const FastRay& r, float coordMax) {
    WideRay w;
    w.o = r.o;
    w.inv = r.inv;
    w.eps = v3((fabsf(r.o.x) + coordMax) * fabsf(r.inv.x) * 0x1p-21f,
               (fabsf(r.o.y) + coordMax) * fabsf(r.inv.y) * 0x1p-21f,
               (fabsf(r.o.z) + coordMax) * fabsf(r.inv.z) * 0x1p-21f);
    return w;
}

// Byte k of q as a float (v_cvt_f32_ubyte).
template <int k>
__device__ __forceinline__ float ubyte(u32 q) {
    return (float)((q >> (8 * k)) & 0xFFu);
}

// One step through wide node `node`: the children that the ray may enter
// before hitT as sort keys (entry distance with the child's number in the two
// lowest bits, top bit set; 0: not entered) in descending order, so that the
// entered children come first, the farthest leading.
constexpr u32 kWideNone = 0xFFFFFFFFu;
struct WideStep {
    u32 key[4];
    u32 child[4];
    __device__ __forceinline__ u32 ref(u32 k) const {
        const u32 lo = (k & 1u) ? child[1] : child[0], hi = (k & 1u) ? child[3] : child[2];
        return (k & 2u) ? hi : lo;
    }
};
template <int k>
__device__ __forceinline__ u32 wide_key(u32 nx, u32 ny, u32 nz, u32 fx, u32 fy, u32 fz, V3 a, V3 bn, V3 bf,
                                        float hitT) {
    const float tn = __builtin_fmaxf(__builtin_fmaxf(__builtin_fmaxf(__builtin_fmaf(ubyte<k>(nx), a.x, bn.x),
                                                                     __builtin_fmaf(ubyte<k>(ny), a.y, bn.y)),
                                                     __builtin_fmaf(ubyte<k>(nz), a.z, bn.z)),
                                     0.0f);
    const float tf = __builtin_fminf(__builtin_fminf(__builtin_fminf(__builtin_fmaf(ubyte<k>(fx), a.x, bf.x),
                                                                     __builtin_fmaf(ubyte<k>(fy), a.y, bf.y)),
                                                     __builtin_fmaf(ubyte<k>(fz), a.z, bf.z)),
                                     hitT);
    return tn <= tf ? ((__float_as_uint(tn) & 0x7FFFFFFCu) | (0x80000000u | (u32)k)) : 0u;
}
__device__ __forceinline__ WideStep wide_step(const float4* __restrict__ nodes, u32 node, const WideRay& w,
                                              float hitT) {
    const float4* nd = nodes + 4 * (size_t)node;
    const float4 n0 = gload(nd), n1 = gload(nd + 1), n2 = gload(nd + 2), n3 = gload(nd + 3);
    const V3 inv = w.inv;
    const V3 a = v3(n0.w * inv.x, n1.x * inv.y, n1.y * inv.z);
    const V3 off = v3(n0.x - w.o.x, n0.y - w.o.y, n0.z - w.o.z);
    const V3 bn = v3(__builtin_fmaf(off.x, inv.x, -w.eps.x), __builtin_fmaf(off.y, inv.y, -w.eps.y),
                     __builtin_fmaf(off.z, inv.z, -w.eps.z));
    const V3 bf = v3(__builtin_fmaf(off.x, inv.x, w.eps.x), __builtin_fmaf(off.y, inv.y, w.eps.y),
                     __builtin_fmaf(off.z, inv.z, w.eps.z));
    const u32 lx = __float_as_uint(n1.z), ly = __float_as_uint(n1.w), lz = __float_as_uint(n2.x);
    const u32 hx = __float_as_uint(n2.y), hy = __float_as_uint(n2.z), hz = __float_as_uint(n2.w);
    const bool sx = inv.x < 0.0f, sy = inv.y < 0.0f, sz = inv.z < 0.0f;
    const u32 nx = sx ? hx : lx, ny = sy ? hy : ly, nz = sz ? hz : lz;
    const u32 fx = sx ? lx : hx, fy = sy ? ly : hy, fz = sz ? lz : hz;
    WideStep r;
    r.key[0] = wide_key<0>(nx, ny, nz, fx, fy, fz, a, bn, bf, hitT);
    r.key[1] = wide_key<1>(nx, ny, nz, fx, fy, fz, a, bn, bf, hitT);
    r.key[2] = wide_key<2>(nx, ny, nz, fx, fy, fz, a, bn, bf, hitT);
    r.key[3] = wide_key<3>(nx, ny, nz, fx, fy, fz, a, bn, bf, hitT);
    auto order = [&](int x, int y) {
        const u32 hi = r.key[x] > r.key[y] ? r.key[x] : r.key[y], lo = r.key[x] > r.key[y] ? r.key[y] : r.key[x];
        r.key[x] = hi;
        r.key[y] = lo;
    };
    order(0, 1);
    order(2, 3);
    order(0, 2);
    order(1, 3);
    order(1, 2);
    r.child[0] = __float_as_uint(n3.x);
    r.child[1] = __float_as_uint(n3.y);
    r.child[2] = __float_as_uint(n3.z);
    r.child[3] = __float_as_uint(n3.w);
    return r;
}

// Stack of a lane: its LDS column (stride kStride), deeper entries in the
// private array `spill` of the caller.
template <int kStride, int kLds>
struct WideStack {
    int* lds;
    int sp;
    bool overflow;  // a push found the stack full
    __device__ __forceinline__ void push(int* spill, int v) {
        if (sp < kLds)
            lds_at(lds, sp * kStride) = v;
        else if (sp < kWideCap)
            spill[sp - kLds] = v;
        if (sp < kWideCap)
            ++sp;
        else
            overflow = true;
    }
    __device__ __forceinline__ int pop(const int* spill) {
        --sp;
        int v = lds_at(lds, (sp < kLds ? sp : kLds - 1) * kStride);
        if (sp >= kLds) v = spill[sp - kLds];
        return v;
    }
    // The entered children of a step: the nearest is returned (kWideNone:
    // none), the others go on the stack, the farthest first. The column takes
    // three entries at once, entered or not (what lies above sp is free).
    __device__ __forceinline__ u32 take(int* spill, const WideStep& r) {
        const bool e0 = r.key[0] != 0u, e1 = r.key[1] != 0u, e2 = r.key[2] != 0u, e3 = r.key[3] != 0u;
        const u32 c0 = r.ref(r.key[0]), c1 = r.ref(r.key[1]), c2 = r.ref(r.key[2]), c3 = r.ref(r.key[3]);
        if (sp + 3 <= kLds) {
            lds_at(lds, sp * kStride) = (int)c0;
            lds_at(lds, (sp + 1) * kStride) = (int)c1;
            lds_at(lds, (sp + 2) * kStride) = (int)c2;
            sp += (e1 ? 1 : 0) + (e2 ? 1 : 0) + (e3 ? 1 : 0);
        } else {
            if (e1) push(spill, (int)c0);
            if (e2) push(spill, (int)c1);
            if (e3) push(spill, (int)c2);
        }
        return e3 ? c3 : (e2 ? c2 : (e1 ? c1 : (e0 ? c0 : kWideNone)));
    }
};

// What the traversal of an object reads of its LoD.
struct ObjectData {
    const float4 *wide, *leafBoxes, *triVerts, *quadV3;
};
__device__ __forceinline__ ObjectData object_data(const DevLod& lod) {
    return {lod.wide, lod.leafBoxes, lod.triVerts, lod.quadV3};
}

// The traversal of one ray, resumable: run() returns when the ray is done or
// when fewer than `minActive` lanes of the wave are still under way, so that
// the caller can hand new rays to the lanes that are done. kSingle: one
// instance (else the instance level, or one instance found at run time).
//
// (1M-triangle mesh, 2.1M camera and 2.1M incoherent rays: 2.98 ms with a ray
// per lane over binary nodes, 1.88 over wide nodes with the lanes handed new
// rays: 24 -> 40 % of the lanes active. What bounds it now: the vector units are
// busy 80 % of the time at that utilization, and the L2 misses stream at the rate
// of a large copy, 4.7 TB/s.)
//
// A turn of run() takes the lanes between objects to their next one (over the
// binary nodes of the instances, in the reference's order), and the lanes
// inside one through node steps with postponed leaves (Aila and Laine 2009,
// "speculative while-while"): a lane that reaches a leaf keeps it and goes on
// descending until it reaches a second one or half of the active lanes hold
// one; then the held leaves are tested, so node steps and leaf tests run with
// more lanes active.
template <bool kAny, bool kSingle, bool kMixed, bool kTies, int kStride, int kLds>
struct Trav {
    static constexpr int kSpill = kWideCap - kLds;
    static constexpr bool kAnyHit = kAny, kMixedLods = kMixed;
    using Binary = BinaryStack<kStride, kLds>;
    WideStack<kStride, kLds> st;
    V3 wo, wd;         // the ray in world space (kSingle: unused)
    V3 dir;            // in the entered object's space, with w
    WideRay w;
    float hitT, scale;
    int hInst, hPrim;
    float hw0, hw1;
    ObjectData data;   // of the entered object (kSingle: see object())
    int inst, base;    // the entered object, the stack height at its entry
    int node, count, offset;  // instance level: node (count 2) or the rest of a leaf
    u32 cur, held;     // node or leaf to do next, the postponed leaf
    bool inObj, done, exact;  // exact: the ray is reference_ray's
    bool flat;                // kTies: the best hit lies before the entry of its leaf's box

    __device__ __forceinline__ void enter(const ObjectEntry& e, const DevLod& lod, int instance) {
        inst = instance;
        hitT = e.tmax;
        scale = e.scale;
        if (!slab_finite(e.ray, lod.coordMax)) {
            exact = done = true;
            return;
        }
        w = make_wide_ray(e.ray, lod.coordMax);
        dir = e.ray.d;
        if (!kSingle) data = object_data(lod);
        base = st.sp;
        inObj = true;
        cur = 0u;
        held = kWideNone;
        if (kTies) flat = false;
    }
    // An object of a single primitive: tested at once. The hit distance takes
    // the way through the object's space and back as for any entered object.
    __device__ __forceinline__ void single_prim(const ObjectEntry& e, const DevLod& lod, int instance) {
        const float4 a = lod.triVerts[0], b = lod.triVerts[1], c = lod.triVerts[2];
        float t, w0, w1, ht = e.tmax;
        if (prim_hit<kMixed>(e.ray, a, b, c, 0, [&] { return lod.quadV3; }, t, w0, w1) &&
            better(t, instance, __float_as_int(a.w), ht, hInst, hPrim)) {
            ht = t;
            hInst = instance;
            hPrim = __float_as_int(a.w);
            hw0 = w0;
            hw1 = w1;
        }
        hitT = ht / e.scale;
    }
    __device__ __forceinline__ void init(const TraceParams& p, V3 o, V3 d, float maxT, int* lstack) {
        st.lds = lstack;
        st.sp = 0;
        st.overflow = false;
        if (!kSingle) {
            wo = o;
            wd = d;
        }
        hitT = maxT;
        hInst = hPrim = -1;
        hw0 = hw1 = 0.0f;
        scale = 1.0f;
        if (kTies) flat = false;
        inObj = done = exact = false;
        cur = held = kWideNone;
        node = count = offset = 0;
        base = 0;
        if (kSingle || p.numInstances == 1) {
            DevLod lod;
            const ObjectEntry e = enter_object(p, 0, o, d, maxT, lod);
            done = true;
            if (!e.hit) return;
            if (lod.numPrims == 1) {
                single_prim(e, lod, 0);
                return;
            }
            done = false;
            enter(e, lod, 0);
        } else {
            count = 2;
        }
    }
    // Instance level: to the next object, or done.
    __device__ __forceinline__ void next_object(const TraceParams& p, int* spill) {
        const BvhChild* const tlas = (const BvhChild*)p.tlasNodes;
        const int tlasInternal = p.tlasNumInternal;
        const FastRay world = make_fast_ray(wo, wd);
        const bool finite = slab_finite(world, p.tlasCoordMax);
        while (true) {
            while (node < tlasInternal && count > 0) {
                const float4* nd = reinterpret_cast<const float4*>(tlas + 2 * (size_t)node);
                const float4 q0 = gload(nd), q1 = gload(nd + 1), q2 = gload(nd + 2), q3 = gload(nd + 3);
                const float lLo[3] = {q0.x, q0.y, q0.z}, lHi[3] = {q0.w, q1.x, q1.y};
                const float rLo[3] = {q2.x, q2.y, q2.z}, rHi[3] = {q2.w, q3.x, q3.y};
                const int lIdx = __float_as_int(q1.z), lCnt = __float_as_int(q1.w);
                const int rIdx = __float_as_int(q3.z), rCnt = __float_as_int(q3.w);
                float c0, c1;
                bool t0, t1;
                slab_pair(__all(finite), lLo, lHi, rLo, rHi, world, hitT, t0, t1, c0, c1);
                if (!t0) c0 = 1e38f;
                if (!t1) c1 = 1e38f;
                if (t0 && t1) {
                    const bool farLeft = c1 < c0;
                    const int far = farLeft ? lIdx : rIdx;
                    if (far >= tlasInternal) st.push(spill, farLeft ? lCnt : rCnt);
                    st.push(spill, far);
                }
                const bool nearLeft = c0 <= c1;
                node = nearLeft ? lIdx : rIdx;
                count = (!t0 && !t1) ? 0 : (node >= tlasInternal ? (nearLeft ? lCnt : rCnt) : 2);
                offset = 0;
            }
            while (count > 0 && !inObj && !done) {
                const int instance = p.tlasPrimIds[node - tlasInternal + offset];
                ++offset;
                --count;
                DevLod lod;
                const ObjectEntry e = enter_object(p, instance, wo, wd, hitT, lod);
                if (!e.hit) continue;
                if (lod.numPrims == 1) {
                    single_prim(e, lod, instance);
                    if (kAny && hInst != -1) done = true;
                } else {
                    enter(e, lod, instance);
                }
            }
            if (st.overflow) exact = done = true;
            if (inObj || done) return;
            if (st.sp == 0) {
                done = true;
                return;
            }
            node = st.pop(spill);
            count = node >= tlasInternal ? st.pop(spill) : 2;
            offset = 0;
        }
    }
    // The primitives of the held leaf: its box, then its records, the next one
    // loaded while one is tested.
    //
    // Where surfaces coincide in flat boxes the closest hit depends on the order
    // of the leaves: such a box has no extent along its normal, so the rounded
    // distance at which a ray enters it may exceed that of the hit inside
    // (entry > t), and whether a second leaf is still entered once a hit is known
    // then depends on which came first. So with kTies a leaf that is entered past
    // the hit by no more than the rounding (make_wide_ray's margin) is tested too,
    // and the ray is the reference traversal's (exact) when it holds a closer hit,
    // or when a hit lies that close behind a best one with entry > t. (1 ray in
    // 1300 in a room whose boxes stand on the floor, none in 10M rays of the
    // Cornell box. kTies takes 1.05 times the time on the 1M-triangle mesh and in
    // the Cornell box, so scenes without flat leaves go without.)
    __device__ __forceinline__ void test_leaf(const ObjectData& od) {
        const u32 first = held & ~kWideLeaf;
        held = kWideNone;
        const float4* bx = od.leafBoxes + 2 * (size_t)first;
        const float4 b0 = gload(bx), b1 = gload(bx + 1);
        const float4* rec = od.triVerts + 3 * (size_t)first;
        float4 a = gload(rec), b = gload(rec + 1), c = gload(rec + 2);
        const float lo[3] = {b0.x, b0.y, b0.z}, hi[3] = {b0.w, b1.x, b1.y};
        const FastRay r{w.o, dir, w.inv, w.o * w.inv};
        float entry;
        bool late = false;
        if constexpr (kTies) {
            float margin = 0.0f;
            if (hInst == inst) margin = __builtin_fmaxf(__builtin_fmaxf(w.eps.x, w.eps.y), w.eps.z);
            if (!slab_fast(lo, hi, r, hitT + margin, entry)) return;
            late = entry > hitT;
        } else {
            if (!slab_fast(lo, hi, r, hitT, entry)) return;
        }
        const int n = __float_as_int(b1.z);
        for (int k = 0;;) {
            float4 na = a, nb = b, nc = c;
            if (k + 1 < n) {
                rec += 3;
                na = gload(rec);
                nb = gload(rec + 1);
                nc = gload(rec + 2);
            }
            float t, w0, w1;
            const int prim = __float_as_int(a.w);
            if (prim_hit<kMixed>(r, a, b, c, (int)first + k, [&] { return od.quadV3; }, t, w0, w1)) {
                if (better(t, inst, prim, hitT, hInst, hPrim)) {
                    if (kTies && late) {
                        exact = done = true;
                        return;
                    }
                    hitT = t;
                    hInst = inst;
                    hPrim = prim;
                    hw0 = w0;
                    hw1 = w1;
                    if (kTies) flat = t < entry;
                    if (kAny) {
                        done = true;
                        return;
                    }
                } else if (kTies && flat && hInst == inst &&
                           t - hitT <= __builtin_fmaxf(__builtin_fmaxf(w.eps.x, w.eps.y), w.eps.z)) {
                    exact = done = true;
                    return;
                }
            }
            if (++k >= n) return;
            a = na;
            b = nb;
            c = nc;
        }
    }
    // The data of the entered object; with one instance the same for every
    // lane, so that it stays in scalar registers.
    __device__ __forceinline__ ObjectData object(const TraceParams& p) const {
        if constexpr (kSingle) return object_data(p.lods[p.instLod[0]]);
        return data;
    }
    __device__ __forceinline__ void run(const TraceParams& p, int* spill, int minActive) {
        ObjectData one;
        if (kSingle) one = object(p);
        while (!done) {
            const ObjectData& od = kSingle ? one : data;
            if (!kSingle) {
                // the instance level, once a quarter of the lanes is there
                const u64 between = __ballot(!inObj), active = __builtin_amdgcn_read_exec();
                if (4 * __popcll(between) >= __popcll(active) && !inObj) next_object(p, spill);
            }
            if (kSingle || (inObj && !done)) {
                while (true) {
                    if (!(cur & kWideLeaf)) cur = st.take(spill, wide_step(od.wide, cur, w, hitT));
                    if ((cur & kWideLeaf) && cur != kWideNone) {
                        if (held != kWideNone) break;  // a second leaf: test the held one first
                        held = cur;
                        cur = kWideNone;
                    }
                    if (cur == kWideNone) {
                        if (st.sp == base) break;
                        cur = (u32)st.pop(spill);
                    }
                    if (2 * __popcll(__ballot(held != kWideNone)) >= __popcll(__builtin_amdgcn_read_exec())) break;
                }
                if (st.overflow) {
                    exact = done = true;
                } else {
                    if (held != kWideNone) test_leaf(od);
                    if (cur == kWideNone && st.sp == base && !done) {  // the object is through
                        hitT /= scale;
                        scale = 1.0f;
                        inObj = false;
                        if (kSingle) {
                            done = true;
                        } else if (count == 0) {
                            if (st.sp == 0)
                                done = true;
                            else {
                                node = st.pop(spill);
                                count = node >= p.tlasNumInternal ? st.pop(spill) : 2;
                                offset = 0;
                            }
                        }
                    }
                }
            }
            if (__popcll(__ballot(!done)) < minActive) break;
        }
    }
    // The hit of a ray that is done (o, d, maxT: as given to init).
    __device__ __forceinline__ TraceHit result(const TraceParams& p, V3 o, V3 d, float maxT) const {
        if (__builtin_expect(exact, 0))
            return reference_ray<kAny, kMixed, kSingle ? 1 : 2>(p, o, d, maxT);
        return hit();
    }
    // The same of a ray that is not exact.
    __device__ __forceinline__ TraceHit hit() const {
        TraceHit h;
        h.t = hitT;
        h.inst = hInst;
        h.prim = hPrim;
        h.w0 = hw0;
        h.w1 = hw1;
        h.overflow = false;
        h.nodeVisits = h.primTests = 0;
        return h;
    }
};

// Traversal specializations of the kernels that trace (their kMode): fixed
// for one scene, or chosen per ray (a batch of scenes mixes single- and
// multi-instance scenes; a scene with quads or spheres takes the general
// form).
constexpr int kTraceMulti = 0;       // instance level, triangle LoDs without flat leaves
constexpr int kTraceSingle = 1;      // one instance, a triangle LoD without flat leaves
constexpr int kTraceBatch = 2;       // per ray, triangle LoDs
constexpr int kTraceMixed = 3;       // per ray, LoDs with quads and spheres
constexpr int kTraceMultiTies = 4;   // instance level, triangle LoDs (Trav's kTies)
constexpr int kTraceSingleTies = 5;  // one instance, a triangle LoD
constexpr int kTraceModes = 6;
constexpr bool mode_single(int mode) { return mode == kTraceSingle || mode == kTraceSingleTies; }
constexpr bool mode_ties(int mode) { return mode != kTraceMulti && mode != kTraceSingle; }
// binary_ray's kInstances for a mode.
constexpr int mode_instances(int mode) {
    return mode_single(mode) ? 1 : (mode == kTraceMulti || mode == kTraceMultiTies ? 0 : 2);
}
// The mode of any hits, which do not depend on the order of the leaves.
constexpr int any_mode(int mode) {
    return mode == kTraceMultiTies ? kTraceMulti : (mode == kTraceSingleTies ? kTraceSingle : mode);
}
// The mode of a kernel tracing one scene.
inline int trace_mode_of(const TraceParams& p) {
    if (p.mixed) return kTraceMixed;
    if (p.numInstances == 1) return p.flat ? kTraceSingleTies : kTraceSingle;
    return p.flat ? kTraceMultiTies : kTraceMulti;
}
// Lanes of each wave that take entries of a queue of n: all 64, or where that
// would leave more than three quarters of the `waves` resident waves without
// any, half as many until it does not (at least 8). A wave with fewer rays
// waits less for its longest, and more waves hide one another's memory latency. (Closest + any hit
// of 12,765 rays through 924 instances: 457 us with 64 lanes, 204 with 8.)
__host__ __device__ __forceinline__ int queue_lanes(int n, int waves) {
    int lanes = 64;
    while (lanes > 8 && n / lanes < waves / 4) lanes /= 2;
    return lanes;
}

// A wave's part of a queue of `n` entries, taken by its first `lanes` lanes: a
// chunk of `chunk` entries by wave index, later chunks from *counter (which
// starts at 0) once every wave has its first. Queues of fewer than four chunks
// a wave are dealt out in turn instead: every wave asks the counter once more
// than it gets, and thousands of atomics on one address take longer than such
// a queue's work may (341,000 rays through a sparse mesh of 3343 triangles: 52 us with the
// counter, 27 dealt out). For the same reason a queue may have several counters,
// each with every split-th chunk after the first ones, for every split-th wave
// (12 ns an atomic: 1M rays that miss every instance take 196 us with one
// counter, 37 with 16, 16 at one ray a lane). Entries go to the lanes in order.
struct WaveQueue {
    int n, lanes, chunk, at, end, first;
    u32 base;  // of the current chunk (the counter may run past n)
    int* counter;
    int step, skip;  // distance of a counter's chunks, entries before its first one
    bool more;       // further chunks may be left
    // counters: `split` of them (at most `waves`), kQueueStride ints apart.
    __device__ __forceinline__ WaveQueue(int n_, int lanes_, int maxChunk, int wave, int waves, int* counters,
                                         int split)
        : n(n_), lanes(lanes_) {
        const bool deal = n < 4 * 64 * waves;
        chunk = deal ? lanes : maxChunk;
        first = waves * chunk;
        const int mine = wave % split;
        step = split * chunk;
        skip = first + mine * chunk;
        counter = deal ? nullptr : counters + kQueueStride * mine;
        start((u32)(wave * chunk));
        more = counter ? skip < n : base + (u32)first < (u32)n;
    }
    __device__ __forceinline__ void start(u32 b) {
        base = b;
        at = b < (u32)n ? (int)b : n;
        end = min(chunk, n - at) + at;
    }
    __device__ __forceinline__ bool left() const { return at < end || more; }
    // The lanes that may take entries, of those with `idle` set.
    __device__ __forceinline__ u64 takers(bool idle) const { return __ballot(idle && (int)__lane_id() < lanes); }
    // Entries for the lanes of `mask`, -1 where there is none.
    __device__ __forceinline__ int take(u64 mask) {
        if (at >= end && more) {
            if (counter) {
                const int leader = __ffsll((long long)mask) - 1;
                int got = 0;
                if ((int)__lane_id() == leader) got = atomicAdd(counter, step);
                start((u32)__shfl(got, leader) + (u32)skip);
                more = base + (u32)step < (u32)n;
            } else {
                start(base + (u32)first);
                more = base + (u32)first < (u32)n;
            }
        }
        const int rank = (int)__builtin_amdgcn_mbcnt_hi((unsigned)(mask >> 32),
                                                        __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0u));
        const int e = at + rank;
        const bool mine = ((mask >> __lane_id()) & 1ull) && e < end;
        at = min(at + __popcll(mask), end);
        return mine ? e : -1;
    }
};

// Traces the rays of a wave's queue: load(entry, o, d, tmax) yields an entry's
// ray (false: nothing to trace), store(entry, hit) takes its hit. Rays end
// after very different numbers of steps, so a lane whose ray has ended takes
// the next one as soon as fewer than 5/8 of the lanes are under way; a wave
// that runs one ray per lane spends most of its steps on its few longest.
//
// A lane whose ray is the reference traversal's (Trav::exact) holds it until a
// quarter of the lanes do, or the queue ends; the wave then finishes what is
// under way and traces the held rays together, where no other traversal's
// state is alive. (Rays with a zero component, 1M of them through a 1M-triangle
// mesh: 0.61 ms, as a call each time 1.01; along a heightfield of 4.5M
// triangles 35 ms, 51.) kInstances: as binary_ray's.
template <class T, int kInstances, class Params, class Load, class Store>
__device__ __forceinline__ void trace_queue(WaveQueue& q, int* lstack, Params params, Load load, Store store) {
    T t;
    int spill[T::kSpill];
    t.done = true;
    t.exact = false;
    int entry = -1;
    while (true) {
        const bool open = 4 * __popcll(__ballot(entry >= 0 && t.exact)) < q.lanes;  // takes further rays
        const u64 idle = q.takers(entry < 0);
        if (idle != 0ull && open && q.left()) {
            const int e = q.take(idle);
            V3 o, d;
            float tmax;
            if (e >= 0 && load(e, o, d, tmax)) {
                entry = e;
                t.init(params(e), o, d, tmax, lstack);
            }
        }
        if (__ballot(entry >= 0 && !t.exact) == 0ull) {
            if (__ballot(entry >= 0) == 0ull) {
                if (!q.left()) break;
                continue;
            }
            if (open && q.left()) continue;
            if (entry >= 0) {
                V3 o, d;
                float tmax;
                load(entry, o, d, tmax);
                const typename T::Binary stack{lstack, 0, false};
                store(entry, binary_ray<T::kAnyHit, false, kInstances, T::kMixedLods>(params(entry), o, d, tmax, stack));
                entry = -1;
            }
            continue;
        }
        if (entry >= 0 && !t.exact) {
            t.run(params(entry), spill, open && q.left() ? q.lanes * 5 / 8 : 0);
            if (t.done && !t.exact) {
                store(entry, t.hit());
                entry = -1;
            }
        }
    }
}

// The traversal of a kernel in mode kMode.
template <int kMode, bool kAny, int kStride, int kLds>
using ModeTrav = Trav<kAny, mode_single(kMode), kMode == kTraceMixed, !kAny && mode_ties(kMode), kStride, kLds>;

// Closest (kAny = false) or any hit in mode kMode.
template <int kMode, bool kAny, int kStride, int kLds>
__device__ __forceinline__ TraceHit trace_mode(const TraceParams& tp, V3 o, V3 d, float tmax, int* lstack) {
    using T = ModeTrav<kMode, kAny, kStride, kLds>;
    T t;
    int spill[T::kSpill];
    t.init(tp, o, d, tmax, lstack);
    t.run(tp, spill, 0);
    return t.result(tp, o, d, tmax);
}

}  // namespace mfh
