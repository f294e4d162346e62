// Closest-hit and any-hit traversal of the BVH4, plus the reference's
// primitive tests.
//
// Result semantics (what must match the reference bit for bit):
//   The reference walks its object BVH depth-first and keeps the first
//   strictly closer hit (lib/src/DataStructure/BoundingVolumeHierarchyDetail.h:11-101),
//   testing each object's own box with a biased slab test first
//   (lib/src/Geometry/AABBDetail.h:18-50). Inner boxes of that tree contain their
//   children's boxes, so the result is: among primitives whose object box passes
//   that biased test, the minimum of (t, reference rank), where rank is the
//   primitive's position in the reference DFS order (mesh triangles in index
//   order inside their mesh). This traversal computes exactly that minimum over
//   its own SAH BVH4: boxes are culled conservatively (slack on both ends of
//   the interval), and the biased object-box test runs lazily, only for a
//   candidate that would become the new best.
//
// Stack: a short per-lane stack in LDS (lane-minor, so a wave's pushes hit 64
// distinct banks), continued in a global spill area for deep trees.
#pragma once

#include <hip/hip_fp16.h>

#include "scene_types.h"

namespace cupbr {

// Triangle::computeRayIntersection, lib/src/Geometry/TriangleDetail.h:21-57.
// Returns true for a hit with t >= 0; NaN results report true with NaN t and are
// discarded by the callers' ordered comparisons, as in the reference.
__device__ __forceinline__ bool mt_test(v3 v1, v3 e1, v3 e2, v3 o, v3 d, float& t) {
    v3 pvec = cross(d, e2);
    float det = dot(e1, pvec);
    if (safe_float_equal(det, 0.0f)) return false;
    float inv_det = 1.0f / det;
    v3 tvec = o - v1;
    float u = dot(tvec, pvec) * inv_det;
    if (u < 0.0f || u > 1.0f) return false;
    v3 qvec = cross(tvec, e1);
    float v = dot(d, qvec) * inv_det;
    if (v < 0.0f || u + v > 1.0f) return false;
    t = dot(e2, qvec) * inv_det;
    return !(t < 0.0f);
}

// Sphere::computeRayIntersection, lib/src/Geometry/SphereDetail.h:33-74
__device__ __forceinline__ bool sphere_test(v3 c, float r, v3 o, v3 d, float& t) {
    v3 os = o - c;
    float b = 2.0f * dot(d, os);
    float cc = dot(os, os) - r * r;
    float disc = b * b - 4.0f * cc;
    if (disc > 0) {
        float s = sqrtf(disc);
        float q = b < 0 ? (-b - s) / 2.0f : (-b + s) / 2.0f;
        float t0 = q, t1 = cc / q;
        float mn = fminf(t0, t1), mx = fmaxf(t0, t1);
        float tt = mn < 0 ? mx : mn;
        if (tt >= 0) { t = tt; return true; }
    }
    return false;
}

// Plane::computeRayIntersection (PlaneDetail.h:19-46) and Quad (QuadDetail.h:21-57)
__device__ __forceinline__ bool plane_quad_test(const UnbRec& u, v3 o, v3 d, float& t) {
    v3 p = mk(u.p.x, u.p.y, u.p.z), n = mk(u.n.x, u.n.y, u.n.z);
    float pdotn = dot(p, n), odotn = dot(o, n), ddotn = dot(d, n);
    if (safe_float_equal(ddotn, 0.0f)) return false;
    float tt = (pdotn - odotn) / ddotn;
    if (tt < 0) return false;
    if (__float_as_int(u.p.w) == kUnbQuad) {
        v3 e1 = mk(u.e1.x, u.e1.y, u.e1.z), e2 = mk(u.e2.x, u.e2.y, u.e2.z);
        v3 ip = o + tt * d;
        float x = dot(ip - p, e1), y = dot(ip - p, e2);
        float s1 = dot(e1, e1), s2 = dot(e2, e2);
        if (x < -s1 || x > s1 || y < -s2 || y > s2) return false;
    }
    t = tt;
    return true;
}

// AABB::hit, lib/src/Geometry/AABBDetail.h:18-50: 1/(d+1e-5) with no sign correction
__device__ __forceinline__ bool ref_aabb_hit(const float* mn, const float* mx, v3 o, v3 d) {
    bool hit = true;
    float tmin = 0.0f, tmax = __builtin_inff();
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        float inv = 1.0f / (comp(d, a) + kEpsilon);
        float t0 = (mn[a] - comp(o, a)) * inv;
        float t1 = (mx[a] - comp(o, a)) * inv;
        if (inv < 0.0f) { float tmp = t0; t0 = t1; t1 = tmp; }
        tmin = t0 > tmin ? t0 : tmin;
        tmax = t1 < tmax ? t1 : tmax;
        if (tmax <= tmin) hit = false;
    }
    return hit;
}

struct TraceResult {
    float t;
    uint32_t prim;  // leaf-order prim index, kUnbBit|unbounded index, or kNoHit
    uint32_t rank;
};

// triangle or sphere test of one primitive record
__device__ __forceinline__ bool prim_test(const PrimRec& pr, v3 o, v3 d, float& t) {
    if ((__float_as_uint(pr.c.w) & 3u) == kPrimTriangle)
        return mt_test(mk(pr.a.x, pr.a.y, pr.a.z), mk(pr.a.w, pr.b.x, pr.b.y), mk(pr.b.z, pr.b.w, pr.c.x), o, d, t);
    return sphere_test(mk(pr.a.x, pr.a.y, pr.a.z), pr.a.w, o, d, t);
}

// the reference's biased test of the primitive's object box (finite boxes only: spheres, meshes)
__device__ __forceinline__ bool object_box_ok(const DevScene& S, const PrimRec& pr, v3 o, v3 d) {
    if (!(__float_as_uint(pr.c.w) & kPrimNeedsBoxCheck)) return true;
    const ObjInfo& ob = S.objs[__float_as_uint(pr.c.z)];
    return ref_aabb_hit(ob.bmin, ob.bmax, o, d);
}

// closest-hit step of one primitive (leaf-order index idx): best <- (t, idx, rank) when the
// primitive is hit at (t, rank) lexicographically below best and passes its object-box test
// (tested last, only for a candidate that would win)
__device__ __forceinline__ void closest_prim(const DevScene& S, const PrimRec& pr, uint32_t idx, v3 o, v3 d,
                                             TraceResult& best) {
    float t;
    if (!prim_test(pr, o, d, t)) return;
    const uint32_t rank = __float_as_uint(pr.c.y);
    if (t < best.t || (t == best.t && rank < best.rank)) {
        if (!object_box_ok(S, pr, o, d)) return;
        best.t = t;
        best.prim = idx;
        best.rank = rank;
    }
}

// Per-lane stack: entries [0, kLds) in LDS at lds[i * lds_stride], the rest in global
// memory at spill[(i - kLds) * spill_stride].
template <int kLds>
struct LaneStack {
    uint32_t* lds;
    uint32_t lds_stride;
    uint32_t* spill;
    uint32_t spill_stride;
    __device__ __forceinline__ void put(int i, uint32_t v) {
        if (i < kLds) lds[i * lds_stride] = v;
        else spill[(size_t)(i - kLds) * spill_stride] = v;
    }
    // The LDS read is unconditional (its address clamped into the LDS part) and the spill read a
    // relaxed atomic load, so that the compiler cannot merge the two into one generic (flat) load
    // of a selected pointer: a pop stays a ds_read.
    __device__ __forceinline__ uint32_t get(int i) const {
        uint32_t v = lds[min(i, kLds - 1) * lds_stride];
        if (i >= kLds)
            v = __hip_atomic_load(spill + (size_t)(i - kLds) * spill_stride, __ATOMIC_RELAXED,
                                  __HIP_MEMORY_SCOPE_WAVEFRONT);
        return v;
    }
};

// visit counters of one lane (only updated by the counting instantiation)
struct TravCount {
    uint32_t nodes = 0, prims = 0;
};

// The primitives of one leaf (leaf word `word`): closest-hit updates of best, or (kAny) true as
// soon as one is hit within [0, dist].
template <bool kAny>
__device__ __forceinline__ bool visit_leaf(const DevScene& S, uint32_t word, v3 o, v3 d, float dist, TraceResult& best) {
    const uint32_t first = leaf_first(word), n_leaf = leaf_count(word);
    for (uint32_t k = 0; k < n_leaf; ++k) {
        const PrimRec pr = S.prims[first + k];
        if (kAny) {
            float t;
            if (!prim_test(pr, o, d, t) || !(t <= dist) || !object_box_ok(S, pr, o, d)) continue;
            return true;
        }
        closest_prim(S, pr, first + k, o, d, best);
    }
    return false;
}

// One inner node `cur`: the children whose boxes overlap [tlo, lim] (conservatively) are pushed
// farthest first, and cur becomes the nearest (closest hit) or a hit one (any hit); false when
// no child overlaps. The node is read in its NodeH form: a lane loads its reference point, the 16-byte block
// of each axis for the sign of its inverse direction (near planes of the 4 children, then far
// planes, as binary16 offsets) and the child words, and takes each plane's distance as one
// mixed-precision FMA, t = h (i 2^k) + (c - o) i. The decoded planes lie outside the FP32 ones by
// a margin that covers the decode's rounding (half_nodes), so the test stays conservative. An
// empty child slot has the box lo = +inf, hi = -inf, which no ray overlaps.
// Children are ordered by integer keys, the entry distance's float bits read as a signed integer
// (non-negative distances in their order, the slightly negative ones of boxes around the origin
// ahead of them), INT_MAX for a culled child; each compare-exchange of the network is a min, a max
// and two selects of the child words, with no branch. The order only decides which overlapping
// child is visited first; the closest hit is the same for any order.
template <bool kAny, int kLds>
__device__ __forceinline__ bool visit_inner(const DevScene& S, uint32_t& cur, v3 o, float ix, float iy, float iz,
                                            float lim, LaneStack<kLds>& st, int& sp) {
    const float tlo = -1e-5f;
    constexpr int kCulled = 0x7FFFFFFF;
    const char* base = reinterpret_cast<const char*>(S.hnodes);
    const uint32_t nb = cur * 128u;  // 32-bit byte offsets: scene_finalize keeps the nodes below 2^25
    const float4 co = *reinterpret_cast<const float4*>(base + nb);
    const uint4 px = *reinterpret_cast<const uint4*>(base + (nb + (ix >= 0.0f ? 16u : 32u)));
    const uint4 py = *reinterpret_cast<const uint4*>(base + (nb + (iy >= 0.0f ? 48u : 64u)));
    const uint4 pz = *reinterpret_cast<const uint4*>(base + (nb + (iz >= 0.0f ? 80u : 96u)));
    const uint4 ch = *reinterpret_cast<const uint4*>(base + (nb + 112u));
    int key[4];
    uint32_t val[4] = {ch.x, ch.y, ch.z, ch.w};
    // per axis: A = i 2^k (exact: k <= 0, and |i| >= 1 for a unit direction), B = (c - o) i
    const uint32_t ex = __float_as_uint(co.w);
    const float ax = __builtin_ldexpf(ix, (int)(int8_t)(ex & 0xFFu));
    const float ay = __builtin_ldexpf(iy, (int)(int8_t)((ex >> 8) & 0xFFu));
    const float az = __builtin_ldexpf(iz, (int)(int8_t)((ex >> 16) & 0xFFu));
    const float bx = (co.x - o.x) * ix, by = (co.y - o.y) * iy, bz = (co.z - o.z) * iz;
    auto lo16 = [](uint32_t w) { return __low2float(*reinterpret_cast<const __half2*>(&w)); };
    auto hi16 = [](uint32_t w) { return __high2float(*reinterpret_cast<const __half2*>(&w)); };
    // child i's near plane: half i of words 0..1 of its axis block; far plane: half i of words 2..3
#define CUPBR_CHILD(i, half, wn, wf)                                                               \
    {                                                                                              \
        const float tn = fmaxf(fmaxf(fmaf(half(px.wn), ax, bx), fmaf(half(py.wn), ay, by)),        \
                               fmaxf(fmaf(half(pz.wn), az, bz), tlo));                              \
        const float tf = fminf(fminf(fmaf(half(px.wf), ax, bx), fmaf(half(py.wf), ay, by)),        \
                               fminf(fmaf(half(pz.wf), az, bz), lim));                              \
        key[i] = tn <= tf * 1.000002f ? __float_as_int(tn) : kCulled;                              \
    }
    CUPBR_CHILD(0, lo16, x, z)
    CUPBR_CHILD(1, hi16, x, z)
    CUPBR_CHILD(2, lo16, y, w)
    CUPBR_CHILD(3, hi16, y, w)
#undef CUPBR_CHILD
    // The child words are only needed once a child overlaps; without this use the compiler moves
    // their load behind that test, and the step then waits for a second memory round trip.
    asm volatile("" ::"v"(val[0]), "v"(val[1]), "v"(val[2]), "v"(val[3]));
#define CUPBR_KSWAP(a, b)                                   \
    {                                                       \
        const bool sw = key[b] < key[a];                    \
        const int klo = min(key[a], key[b]);                \
        key[b] = max(key[a], key[b]);                       \
        key[a] = klo;                                       \
        const uint32_t va = val[a];                         \
        val[a] = sw ? val[b] : va;                          \
        val[b] = sw ? va : val[b];                          \
    }
    if (!kAny) {  // nearest child first; an any-hit query only needs the ones that were hit
        CUPBR_KSWAP(0, 1)
        CUPBR_KSWAP(2, 3)
        CUPBR_KSWAP(0, 2)
        CUPBR_KSWAP(1, 3)
        CUPBR_KSWAP(1, 2)
    } else {
        CUPBR_KSWAP(0, 1)  // the nearest hit child, if any, into slot 0
        CUPBR_KSWAP(0, 2)
        CUPBR_KSWAP(0, 3)
    }
#undef CUPBR_KSWAP
    if (key[0] == kCulled) return false;
    if (key[3] != kCulled) st.put(sp++, val[3]);
    if (key[2] != kCulled) st.put(sp++, val[2]);
    if (key[1] != kCulled) st.put(sp++, val[1]);
    cur = val[0];
    return true;
}

// kAny=false: closest hit (best.t = +inf, best.prim = kNoHit on a miss).
// kAny=true : any valid hit with t <= dist; returns whether one exists.
template <bool kAny, int kLds, bool kCount = false>
__device__ __forceinline__ bool traverse(const DevScene& S, v3 o, v3 d, float dist, LaneStack<kLds>& st,
                                         TraceResult& best, TravCount* cnt = nullptr) {
    best.t = __builtin_inff();
    best.prim = kNoHit;
    best.rank = 0xFFFFFFFFu;

    // planes and quads first: their hits tighten the interval for the BVH
    for (uint32_t i = 0; i < S.n_unb; ++i) {
        const UnbRec u = S.unb[i];
        float t;
        if (!plane_quad_test(u, o, d, t)) continue;
        if (kAny) {
            if (t <= dist) return true;
            continue;
        }
        uint32_t rank = __float_as_uint(u.n.w);
        if (t < best.t || (t == best.t && rank < best.rank)) {
            best.t = t;
            best.prim = kUnbBit | i;
            best.rank = rank;
        }
    }
    if (S.n_nodes == 0) return false;

    const float ix = 1.0f / d.x, iy = 1.0f / d.y, iz = 1.0f / d.z;
    int sp = 0;
    uint32_t cur = 0;
    for (;;) {
        if (cur & kLeafBit) {
            if (kCount) cnt->prims += leaf_count(cur);
            if (visit_leaf<kAny>(S, cur, o, d, dist, best)) return true;
        } else {
            if (kCount) cnt->nodes += 1;
            const float lim = kAny ? dist * 1.0001f + 1e-6f : best.t * 1.0001f + 1e-6f;
            if (visit_inner<kAny>(S, cur, o, ix, iy, iz, lim, st, sp)) continue;
        }
        if (sp == 0) break;
        cur = st.get(--sp);
    }
    return false;
}

// The same traversal as a resumable state, one node or leaf per step, for kernels that hand a
// new ray to a lane as soon as its previous one ends. best.t holds the query distance of an
// any-hit ray.
struct RayState {
    v3 o, d;
    float ix, iy, iz;
    TraceResult best;
    uint32_t cur;
    int sp;
};

// Starts a ray: planes and quads first (as in traverse). Returns whether BVH steps follow; when
// not, the result is final (closest hit in best; any hit in `hit`).
template <bool kAny>
__device__ __forceinline__ bool ray_begin(const DevScene& S, RayState& r, v3 o, v3 d, float dist, bool& hit) {
    r.o = o;
    r.d = d;
    r.best.t = kAny ? dist : __builtin_inff();
    r.best.prim = kNoHit;
    r.best.rank = 0xFFFFFFFFu;
    hit = false;
    for (uint32_t i = 0; i < S.n_unb; ++i) {
        const UnbRec u = S.unb[i];
        float t;
        if (!plane_quad_test(u, o, d, t)) continue;
        if (kAny) {
            if (t <= dist) {
                hit = true;
                return false;
            }
            continue;
        }
        const uint32_t rank = __float_as_uint(u.n.w);
        if (t < r.best.t || (t == r.best.t && rank < r.best.rank)) {
            r.best.t = t;
            r.best.prim = kUnbBit | i;
            r.best.rank = rank;
        }
    }
    r.ix = 1.0f / d.x;
    r.iy = 1.0f / d.y;
    r.iz = 1.0f / d.z;
    r.cur = 0;
    r.sp = 0;
    return S.n_nodes != 0;
}

// One inner node or one primitive of a started ray; false when its traversal has ended. A leaf
// takes one step per primitive, so that lanes at leaves of different sizes do not hold the wave
// for the largest one.
template <bool kAny, int kLds>
__device__ __forceinline__ bool ray_step(const DevScene& S, RayState& r, LaneStack<kLds>& st, bool& hit) {
    if (r.cur & kLeafBit) {
        // one primitive per step: the leaf word keeps the rest of the leaf (first + 1, count - 1)
        const uint32_t first = leaf_first(r.cur);
        const PrimRec pr = S.prims[first];
        if (kAny) {
            float t;
            if (prim_test(pr, r.o, r.d, t) && t <= r.best.t && object_box_ok(S, pr, r.o, r.d)) {
                hit = true;
                return false;
            }
        } else {
            closest_prim(S, pr, first, r.o, r.d, r.best);
        }
        if (leaf_count(r.cur) > 1u) {
            r.cur += 15u;  // first + 1 (bits 4..30), count - 1 (bits 0..3)
            return true;
        }
    } else {
        const float lim = r.best.t * 1.0001f + 1e-6f;  // the query distance of an any-hit ray
        if (visit_inner<kAny>(S, r.cur, r.o, r.ix, r.iy, r.iz, lim, st, r.sp)) return true;
    }
    if (r.sp == 0) return false;
    r.cur = st.get(--r.sp);
    return true;
}

// the minimum of (t, rank) over a group of kGroup lanes, in every lane of it
template <uint32_t kGroup>
__device__ __forceinline__ TraceResult group_min(TraceResult r) {
#pragma unroll
    for (uint32_t off = 1; off < kGroup; off <<= 1) {
        const float t = __shfl_xor(r.t, off);
        const uint32_t prim = __shfl_xor(r.prim, off), rank = __shfl_xor(r.rank, off);
        if (t < r.t || (t == r.t && rank < r.rank)) r = TraceResult{t, prim, rank};
    }
    return r;
}

// One ray per group of kGroup lanes of a wave: each step takes the kGroup / 4 entries on top of the ray's
// stack, four lanes to an entry, a lane testing one child of an inner node or every fourth primitive of a
// leaf. What bounds a batch too small to fill the chip is the longest ray's chain of dependent steps, each
// a round trip to memory; this shortens the chain by up to kGroup / 4 at the price of visits that the
// sequential order would have culled. The tests are those of traverse, and the result, a minimum of
// (t, rank) over all primitives of overlapping boxes (any-hit: whether there is one), is the same for any
// order of visits.
// stack(k): entry k of kCapacity words of LDS of the group's own. reserve, three words per level of the
// tree, is what walking one entry at a time can add; a step takes one entry only while its pushes could
// leave less than that, so reserve < kCapacity is all the stack needs.
// In: best, a closest hit found already (none: t = inf, rank = 0xFFFFFFFF). Called by whole waves; a group
// with valid = false only takes part in the wave's votes. Returns (any-hit) whether there is a hit.
template <bool kAny, uint32_t kGroup, uint32_t kCapacity, class Stack>
__device__ __forceinline__ bool traverse_group(const DevScene& S, v3 o, v3 d, float dist, bool valid, uint32_t reserve,
                                               Stack stack, TraceResult& best) {
    constexpr uint32_t kEntries = kGroup / 4;
    constexpr int kCulled = 0x7FFFFFFF;
    const uint32_t lane = __lane_id(), sub = lane % kGroup, entry = sub >> 2, c = sub & 3u;
    const auto group_bits = [&](bool b) {  // the group's votes, lane sub in bit sub
        return (__ballot(b) >> (lane - sub)) & (~0ull >> (64u - kGroup));
    };
    bool any = false;
    const float ix = 1.0f / d.x, iy = 1.0f / d.y, iz = 1.0f / d.z;
    const float tlo = -1e-5f;
    uint32_t sp = valid && S.n_nodes ? 1u : 0u;
    if (sub == 0u) stack(0u) = 0u;
    while (__ballot(sp != 0u)) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();  // the entries pushed by other lanes
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const uint32_t take = min(sp, sp + 3u * kEntries + reserve <= kCapacity ? kEntries : 1u);
        const bool mine = entry < take;
        const uint32_t word = mine ? stack(sp - 1u - entry) : kLeafBit;
        sp -= take;
        int key = kCulled;
        uint32_t child = 0u;
        TraceResult found = best;
        bool hit = false;
        if (!(word & kLeafBit)) {
            const float lim = (kAny ? dist : best.t) * 1.0001f + 1e-6f;
            const char* base = reinterpret_cast<const char*>(S.hnodes) + (size_t)word * 128u;
            const float4 co = *reinterpret_cast<const float4*>(base);
            const uint4 px = *reinterpret_cast<const uint4*>(base + (ix >= 0.0f ? 16u : 32u));
            const uint4 py = *reinterpret_cast<const uint4*>(base + (iy >= 0.0f ? 48u : 64u));
            const uint4 pz = *reinterpret_cast<const uint4*>(base + (iz >= 0.0f ? 80u : 96u));
            child = *reinterpret_cast<const uint32_t*>(base + 112u + 4u * c);
            const uint32_t ex = __float_as_uint(co.w);
            const float ax = __builtin_ldexpf(ix, (int)(int8_t)(ex & 0xFFu));
            const float ay = __builtin_ldexpf(iy, (int)(int8_t)((ex >> 8) & 0xFFu));
            const float az = __builtin_ldexpf(iz, (int)(int8_t)((ex >> 16) & 0xFFu));
            const float bx = (co.x - o.x) * ix, by = (co.y - o.y) * iy, bz = (co.z - o.z) * iz;
            const auto half = [&](uint32_t w01, uint32_t w23) {  // half c of the four
                const uint32_t w = (c & 2u ? w23 : w01) >> (c & 1u ? 16 : 0);
                return __low2float(*reinterpret_cast<const __half2*>(&w));
            };
            const float tn = fmaxf(fmaxf(fmaf(half(px.x, px.y), ax, bx), fmaf(half(py.x, py.y), ay, by)),
                                   fmaxf(fmaf(half(pz.x, pz.y), az, bz), tlo));
            const float tf = fminf(fminf(fmaf(half(px.z, px.w), ax, bx), fmaf(half(py.z, py.w), ay, by)),
                                   fminf(fmaf(half(pz.z, pz.w), az, bz), lim));
            if (tn <= tf * 1.000002f) key = __float_as_int(tn);
        } else if (mine) {
            const uint32_t first = leaf_first(word), n_leaf = leaf_count(word);
            for (uint32_t k = c; k < n_leaf; k += 4u) {
                const PrimRec pr = S.prims[first + k];
                if (kAny) {
                    float t;
                    hit = hit || (prim_test(pr, o, d, t) && t <= dist && object_box_ok(S, pr, o, d));
                } else {
                    closest_prim(S, pr, first + k, o, d, found);
                }
            }
            if (!kAny) hit = found.prim != best.prim;
        }
        // the hit children go on top, the first entry's topmost and each entry's nearest first
        uint32_t nearer = 0;
#pragma unroll
        for (uint32_t x = 1; x < 4; ++x) {
            constexpr int kPerm[4] = {0, 0xB1, 0x4E, 0x1B};  // quad lanes c ^ 1, c ^ 2, c ^ 3
            const int k = x == 1 ? __builtin_amdgcn_mov_dpp(key, kPerm[1], 0xF, 0xF, true)
                        : x == 2 ? __builtin_amdgcn_mov_dpp(key, kPerm[2], 0xF, 0xF, true)
                                 : __builtin_amdgcn_mov_dpp(key, kPerm[3], 0xF, 0xF, true);
            nearer += k < key || (k == key && (c ^ x) < c) ? 1u : 0u;
        }
        const unsigned long long pushed = group_bits(key != kCulled);
        const uint32_t siblings = (uint32_t)__popcll((pushed >> (4u * entry)) & 15u);
        const uint32_t below = (uint32_t)__popcll(pushed >> (4u * entry) >> 4);
        if (key != kCulled) stack(sp + below + siblings - 1u - nearer) = child;
        sp += (uint32_t)__popcll(pushed);
        if (kAny) {
            any = any || group_bits(hit) != 0ull;
            if (any) sp = 0u;
        } else if (__ballot(hit)) {
            best = group_min<kGroup>(found);
        }
    }
    return any;
}

// traverse with a group of kGroup lanes per ray
template <bool kAny, uint32_t kGroup, uint32_t kCapacity, class Stack>
__device__ __forceinline__ bool trace_group(const DevScene& S, v3 o, v3 d, float dist, bool valid, uint32_t reserve,
                                            Stack stack, TraceResult& best) {
    best = TraceResult{__builtin_inff(), kNoHit, 0xFFFFFFFFu};
    bool any = false;
    if (valid)  // planes and quads first, as in traverse
        for (uint32_t i = __lane_id() % kGroup; i < S.n_unb; i += kGroup) {
            const UnbRec u = S.unb[i];
            float t;
            if (!plane_quad_test(u, o, d, t)) continue;
            const uint32_t rank = __float_as_uint(u.n.w);
            any = any || t <= dist;
            if (t < best.t || (t == best.t && rank < best.rank)) best = TraceResult{t, kUnbBit | i, rank};
        }
    if (kAny) {
        const uint32_t first = __lane_id() / kGroup * kGroup;
        any = ((__ballot(any) >> first) & (~0ull >> (64u - kGroup))) != 0ull;
    } else if (S.n_unb) {
        best = group_min<kGroup>(best);
    }
    return traverse_group<kAny, kGroup, kCapacity>(S, o, d, dist, valid && !(kAny && any), reserve, stack, best) || (kAny && any);
}

// traverse for the active lanes of a wave (all of which call it), each with its own ray: one lane per ray, or 8 lanes
// each for the last rays (up to 16) of a wave whose other paths have ended.
template <bool kAny, int kLds>
__device__ __forceinline__ bool trace_lanes(const DevScene& S, bool active, v3 o, v3 d, float dist, LaneStack<kLds>& st,
                                            TraceResult& r) {
    constexpr uint32_t kGroup = 8, kRays = 64 / kGroup, kWords = kLds * kGroup;
    const unsigned long long m = __ballot(active);
    const uint32_t n = (uint32_t)__popcll(m), lane = __lane_id();
    bool any = false;
    if (n > 16u || S.stack_reserve >= kWords) {
        if (active) any = traverse<kAny>(S, o, d, dist, st, r);
        return any;
    }
    // lane k gets the number of the k-th active lane
    const uint32_t rank = (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
    const int ids = __builtin_amdgcn_ds_permute((int)(active ? rank : n + lane - rank) * 4, (int)lane);
    for (uint32_t first = 0; first < n; first += kRays) {
        const uint32_t k = first + lane / kGroup;
        const int src = __shfl(ids, (int)min(k, 63u));
        const auto from = [&](float x) { return __shfl(x, src); };
        const v3 go = mk(from(o.x), from(o.y), from(o.z)), gd = mk(from(d.x), from(d.y), from(d.z));
        const float gdist = from(dist);
        uint32_t* words = st.lds - lane;  // the wave's stack words: row by row, 64 each
        const uint32_t row = st.lds_stride, base = lane / kGroup * kWords;
        TraceResult best;
        const bool hit = trace_group<kAny, kGroup, kWords>(
            S, go, gd, gdist, k < n, S.stack_reserve,
            [&](uint32_t e) -> uint32_t& { return words[((base + e) >> 6) * row + ((base + e) & 63u)]; }, best);
        const int back = (int)((rank % kRays) * kGroup);
        const bool mine = active && rank / kRays * kRays == first;
        if (kAny) {
            const bool h = __shfl((int)hit, back) != 0;
            any = mine ? h : any;
        } else {
            const TraceResult b{__shfl(best.t, back), (uint32_t)__shfl((int)best.prim, back), (uint32_t)__shfl((int)best.rank, back)};
            if (mine) r = b;
        }
    }
    return any;
}

// Lanes of the refill loop that must be at a leaf before a wave runs a leaf step (inner-node steps
// otherwise), at most: a wave runs its leaf step once half of its rays wait at a leaf, capped at
// this many lanes. 32 (always half) measured best with the half rule (1080p, 1M triangles: cap 12
// / 16 / 20 / 24 / 28 / 32 -> 1143 / 1155-1159 / 1163 / 1164-1168 / 1168 / 1168 Msamples/s). With
// a fixed count instead (an earlier build): 8 / 16 / 24 / 32 -> 901 / 932 / 920 / 843; leaf and
// inner steps taken together every iteration: 889.
constexpr uint32_t kLeafBatch = 32;
// lanes per ray for a wave's last rays
constexpr uint32_t kTailGroup = 16;

// The rays of a wave's share, with per-lane refill: the wave gives fresh rays to its idle lanes whenever at
// least kIdle of them are idle (or all are), so that a lane whose ray ended does not wait for the slowest
// ray of a 64-ray chunk. The share has a current piece [at, end); refill() makes a new one (false when
// there is none), index(k) names its ray k. load(i, o, d, dist) reads ray i, finish(i, hit, r) consumes
// its result. Two ways of stepping:
//   kPhased   leaf steps and inner-node steps of the wave apart (below): most rays per second where a
//             wave refills many times
//   otherwise every lane its own step, and the last rays of the share by kTailGroup lanes each
//             (traverse_group), which start them over with the hit found so far: shortest where a wave
//             has only a few rays per lane and its longest ray bounds it. The path tracer's trace kernel
//             does not take it: the second walk costs it 14 spilled registers (109.6 -> 114.4 ms a frame
//             of 1080p, 1M triangles, 64 spp) and saves 1% of a 1-spp frame.
template <bool kAny, bool kPhased, class Share, int kLds, class Load, class Finish>
__device__ __forceinline__ void trace_pool(const DevScene& S, Share& share, LaneStack<kLds>& st, Load load,
                                           Finish finish) {
    constexpr uint32_t kTailWords = kLds * kTailGroup;
    constexpr int kIdle = kPhased ? 32 : 16;
    const uint32_t lane = __lane_id();
    bool active = false, pool = true, hit = false;
    decltype(share.index(0u)) my = 0;
    RayState rs;
    for (;;) {
        const unsigned long long idle = __ballot(!active);
        if (pool && (__popcll(idle) >= kIdle || idle == ~0ull)) {
            if (share.at >= share.end) pool = share.refill();
            if (!active) {
                const uint32_t idx = share.at + (uint32_t)__popcll(idle & ((1ull << lane) - 1ull));
                if (idx < share.end) {
                    my = share.index(idx);
                    v3 o, d;
                    float dist;
                    load(my, o, d, dist);
                    active = ray_begin<kAny>(S, rs, o, d, dist, hit);
                    if (!active) finish(my, hit, rs.best);
                }
            }
            share.at = min(share.at + (uint32_t)__popcll(idle), share.end);
        }
        const unsigned long long am = __ballot(active);
        if (am == 0ull) {
            if (!pool) break;
            continue;
        }
        if (!kPhased && !pool && (uint32_t)__popcll(am) <= 64u / kTailGroup && S.stack_reserve < kTailWords) {
            unsigned long long m = am;
            for (uint32_t k = lane / kTailGroup; k != 0u; --k) m &= m - 1ull;  // 0 from the last ray on
            const bool valid = m != 0ull;
            const int src = valid ? __builtin_ctzll(m) : 0;
            const auto from = [&](float x) { return __shfl(x, src); };
            const v3 o = mk(from(rs.o.x), from(rs.o.y), from(rs.o.z)), d = mk(from(rs.d.x), from(rs.d.y), from(rs.d.z));
            TraceResult best{from(rs.best.t), (uint32_t)__shfl((int)rs.best.prim, src), (uint32_t)__shfl((int)rs.best.rank, src)};
            my = __shfl(my, src);
            const uint32_t first = lane / kTailGroup * kTailWords;  // the wave's stacks end here: row by row, 64 words each
            uint32_t* words = st.lds - lane;
            const uint32_t row = st.lds_stride;
            const bool any = traverse_group<kAny, kTailGroup, kTailWords>(
                S, o, d, best.t, valid, S.stack_reserve,
                [&](uint32_t k) -> uint32_t& { return words[((first + k) >> 6) * row + ((first + k) & 63u)]; }, best);
            if (valid && lane % kTailGroup == 0u) finish(my, any, best);
            break;
        }
        // Wave-uniform phases: a primitive step for the lanes at a leaf once half of the wave's rays
        // are there (at most kLeafBatch lanes), or all of them (no lane has an inner node
        // left); an inner-node step for the others otherwise. A lane whose ray reached a leaf waits
        // during inner phases, so that the primitive test runs for many lanes at once instead of a
        // few in every iteration (before: leaf code in 97% of iterations for 9 of 64 lanes). Counted
        // against the wave's own rays, the rule also keeps a nearly empty wave (the last rays of a
        // launch) from holding its leaf lanes back until every other ray reaches a leaf (1080p, 1M
        // triangles: a fixed 16 lanes 1147, half capped at 16 1155-1159, half 1168 Msamples/s).
        const bool at_leaf = active && (rs.cur & kLeafBit);
        const uint32_t n_leaf = (uint32_t)__popcll(__ballot(at_leaf));
        const uint32_t n_act = (uint32_t)__popcll(am);
        const bool leaf_phase = n_leaf >= min(kLeafBatch, (n_act + 1u) / 2u) || n_leaf == n_act;
        const bool go = !kPhased ? active : leaf_phase ? at_leaf : active && !at_leaf;
        if (go && !ray_step<kAny>(S, rs, st, hit)) {
            finish(my, hit, rs.best);
            active = false;
        }
    }
}

// a load whose address is the same in every lane, issued as a scalar load (records of the
// BVH and primitive arrays, which no kernel writes while it traverses them)
__device__ __forceinline__ float4 uniform_load4(const void* p) {
    typedef float f4 __attribute__((ext_vector_type(4)));
    const f4 v = *(const __attribute__((address_space(4))) f4*)p;
    return make_float4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ PrimRec uniform_prim(const PrimRec* p) {
    return PrimRec{uniform_load4(&p->a), uniform_load4(&p->b), uniform_load4(&p->c)};
}

// Entries of the wave-uniform stack of traverse_packet: entry k is held by lane k % 64 of
// register k / 64.
constexpr uint32_t kPacketStack = 128;

// Closest hit for the 64 rays of a wave traversed as one packet (rays with a common origin and
// nearby directions, such as the camera rays of an 8x8 pixel tile). Every node and leaf is
// visited by the whole wave: its record is a wave-uniform scalar load, each lane tests its own
// ray, and a child is entered when its box overlaps the current interval of any lane (the same
// conservative test as traverse), nearest first by the entry distance of the first such lane.
// Every lane therefore tests a superset of the primitives its own traversal would test, none
// outside the object boxes' candidates, and the closest hit, a minimum of (t, reference rank)
// over them, is the same. Lanes with valid = false take part in the traversal (the stack is
// one value per wave, spread over the lanes) but have an empty interval and keep no hit.
// Requires the BVH's worst-case stack (3 entries per BVH4 level + 1) <= kPacketStack and the
// whole wave active. kUniformSigns: every valid lane's direction has the signs (ux, uy, uz), so
// the near and far planes of a box are chosen once per wave.
template <bool kUniformSigns>
__device__ __forceinline__ void traverse_packet_impl(const DevScene& S, v3 o, v3 d, bool valid, bool ux, bool uy,
                                                     bool uz, TraceResult& best) {
    const float inf = __builtin_inff();
    best.t = valid ? inf : -1.0f;
    best.prim = kNoHit;
    best.rank = 0xFFFFFFFFu;
    for (uint32_t i = 0; i < S.n_unb; ++i) {  // planes and quads, as in traverse
        const UnbRec u = S.unb[i];
        float t;
        if (!valid || !plane_quad_test(u, o, d, t)) continue;
        const uint32_t rank = __float_as_uint(u.n.w);
        if (t < best.t || (t == best.t && rank < best.rank)) {
            best.t = t;
            best.prim = kUnbBit | i;
            best.rank = rank;
        }
    }
    if (S.n_nodes == 0) return;

    const float ix = 1.0f / d.x, iy = 1.0f / d.y, iz = 1.0f / d.z;
    const bool sx = kUniformSigns ? ux : ix >= 0.0f, sy = kUniformSigns ? uy : iy >= 0.0f,
               sz = kUniformSigns ? uz : iz >= 0.0f;
    const float tlo = -1e-5f;
    // byte offsets of the NodeH plane blocks for the wave's signs (near planes of the 4 children,
    // then far planes); the mixed-sign instantiation loads both blocks of an axis and selects
    const uint32_t obx = __builtin_amdgcn_readfirstlane(sx ? 16 : 32);
    const uint32_t oby = __builtin_amdgcn_readfirstlane(sy ? 48 : 64);
    const uint32_t obz = __builtin_amdgcn_readfirstlane(sz ? 80 : 96);
    const uint32_t lane = __lane_id();
    uint32_t stk0 = 0, stk1 = 0;  // the wave's stack
    uint32_t sp = 0, cur = 0;     // wave-uniform
    for (;;) {
        if (cur & kLeafBit) {
            const uint32_t first = leaf_first(cur), n_leaf = leaf_count(cur);
            for (uint32_t k = 0; k < n_leaf; ++k) closest_prim(S, uniform_prim(S.prims + first + k), first + k, o, d, best);
        } else {
            // the node in its NodeH form, as in visit_inner: plane t = h (i 2^k) + (c - o) i
            const char* hb = reinterpret_cast<const char*>(S.hnodes) + (size_t)cur * 128u;
            const float4 co = uniform_load4(hb);
            const float4 cw = uniform_load4(hb + 112);
            const uint32_t child[4] = {__float_as_uint(cw.x), __float_as_uint(cw.y), __float_as_uint(cw.z),
                                       __float_as_uint(cw.w)};
            float4 BX, BY, BZ;  // near planes of the 4 children in words 0..1, far planes in 2..3
            // (below, nx .. fz are the distances to those planes)
            if (kUniformSigns) {
                BX = uniform_load4(hb + obx), BY = uniform_load4(hb + oby), BZ = uniform_load4(hb + obz);
            } else {
                const float4 x0 = uniform_load4(hb + 16), x1 = uniform_load4(hb + 32);
                const float4 y0 = uniform_load4(hb + 48), y1 = uniform_load4(hb + 64);
                const float4 z0 = uniform_load4(hb + 80), z1 = uniform_load4(hb + 96);
                BX = sx ? x0 : x1, BY = sy ? y0 : y1, BZ = sz ? z0 : z1;
            }
            const uint32_t ex = __float_as_uint(co.w);
            const float ax = __builtin_ldexpf(ix, (int)(int8_t)(ex & 0xFFu));
            const float ay = __builtin_ldexpf(iy, (int)(int8_t)((ex >> 8) & 0xFFu));
            const float az = __builtin_ldexpf(iz, (int)(int8_t)((ex >> 16) & 0xFFu));
            const float bx = (co.x - o.x) * ix, by = (co.y - o.y) * iy, bz = (co.z - o.z) * iz;
            auto lo16 = [](float w) { const uint32_t u = __float_as_uint(w); return __low2float(*reinterpret_cast<const __half2*>(&u)); };
            auto hi16 = [](float w) { const uint32_t u = __float_as_uint(w); return __high2float(*reinterpret_cast<const __half2*>(&u)); };
            const float nx[4] = {fmaf(lo16(BX.x), ax, bx), fmaf(hi16(BX.x), ax, bx), fmaf(lo16(BX.y), ax, bx),
                                 fmaf(hi16(BX.y), ax, bx)};
            const float fx[4] = {fmaf(lo16(BX.z), ax, bx), fmaf(hi16(BX.z), ax, bx), fmaf(lo16(BX.w), ax, bx),
                                 fmaf(hi16(BX.w), ax, bx)};
            const float ny[4] = {fmaf(lo16(BY.x), ay, by), fmaf(hi16(BY.x), ay, by), fmaf(lo16(BY.y), ay, by),
                                 fmaf(hi16(BY.y), ay, by)};
            const float fy[4] = {fmaf(lo16(BY.z), ay, by), fmaf(hi16(BY.z), ay, by), fmaf(lo16(BY.w), ay, by),
                                 fmaf(hi16(BY.w), ay, by)};
            const float nz[4] = {fmaf(lo16(BZ.x), az, bz), fmaf(hi16(BZ.x), az, bz), fmaf(lo16(BZ.y), az, bz),
                                 fmaf(hi16(BZ.y), az, bz)};
            const float fz[4] = {fmaf(lo16(BZ.z), az, bz), fmaf(hi16(BZ.z), az, bz), fmaf(lo16(BZ.w), az, bz),
                                 fmaf(hi16(BZ.w), az, bz)};
            const float lim = best.t * 1.0001f + 1e-6f;  // < tlo for an invalid lane: nothing overlaps
            // ordering key of a child: the entry distance of the first lane that overlaps it, as
            // float bits (negative distances as 0, so the keys order as unsigned integers on the
            // scalar unit); 0xFFFFFFFF when no lane overlaps it
            uint32_t key[4], val[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const float tn = fmaxf(fmaxf(nx[c], ny[c]), fmaxf(nz[c], tlo));
                const float tf = fminf(fminf(fx[c], fy[c]), fminf(fz[c], lim));
                const unsigned long long m = child[c] != kChildEmpty ? __ballot(tn <= tf * 1.000002f) : 0ull;
                uint32_t k = 0xFFFFFFFFu;
                if (m) {
                    k = (uint32_t)__builtin_amdgcn_readlane(__float_as_int(tn), (int)__builtin_ctzll(m));
                    k = (k >> 31) ? 0u : k;
                }
                key[c] = k;
                val[c] = child[c];
            }
#define CUPBR_PSWAP(a, b)                                                  \
    if (key[b] < key[a]) {                                                  \
        const uint32_t tk = key[a]; key[a] = key[b]; key[b] = tk;           \
        const uint32_t tv = val[a]; val[a] = val[b]; val[b] = tv;           \
    }
            CUPBR_PSWAP(0, 1)
            CUPBR_PSWAP(2, 3)
            CUPBR_PSWAP(0, 2)
            CUPBR_PSWAP(1, 3)
            CUPBR_PSWAP(1, 2)
#undef CUPBR_PSWAP
            if (key[0] != 0xFFFFFFFFu) {
#pragma unroll
                for (int c = 3; c >= 1; --c) {
                    if (key[c] == 0xFFFFFFFFu) continue;
                    if (sp < 64) stk0 = lane == sp ? val[c] : stk0;
                    else stk1 = lane == sp - 64 ? val[c] : stk1;
                    ++sp;
                }
                cur = val[0];
                continue;
            }
        }
        if (sp == 0) break;
        --sp;
        cur = (uint32_t)__builtin_amdgcn_readlane((int)(sp < 64 ? stk0 : stk1), (int)(sp & 63u));
    }
}

__device__ __forceinline__ void traverse_packet(const DevScene& S, v3 o, v3 d, bool valid, TraceResult& best) {
    // an invalid lane's interval is empty whatever planes it is given, so only valid lanes vote
    const unsigned long long v = __ballot(valid);
    const unsigned long long px = __ballot(valid && 1.0f / d.x >= 0.0f), py = __ballot(valid && 1.0f / d.y >= 0.0f),
                             pz = __ballot(valid && 1.0f / d.z >= 0.0f);
    if ((px == 0 || px == v) && (py == 0 || py == v) && (pz == 0 || pz == v))
        traverse_packet_impl<true>(S, o, d, valid, px != 0, py != 0, pz != 0, best);
    else
        traverse_packet_impl<false>(S, o, d, valid, false, false, false, best);
}

// Tracing::traceRay(scene, ray, index), TracingDetail.h:68-116: one object's primitives in order,
// no box test; a mesh keeps its first strictly-closer triangle (MeshDetail.h:28-35)
__device__ __forceinline__ bool object_trace(const DevScene& S, uint32_t obj, v3 o, v3 d, TraceResult& r) {
    r.t = __builtin_inff();
    r.prim = kNoHit;
    r.rank = 0xFFFFFFFFu;
    const ObjInfo& oi = S.objs[obj];
    for (uint32_t k = 0; k < oi.rank_count; ++k) {
        const uint32_t prim = S.rank_prim[oi.rank_base + k];
        if (prim == kNoHit) continue;
        float t;
        bool h;
        if (prim & kUnbBit) {
            h = plane_quad_test(S.unb[prim & ~kUnbBit], o, d, t);
        } else {
            const PrimRec pr = S.prims[prim];
            if ((__float_as_uint(pr.c.w) & 3u) == kPrimTriangle)
                h = mt_test(mk(pr.a.x, pr.a.y, pr.a.z), mk(pr.a.w, pr.b.x, pr.b.y), mk(pr.b.z, pr.b.w, pr.c.x), o, d, t);
            else
                h = sphere_test(mk(pr.a.x, pr.a.y, pr.a.z), pr.a.w, o, d, t);
        }
        if (h && t < r.t) {
            r.t = t;
            r.prim = prim;
            r.rank = oi.rank_base + k;
        }
    }
    return r.prim != kNoHit;
}

// object id and triangle-in-mesh index of a closest-hit result
__device__ __forceinline__ void hit_ids(const DevScene& S, const TraceResult& r, int32_t& obj, int32_t& tri) {
    if (r.prim == kNoHit) { obj = -1; tri = -1; return; }
    if (r.prim & kUnbBit) {
        obj = (int32_t)__float_as_uint(S.unb[r.prim & ~kUnbBit].e1.w);
        tri = -1;
        return;
    }
    obj = (int32_t)__float_as_uint(S.prims[r.prim].c.z);
    const ObjInfo& ob = S.objs[obj];
    tri = ob.type == CUPBR_MESH ? (int32_t)(r.rank - ob.rank_base) : -1;
}

}  // namespace cupbr
