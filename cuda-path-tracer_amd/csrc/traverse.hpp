// Closest-hit traversal over the 64-byte node records (reference: CUDA::trace,
// trace.h:73-169).  Visiting order is the reference's: test both children,
// descend into the nearer (left on ties), defer the farther internal child on
// a stack.  For the lowest-id tie rule the culling keeps children at exactly
// the best distance, and a triangle replaces the best hit when nearer, or
// equally near with a lower original id.  Loops that test triangles later or
// several nodes at once give the same hit: see "the reference's hit from other
// visiting orders".
//
// A node is known by its child word (left child's index << 2 | left internal
// | right internal << 1) before it is visited: its record sits in slot
// word >> 2 and carries its children's words beside their boxes, and its leaf
// children are triangles word >> 2 and (word >> 2) + 1.  So a visit issues
// the record's loads and its leaf triangles' loads together, and waits for
// memory once; with the word inside the record it waited for the record, then
// for the first triangle, then for the second.
#pragma once

#include <algorithm>

#include "devmath.hpp"
#include "pt_api.h"

namespace pt {

struct TraceHit {
    float t;        // FLT_MAX on a miss
    uint32_t id;    // original triangle id, kInvalid on a miss
    float u, v;     // barycentrics of v1, v2
};

// Measurement counts of one lane: node visits, box tests, triangle tests and
// the deepest deferred-node stack reached.
struct TraceCount {
    uint32_t iters, boxes, tris, depth;
};

// Stack bound: every deferred node is the sibling of a distinct ancestor of
// the current node, and a radix tree over < 2^30 augmented 62-bit keys is at
// most 63 internal levels deep.  A push past the bound is not made; it sets
// kStatusStackOverflow in the caller's status word (which the host reports
// as PT_E_INTERNAL), so a violated bound cannot pass silently.
constexpr int kStackMax = 64;
constexpr uint32_t kStatusStackOverflow = PT_STATUS_STACK_OVERFLOW;

__device__ __forceinline__ void raise_status(uint32_t* status, uint32_t bit) {
    if (status) atomicOr(status, bit);
}

template <bool COUNT, bool FINITE>
__device__ __forceinline__ float child_box(V3 o, V3 dinv, float a, float b, float c, float d,
                                           float e, float f) {
    return FINITE ? slab_test_finite(o, dinv, a, b, c, d, e, f) : slab_test(o, dinv, a, b, c, d, e, f);
}

// A triangle record in registers: p0 with the original id, and the edges.
struct TriRec {
    float4 p;
    V3 e1, e2;
};

__device__ __forceinline__ TriRec load_tri(const float4* __restrict__ tris, uint32_t k) {
    const float4* rec = tris + 3 * static_cast<size_t>(k);
    const float* e1 = reinterpret_cast<const float*>(rec + 1);
    const float* e2 = reinterpret_cast<const float*>(rec + 2);
    return TriRec{rec[0], v3(e1[0], e1[1], e1[2]), v3(e2[0], e2[1], e2[2])};
}

__device__ __forceinline__ float tri_test(const TriRec& c, V3 o, V3 d, float& u, float& v) {
    return mt_test(o, d, v3(c.p.x, c.p.y, c.p.z), c.e1, c.e2, u, v);
}

// Closest hit of one ray in a scene of fewer than two triangles, which has no
// internal node: its one triangle `single`, or kInvalid when it is empty.
template <bool COUNT>
__device__ __forceinline__ TraceHit trace_single(const float4* __restrict__ tris, uint32_t single, V3 o, V3 d,
                                                 TraceCount& cnt) {
    TraceHit miss{kFltMax, kInvalid, 0.0f, 0.0f};
    if (single == kInvalid) return miss;
    float u = 0.0f, v = 0.0f;
    if (COUNT) cnt.tris++;
    const TriRec c = load_tri(tris, single);
    const float h = tri_test(c, o, d, u, v);
    return h <= kMinTInit ? TraceHit{h, __float_as_uint(c.p.w), u, v} : miss;
}

// Where a lane keeps a shadow ray's deferred nodes: its column of an LDS
// stack (entry k at lds[k * stride], the first `depth` entries) and a
// private array for the rest; lds == nullptr: a private array throughout.
struct ShadowStack {
    uint32_t* lds = nullptr;
    uint32_t stride = 0;
    int depth = 0;
    uint32_t* spill = nullptr;
};

// Whether a ray hits any triangle of the scene in [b, e) (root word `root`) that the closest-hit
// search would accept (the shadow-ray question of computeL,
// LightAlgorithms.h:12-20: closest-hit t < FLT_MAX).  Until its first hit
// the closest-hit search culls nothing (its bound is still the initial
// one), so it visits the same boxes as this search does and finds a hit
// exactly when this one does; this one stops at the first.  LDSS: the
// deferred nodes go to `ss` (a lane whose own traversal stack is empty
// lends it to its shadow rays) instead of a private array.
template <bool LDSS = false>
__device__ __forceinline__ bool any_hit_in(const float4* __restrict__ nodes, const float4* __restrict__ tris,
                                          uint32_t root, uint32_t b, uint32_t e, V3 o, V3 d, uint32_t* status,
                                          const ShadowStack& ss = ShadowStack{}) {
    float u, v;
    if (e - b == 0) return false;
    if (e - b == 1) return tri_test(load_tri(tris, b), o, d, u, v) <= kMinTInit;
    const V3 dinv = v3(1.0f / d.x, 1.0f / d.y, 1.0f / d.z);
    uint32_t stack[LDSS ? 1 : kStackMax];
    int sp = 0;
    uint32_t word = root;
    for (;;) {
        const uint32_t l = word >> 2;
        const bool in0 = (word & 1u) != 0, in1 = (word & 2u) != 0;
        const float4* rec = nodes + 4 * static_cast<size_t>(l);
        const float4 r0 = rec[0], r1 = rec[1], r2 = rec[2];
        const uint2 cw = *reinterpret_cast<const uint2*>(rec + 3);
        TriRec ta, tb;
        if (!in0) ta = load_tri(tris, l);
        if (!in1) tb = load_tri(tris, l + 1);
        const float h0 = slab_test(o, dinv, r0.x, r0.y, r0.z, r0.w, r1.x, r1.y);
        const float h1 = slab_test(o, dinv, r1.z, r1.w, r2.x, r2.y, r2.z, r2.w);
        uint32_t wt = word;
        asm volatile("" : "+v"(wt));  // keeps the loads above the box tests (see test_children)
        if ((wt & 1u) == 0u && tri_test(ta, o, d, u, v) <= kMinTInit) return true;
        if ((wt & 2u) == 0u && tri_test(tb, o, d, u, v) <= kMinTInit) return true;
        const bool go0 = in0 && h0 <= kMinTInit, go1 = in1 && h1 <= kMinTInit;
        if (go0 && go1) {
            if constexpr (LDSS) {
                if (sp < ss.depth) ss.lds[static_cast<uint32_t>(sp) * ss.stride] = cw.y;
                else if (sp < kStackMax) ss.spill[sp - ss.depth] = cw.y;
                else raise_status(status, kStatusStackOverflow);
                if (sp < kStackMax) ++sp;
            } else {
                if (sp < kStackMax) stack[sp++] = cw.y;
                else raise_status(status, kStatusStackOverflow);
            }
            word = cw.x;
        } else if (go0 || go1) {
            word = go0 ? cw.x : cw.y;
        } else {
            if (sp == 0) return false;
            --sp;
            if constexpr (LDSS) word = sp < ss.depth ? ss.lds[static_cast<uint32_t>(sp) * ss.stride] : ss.spill[sp - ss.depth];
            else word = stack[sp];
        }
    }
}

// ---- persistent traversal -------------------------------------------------
//
// One lane = one ray at a time, advanced one node visit per loop iteration;
// a lane whose ray has finished takes the next ray from its wave's pool, so
// long rays do not hold a whole wave's lanes idle.  The visiting order per ray
// is the reference's.  The deferred-node stack keeps its first LDS entries (8,
// 16 or 32, tuned) in LDS ([depth][thread] so a wave's lanes hit distinct
// banks) and the rest in a private array (scratch), touched only by deep rays.
constexpr int kPersistThreads = 256;

struct RayState {
    V3 o, d, dinv;
    float minT;
    uint32_t best;
    float bu, bv;
    float bound;    // culling distance of the loops that defer or group (see there)
    uint32_t flags; // kRayExact ...
    uint32_t word;  // the node to visit, as its child word
    int sp;
    bool finite;
};
enum : uint32_t {
    kRayExact = 1u,  // walks in the reference's order
    kRayTie = 2u,    // the hit may depend on the order: to be walked again with kRayExact
};

__device__ __forceinline__ void init_ray(RayState& r, uint32_t root, uint32_t flags) {
    r.dinv = v3(1.0f / r.d.x, 1.0f / r.d.y, 1.0f / r.d.z);
    auto normal = [](float x) { return __builtin_fabsf(x) <= kFltMax && x != 0.0f; };
    r.finite = normal(r.dinv.x) && normal(r.dinv.y) && normal(r.dinv.z);
    r.minT = kMinTInit;
    r.best = kInvalid;
    r.bu = 0.0f;
    r.bv = 0.0f;
    r.bound = kMinTInit;
    r.flags = flags;
    r.word = root;
    r.sp = 0;
}

// ---- the reference's hit from other visiting orders ---------------------------
//
// The reference culls a box with h <= (best distance so far), h from the slab
// test and the distance from Moller-Trumbore, which round independently: a
// triangle's t may lie an ulp or more below the h of a box that holds it (flat
// boxes, grazing rays).  Then which triangles are tested, and with equal or
// nearly equal distances which one wins, depends on the order of the tests.  The
// loops below test triangles later than the reference, or many nodes at once,
// and still return its hit:
//
//  - They visit every node that the reference visits.  A node's children are
//    culled with a bound, the minimum of max(t, h of the triangle's own box)
//    over some of the triangles that come before the node in the reference's
//    depth-first order.  Boxes are exact minima and maxima and every step of the
//    slab test is monotonic, so that h is no less than the h of any box around
//    the triangle; and a triangle the reference did not test lies in a box that
//    it had culled, with h above its best distance then, which only falls.  So
//    the bound is never below the reference's best distance at that node.
//  - Of all triangles they test, the lexicographic minimum W of (t, id) is the
//    reference's hit if the reference tested it, and it did unless another
//    triangle's t is below max(t, h) of W: up to W its best distance was no less
//    than the other triangles' minimum, so it culled no box around W.
//  - Where another t is below (kRayTie: overlapping or repeated triangles in a
//    plane along the axes, rays through shared edges), the ray is walked again in
//    the reference's order (kRayExact).  On a model of these loops, 0 of 40,000
//    rays are in soups and rooms, 7 % at the edges of a wall of 3,200 triangles,
//    9 % on two tessellations of one wall, 83 % on 4,000 overlapping decals.
//  - The slab test is monotonic unless a product is NaN: a ray with an infinite
//    or zero dinv component is a tie when one arises, and where a triangle's box is
//    NaN (strict, from the build) every ray walks in the reference's order.
// Against culling by the best distance alone, with the visiting order deciding:
// 16M shell rays 868 us for 869, 2M hair ball rays 1,216 for 1,189, 2,000 rays in a
// soup 20.7 for 18.9, two room frames 4,229 for 4,047; 3,000 to 200,000 rays 5 to
// 20 % more.  Most where the longest walks decide: 200,000 rays onto a closed room
// of 800,000 triangles 58 us for 25 (one lane per ray 189), as the wall that a
// ray hits no longer spares it the mesh behind, which the reference visits first (on
// the model 5.2 visits a ray for 4.5, but 29 rounds for 7 at most).  Where many rays
// are ties (2M rays on 1,500 decals in one plane 1,231 us) it is slower than one
// lane per ray in the reference's order (950).

// Minimum and maximum of distances that are no NaN and no less than zero (the
// maximum also of -0 and, with another that is not, negative ones): of their
// bits, without the canonicalizing instructions of fminf and fmaxf.
__device__ __forceinline__ float near_of(float a, float b) {
    return __int_as_float(min(__float_as_int(a), __float_as_int(b)));
}
__device__ __forceinline__ float far_of(float a, float b) {
    return __int_as_float(max(__float_as_int(a), __float_as_int(b)));
}

// One tested triangle: its distance t (+inf: missed) and the h of its own box
// (0 for kRayExact rays, whose bound is the best distance itself).  Returns
// max(t, h, 0) (t is no less than zero).
__device__ __forceinline__ float take_hit(RayState& r, float t, uint32_t id, float u, float v, float h) {
    const float c = far_of(far_of(t, h), 0.0f);
    const bool better = (t < r.minT) | ((t == r.minT) & (id < r.best));
    const float other = far_of(t, r.minT);  // of the two, not the best
    r.bound = better ? c : r.bound;         // lower, unless it is a tie
    r.minT = better ? t : r.minT;
    r.best = better ? id : r.best;
    r.bu = better ? u : r.bu;
    r.bv = better ? v : r.bv;
    r.flags |= other < r.bound ? kRayTie : 0u;
    return c;
}

// Whether a product of the slab test of a box is NaN.
__device__ __forceinline__ bool slab_nan(V3 o, V3 dinv, float minx, float maxx, float miny, float maxy, float minz,
                                         float maxz) {
    return __builtin_isunordered((minx - o.x) * dinv.x, (maxx - o.x) * dinv.x) ||
           __builtin_isunordered((miny - o.y) * dinv.y, (maxy - o.y) * dinv.y) ||
           __builtin_isunordered((minz - o.z) * dinv.z, (maxz - o.z) * dinv.z);
}

__device__ __forceinline__ TraceHit final_hit(const RayState& r) {
    TraceHit h;
    h.id = r.best;
    h.t = r.best == kInvalid ? kFltMax : r.minT;
    h.u = r.best == kInvalid ? 0.0f : r.bu;
    h.v = r.best == kInvalid ? 0.0f : r.bv;
    return h;
}

// Keeps a lane's private array of deferred nodes in scratch memory.  The
// compiler would otherwise hold a short one (the 32 entries past a 32-entry
// LDS stack) in vector registers: 31 of them in every lane for entries that
// hardly any ray reaches, 4 waves per SIMD for 6.  Not only for that: with the
// array of a 32-entry LDS stack in registers (select chains over its elements)
// the first form of the group code returned wrong hits.  Why is not known; every
// user keeps its array in memory.
__device__ __forceinline__ void keep_in_memory(uint32_t* spill) { asm volatile("" : : "v"(spill) : "memory"); }

// What a visit finds about the node's two children: their box distances (of
// internal children; a leaf's slot holds a box too, its value is discarded)
// and their own words.
struct Children {
    float h0, h1;
    uint32_t w0, w1;
};

// The tests of one visit, in the reference's order.  Leaf children fold into the best hit first.  The
// reference orders a node's two children by distance and lets a leaf replace
// the best hit when nearer, or equally near with a lower id (trace.h:125-160):
// over the leaves of one node that is the lexicographic minimum of (t, id),
// whatever their order.  Taking it before deciding on the internal children
// visits the same nodes: an internal child nearer than a leaf stays within
// the updated best distance, and one farther than a leaf is culled against
// the distance the leaf set, as in the reference.
// ORDERED false: for a group's lane (take_hit); `reach` is lowered to the leaf
// children's max(t, h).
template <bool COUNT, bool FINITE, bool ORDERED = true>
__device__ __forceinline__ Children test_children(const float4* __restrict__ nodes, const float4* __restrict__ tris,
                                                  RayState& r, TraceCount& cnt, float* reach = nullptr) {
    const uint32_t w = r.word;
    const uint32_t l = w >> 2;
    const float4* rec = nodes + 4 * static_cast<size_t>(l);
    const float4 r0 = rec[0], r1 = rec[1], r2 = rec[2];
    const float4 r3 = rec[3];
    // The first leaf child (the left one unless it is internal), and the
    // second of a node with two.
    TriRec ta, tb;
    if ((w & 3u) != 3u) {
        ta = load_tri(tris, (w & 1u) ? l + 1 : l);
        if ((w & 3u) == 0u) tb = load_tri(tris, l + 1);
    }
    if (COUNT) cnt.iters++;
    Children c;
    c.h0 = child_box<COUNT, FINITE>(r.o, r.dinv, r0.x, r0.y, r0.z, r0.w, r1.x, r1.y);
    c.h1 = child_box<COUNT, FINITE>(r.o, r.dinv, r1.z, r1.w, r2.x, r2.y, r2.z, r2.w);
    c.w0 = __float_as_uint(r3.x);
    c.w1 = __float_as_uint(r3.y);
    if (COUNT) cnt.boxes += (w & 1u) + ((w >> 1) & 1u);
    if constexpr (!ORDERED && !FINITE) {
        if (!(r.flags & kRayExact) && (slab_nan(r.o, r.dinv, r0.x, r0.y, r0.z, r0.w, r1.x, r1.y) ||
                                       slab_nan(r.o, r.dinv, r1.z, r1.w, r2.x, r2.y, r2.z, r2.w)))
            r.flags |= kRayTie;
    }
    // An opaque copy of the word: with the same condition as above the
    // compiler would merge the two branches and issue the triangle loads
    // only after the box tests, a second memory round trip.  The record's unused
    // words stay alive up to here too: as registers of a load on its way they
    // would be taken for the triangles' addresses, which then wait for it.
    uint32_t wt = w;
    asm volatile("" : "+v"(wt) : "v"(r3.z), "v"(r3.w));
    if ((wt & 3u) != 3u) {
        float u, v;
        const float t = tri_test(ta, r.o, r.d, u, v);
        const uint32_t id = __float_as_uint(ta.p.w);
        if (COUNT) cnt.tris++;
        if constexpr (!ORDERED) {
            *reach = near_of(*reach, take_hit(r, t, id, u, v, (r.flags & kRayExact) ? 0.0f : ((wt & 1u) ? c.h1 : c.h0)));
        } else if (t < r.minT || (t == r.minT && id < r.best)) {
            r.minT = t; r.best = id; r.bu = u; r.bv = v;
        }
        if ((wt & 3u) == 0u) {
            float u2, v2;
            const float t2 = tri_test(tb, r.o, r.d, u2, v2);
            const uint32_t id2 = __float_as_uint(tb.p.w);
            if (COUNT) cnt.tris++;
            if constexpr (!ORDERED) {
                *reach = near_of(*reach, take_hit(r, t2, id2, u2, v2, (r.flags & kRayExact) ? 0.0f : c.h1));
            } else if (t2 < r.minT || (t2 == r.minT && id2 < r.best)) {
                r.minT = t2; r.best = id2; r.bu = u2; r.bv = v2;
            }
        }
    }
    return c;
}

template <bool COUNT, int LDS, bool FINITE, int COLS = kPersistThreads>
__device__ __forceinline__ bool visit_step(const float4* __restrict__ nodes,
                                           const float4* __restrict__ tris, RayState& r,
                                           uint32_t (*s_stack)[COLS],
                                           uint32_t* spill, TraceCount& cnt, uint32_t* status) {
    const bool in0 = (r.word & 1u) != 0, in1 = (r.word & 2u) != 0;
    const Children c = test_children<COUNT, FINITE>(nodes, tris, r, cnt);
    const float h0 = c.h0, h1 = c.h1;
    const bool g0 = in0 && h0 <= r.minT, g1 = in1 && h1 <= r.minT;
    if (g0 || g1) {
        const bool sw = g1 && (!g0 || h1 < h0);  // left child wins ties (trace.h:125)
        r.word = sw ? c.w1 : c.w0;
        if (g0 && g1) {
            const uint32_t far = sw ? c.w0 : c.w1;
            const int sp = r.sp;
            if (sp < LDS) {
                s_stack[sp][threadIdx.x] = far;
                r.sp = sp + 1;
            } else if (sp < kStackMax) {
                spill[sp - LDS] = far;
                r.sp = sp + 1;
            } else {
                raise_status(status, kStatusStackOverflow);
            }
            if (COUNT) cnt.depth = max(cnt.depth, static_cast<uint32_t>(r.sp));
        }
        return true;
    }
    if (r.sp == 0) return false;
    const int sp = r.sp - 1;
    // The LDS entry is read by every lane and passed through an empty asm
    // statement, so the compiler keeps the LDS and scratch reads apart (a
    // select of the two addresses would become one slower flat load).
    uint32_t next = s_stack[sp < LDS ? sp : LDS - 1][threadIdx.x];
    asm volatile("" : "+v"(next));
    if (sp >= LDS) next = spill[sp - LDS];
    r.word = next;
    r.sp = sp;
    return true;
}

// ---- deferred leaf tests ----------------------------------------------------
//
// In a wave of lanes walking different rays nearly every visit finds a leaf
// child on a few lanes (2.8 of 64 on average), and testing those triangles at
// once costs the whole wave two triangle tests' instructions per visit, more
// than half of all it issues.  walk_step instead notes a node's leaf children
// in the lane's column of an LDS list, with the distances of their boxes, and
// walks on; the wave tests all noted triangles together (test_pending) once
// kFlushLanes lanes cannot go on -- list full, or nothing left to walk -- or no
// lane can.  The bound shrinks a few visits later, so a ray visits somewhat more
// nodes; its hit is the reference's (see above).  A kRayExact lane tests leaf
// children at once.
// Measured (us; 16M shell rays on the 871,200-triangle mesh, 2M camera rays on
// the 2.88M-triangle hair ball, two 1,024 x 1,024 room frames): four entries and
// 6 / 12 / 20 / 32 lanes 879 / 862 / 885 / 1,044, 1,220 / 1,217 / 1,260 / 1,452,
// 4,650 / 4,550 / 4,475 / 4,800; six entries and 12 lanes 869, 1,218, 5,035.  When
// the list came in (tests at once -> four entries, 12 lanes): 897 -> 863, 1,464 ->
// 1,364, 5,790 -> 5,490.
constexpr uint32_t kPend = 4;  // list entries per lane
constexpr uint32_t kFlushLanes = 12;
// LDS words per lane: its stack, then its list (triangles, then distances).
template <int LDS>
constexpr int kRayRows = LDS + 2 * static_cast<int>(kPend);

template <int LDS, bool FINITE, int COLS>
__device__ __forceinline__ void walk_step(const float4* __restrict__ nodes, const float4* __restrict__ tris,
                                          RayState& r, uint32_t& pend, uint32_t (*s_ray)[COLS], uint32_t* spill,
                                          uint32_t* status) {
    const uint32_t w = r.word;
    const uint32_t l = w >> 2;
    const float4* rec = nodes + 4 * static_cast<size_t>(l);
    const float4 r0 = rec[0], r1 = rec[1], r2 = rec[2];
    const uint2 cw = *reinterpret_cast<const uint2*>(rec + 3);
    const float h0 = child_box<false, FINITE>(r.o, r.dinv, r0.x, r0.y, r0.z, r0.w, r1.x, r1.y);
    const float h1 = child_box<false, FINITE>(r.o, r.dinv, r1.z, r1.w, r2.x, r2.y, r2.z, r2.w);
    if constexpr (!FINITE) {
        if (!(r.flags & kRayExact) && (slab_nan(r.o, r.dinv, r0.x, r0.y, r0.z, r0.w, r1.x, r1.y) ||
                                       slab_nan(r.o, r.dinv, r1.z, r1.w, r2.x, r2.y, r2.z, r2.w))) {
            r.flags |= kRayTie;  // ends here
            r.word = kInvalid;
            pend = 0u;
            return;
        }
    }
    if ((w & 3u) != 3u) {
        if (r.flags & kRayExact) {
#pragma unroll 1
            for (uint32_t k = w & 1u; k <= (~w & 2u) >> 1; ++k) {
                const TriRec c = load_tri(tris, l + k);
                float u, v;
                const float t = tri_test(c, r.o, r.d, u, v);
                take_hit(r, t, __float_as_uint(c.p.w), u, v, 0.0f);
            }
        } else {
            uint32_t (*s_pend)[COLS] = s_ray + LDS;
            s_pend[pend][threadIdx.x] = (w & 1u) ? l + 1 : l;
            s_pend[kPend + pend][threadIdx.x] = __float_as_uint((w & 1u) ? h1 : h0);
            if ((w & 3u) == 0u) {
                s_pend[pend + 1u][threadIdx.x] = l + 1;
                s_pend[kPend + pend + 1u][threadIdx.x] = __float_as_uint(h1);
            }
            pend += (w & 3u) == 0u ? 2u : 1u;
        }
    }
    const bool g0 = (w & 1u) && h0 <= r.bound, g1 = (w & 2u) && h1 <= r.bound;
    if (g0 || g1) {
        const bool sw = g1 && (!g0 || h1 < h0);  // left child wins ties (trace.h:125)
        r.word = sw ? cw.y : cw.x;
        if (g0 && g1) {
            const uint32_t far = sw ? cw.x : cw.y;
            const int sp = r.sp;
            if (sp < LDS) {
                s_ray[sp][threadIdx.x] = far;
                r.sp = sp + 1;
            } else if (sp < kStackMax) {
                spill[sp - LDS] = far;
                r.sp = sp + 1;
            } else {
                raise_status(status, kStatusStackOverflow);
            }
        }
        return;
    }
    if (r.sp == 0) {
        r.word = kInvalid;  // nothing left to walk
        return;
    }
    const int sp = r.sp - 1;
    uint32_t next = s_ray[sp < LDS ? sp : LDS - 1][threadIdx.x];
    asm volatile("" : "+v"(next));  // as in visit_step
    if (sp >= LDS) next = spill[sp - LDS];
    r.word = next;
    r.sp = sp;
}

// Tests every noted triangle of the wave, the next one's record on its way
// while one is tested.  A ray that has become a tie ends its walk.
template <int LDS, int COLS>
__device__ __forceinline__ void test_pending(const float4* __restrict__ tris, RayState& r, uint32_t& pend,
                                             uint32_t (*s_ray)[COLS]) {
    uint32_t (*s_pend)[COLS] = s_ray + LDS;
    TriRec rec[2];
    if (pend > 0u) rec[0] = load_tri(tris, s_pend[0][threadIdx.x]);
#pragma unroll
    for (uint32_t k = 0; k < kPend; ++k) {
        if (__ballot(k < pend) == 0ull) break;
        if (k + 1u < pend) rec[(k + 1u) & 1u] = load_tri(tris, s_pend[k + 1u][threadIdx.x]);
        if (k < pend) {
            const TriRec& c = rec[k & 1u];
            float u, v;
            const float t = tri_test(c, r.o, r.d, u, v);
            take_hit(r, t, __float_as_uint(c.p.w), u, v, __uint_as_float(s_pend[kPend + k][threadIdx.x]));
        }
    }
    pend = 0u;
    if (r.flags & kRayTie) {
        r.word = kInvalid;
        r.sp = 0;
    }
}

// One iteration of the wave's walking lanes (`busy`: the lane has a ray), with
// the pending tests when they are due.  Returns whether the lane's ray has
// ended: with kRayTie, to be started again with kRayExact.
template <int LDS, int COLS>
__device__ __forceinline__ bool walk_wave(const float4* __restrict__ nodes, const float4* __restrict__ tris,
                                          RayState& r, uint32_t& pend, bool busy, uint32_t (*s_ray)[COLS],
                                          uint32_t* spill, uint32_t* status) {
    if (busy && r.word != kInvalid && pend <= kPend - 2u) {
        if (r.finite) walk_step<LDS, true>(nodes, tris, r, pend, s_ray, spill, status);
        else walk_step<LDS, false>(nodes, tris, r, pend, s_ray, spill, status);
    }
    const bool stuck = busy && ((r.word == kInvalid && pend > 0u) || pend > kPend - 2u);
    const uint64_t ns = __ballot(stuck);
    if (ns != 0ull && (static_cast<uint32_t>(__popcll(ns)) >= kFlushLanes ||
                       __ballot(busy && !stuck && r.word != kInvalid) == 0ull))
        test_pending<LDS>(tris, r, pend, s_ray);
    return busy && r.word == kInvalid && pend == 0u;
}

// Where many rays are ties, a wave goes over to walking all its further rays in
// the reference's order: once kTieLimit of them were ties, counted with half the
// weight for each pool before (64 rays or more).
constexpr uint32_t kTieLimit = 16;
__device__ __forceinline__ void note_ties(bool tie, uint32_t& ties, uint32_t& flags) {
    const uint64_t tied = __ballot(tie);
    if (tied != 0ull) {
        ties += static_cast<uint32_t>(__popcll(tied));
        if (ties >= kTieLimit) flags = kRayExact;
    }
}

// ---- group traversal -------------------------------------------------------
//
// A ray's visits form a chain: each waits for its record's loads (0.5-1 us
// from the memory side) before it knows the next.  Where a wave has lanes to
// spare -- a launch of fewer rays than the GPU has lanes, or the end of a
// persistent loop, when the few longest rays of each wave are left -- 2^lg
// lanes share one ray: a round takes up to 2^lg nodes off the ray's stack,
// one per lane, tests them together, and puts their surviving children back,
// nearer ones on top of farther ones.  The chain shrinks to about a quarter
// at 8 lanes (longest ray over a 65,536-triangle soup: 282 visits, 44 rounds).
//
// All lanes of a group hold the ray; each keeps the best of the triangles that
// it tested itself (group_best makes the group's hit of them at the end).  The
// stack is in the reference's order from the top down, so what a lane finds
// comes before the nodes of the lanes below it and before the rest of the
// stack, but not before the nodes above: entries are (word, bound) pairs.  A
// round lowers each lane's bound to the minimum over the lanes from it to the
// top, gives that to the children it puts back, and the whole round's minimum to
// the entry below the round's nodes; that entry hands it on when its turn comes.
// (With one bound for the whole group, 27 % of rays on overlapping coplanar
// triangles got another hit than the reference's; on soups and rooms the rounds
// rise by 0.3 %.)  A kRayExact group takes one node a round, which is the
// reference's walk.
//
// The group's stack takes its lanes' columns of the wave's LDS, stacks and leaf
// lists together: words in the first half of the rows, bounds in the second,
// entry e in row e >> lg of column e mod 2^lg.  (As 8-byte pairs a wave's rows
// would overlap those of the workgroup's other waves, which may still walk.)
// With fewer than kGroupReserve free
// entries left the group takes one node a round, which is the depth-first walk of
// one lane: that adds at most 63 entries, and those that do not fit go, as words,
// to the first lane's private array.  One-node rounds pop them with the last
// round's bound (`run`), as everything tested since they were put there comes
// before them.
constexpr uint32_t kGroupReserve = 2 * kPend;
constexpr uint32_t kGroupSpill = kStackMax - kGroupReserve;
static_assert(kGroupReserve + kGroupSpill >= 63, "a one-lane walk from a full group stack");
template <int LDS>
constexpr uint32_t kGroupRows = kRayRows<LDS> / 2;
// Private entries of a lane that walks alone or in a group.
template <int LDS>
constexpr uint32_t kSpillMax = std::max(static_cast<uint32_t>(kStackMax - LDS), kGroupSpill);

// A group's stack size, lanes per group (log2), where the last round's nodes
// began (kInvalid: unknown) and its bound.
struct Group {
    uint32_t sp, lg, from;
    float run;
};

// Whether the group can be given more lanes: its stack is in LDS, or it is a lane
// that walked alone, with at most LDS words.
template <int LDS>
__device__ __forceinline__ bool group_movable(const Group& g) {
    return g.sp <= (g.lg == 0u ? static_cast<uint32_t>(LDS) : kGroupRows<LDS> << g.lg);
}

__device__ __forceinline__ uint32_t lane_u32(uint32_t v, uint32_t src) {
    return static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute(static_cast<int>(src << 2), static_cast<int>(v)));
}
__device__ __forceinline__ float lane_f32(float v, uint32_t src) {
    return __uint_as_float(lane_u32(__float_as_uint(v), src));
}
__device__ __forceinline__ V3 lane_v3(V3 v, uint32_t src) {
    return v3(lane_f32(v.x, src), lane_f32(v.y, src), lane_f32(v.z, src));
}

// Lane operations on rows of 16 lanes without the LDS unit's latency.
template <int CTRL>
__device__ __forceinline__ uint32_t dpp(uint32_t v, uint32_t old) {
    return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(static_cast<int>(old), static_cast<int>(v), CTRL, 0xf, 0xf, false));
}
__device__ __forceinline__ uint32_t bits(uint32_t v) { return v; }
__device__ __forceinline__ uint32_t bits(float v) { return __float_as_uint(v); }
__device__ __forceinline__ void set_bits(uint32_t& v, uint32_t b) { v = b; }
__device__ __forceinline__ void set_bits(float& v, uint32_t b) { v = __uint_as_float(b); }

// The minimum over the lane's group of 2^lg lanes, on all of them.
template <class T, class Min>
__device__ __forceinline__ T group_min(T x, uint32_t lg, Min min2) {
    auto with = [&](uint32_t other) {
        T y;
        set_bits(y, other);
        x = min2(x, y);
    };
    if (lg > 0u) with(dpp<0xB1>(bits(x), bits(x)));   // quad_perm 1,0,3,2
    if (lg > 1u) with(dpp<0x4E>(bits(x), bits(x)));   // quad_perm 2,3,0,1
    if (lg > 2u) with(dpp<0x141>(bits(x), bits(x)));  // row_half_mirror
    if (lg > 3u) with(dpp<0x140>(bits(x), bits(x)));  // row_mirror
    if (lg > 4u) with(lane_u32(bits(x), (threadIdx.x & 63u) ^ 16u));
    if (lg > 5u) with(lane_u32(bits(x), (threadIdx.x & 63u) ^ 32u));
    return x;
}

// The minimum over the lanes of the group from this one, its j-th, to the last.
__device__ __forceinline__ float min_from_here(float x, uint32_t lg, uint32_t j) {
    const uint32_t G = 1u << lg, none = __float_as_uint(__builtin_huge_valf());
    auto with = [&](uint32_t up, uint32_t by) {
        x = j + by < G ? near_of(x, __uint_as_float(up)) : x;
    };
    const uint32_t lane = threadIdx.x & 63u;
    with(dpp<0x101>(__float_as_uint(x), none), 1u);  // row_shl: from the lane above
    if (lg > 1u) with(dpp<0x102>(__float_as_uint(x), none), 2u);
    if (lg > 2u) with(dpp<0x104>(__float_as_uint(x), none), 4u);
    if (lg > 3u) with(dpp<0x108>(__float_as_uint(x), none), 8u);
    // Of a larger group each row's minimum is in its first lane now.
    if (lg > 4u) {
        float rows = __builtin_huge_valf();
        for (uint32_t k = 16u; k < G; k += 16u) {
            const float row = lane_f32(x, lane - j + k);
            rows = k > j ? near_of(rows, row) : rows;
        }
        x = near_of(x, rows);
    }
    return x;
}

// The lanes of this lane's group.
__device__ __forceinline__ uint64_t group_mask(uint32_t lg) {
    const uint32_t lane = threadIdx.x & 63u;
    return (~0ull >> (64u - (1u << lg))) << (lane & ~((1u << lg) - 1u));
}

// Orders the wave's LDS accesses across its lanes (they execute in order; this
// keeps the compiler from moving them).
__device__ __forceinline__ void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// A group stack's entry: word and bound.
template <int LDS, int COLS>
__device__ __forceinline__ uint2 get_entry(uint32_t (*s_ray)[COLS], uint32_t row, uint32_t col) {
    return make_uint2(s_ray[row][col], s_ray[kGroupRows<LDS> + row][col]);
}
template <int LDS, int COLS>
__device__ __forceinline__ void put_entry(uint32_t (*s_ray)[COLS], uint32_t row, uint32_t col, uint32_t word, float bound) {
    s_ray[row][col] = word;
    s_ray[kGroupRows<LDS> + row][col] = __float_as_uint(bound);
}

// Starts the group's ray at `root`.
template <int LDS, int COLS>
__device__ __forceinline__ void group_start(RayState& r, uint32_t root, uint32_t flags, Group& g,
                                            uint32_t (*s_ray)[COLS]) {
    init_ray(r, root, flags);
    if ((threadIdx.x & ((1u << g.lg) - 1u)) == 0u)
        put_entry<LDS>(s_ray, 0u, threadIdx.x, root, kMinTInit);
    g.sp = 1u;
    g.from = kInvalid;
    g.run = kMinTInit;
}

// One round of every group of the wave whose stack is not empty.
template <int LDS, int COLS>
__device__ __forceinline__ void group_round(const float4* __restrict__ nodes, const float4* __restrict__ tris,
                                            RayState& r, Group& gr, uint32_t (*s_ray)[COLS], uint32_t* spill,
                                            uint32_t* status) {
    const uint32_t lg = gr.lg, sp = gr.sp;
    const uint32_t G = 1u << lg, j = threadIdx.x & (G - 1u), first = threadIdx.x - j;
    const uint32_t cap = kGroupRows<LDS> << lg;
    uint32_t (*s_bound)[COLS] = s_ray + kGroupRows<LDS>;
    const uint32_t room =
        !(r.flags & kRayExact) && sp + kGroupReserve < cap ? cap - kGroupReserve - sp : 1u;
    const uint32_t k = min(min(sp, G), room);
    const uint32_t base = sp - k;
    const bool mine = j < k;
    const bool hands_on = j == 0u && base > 0u && base <= cap;  // to the entry below, base - 1
    Children c{0.0f, 0.0f, 0u, 0u};
    TraceCount cnt{0, 0, 0, 0};
    float bound = __builtin_huge_valf(), reach = __builtin_huge_valf();
    wave_fence();
    if (mine) {
        const uint32_t e = base + j;
        const uint2 pair = get_entry<LDS>(s_ray, e < cap ? e >> lg : 0u, first + (e & (G - 1u)));
        uint32_t word = pair.x;
        asm volatile("" : "+v"(word));  // keeps the LDS and scratch reads apart, as in visit_step
        bound = __uint_as_float(pair.y);
        if (e >= cap) {
            word = spill[min(e - cap, kGroupSpill - 1u)];
            bound = gr.run;
        }
        r.word = word;
        c = r.finite ? test_children<false, true, false>(nodes, tris, r, cnt, &reach)
                     : test_children<false, false, false>(nodes, tris, r, cnt, &reach);
    }
    // Bounds of a round's nodes fall from the top down already unless one of them
    // found a hit or lies below the entry that the last round's minimum went to.
    const bool scan = __ballot(mine & ((reach < bound) | (base + 1u < gr.from))) != 0ull;
    bound = near_of(bound, reach);
    if (scan) bound = min_from_here(bound, lg, j);
    const bool g0 = mine && (r.word & 1u) && c.h0 <= bound, g1 = mine && (r.word & 2u) && c.h1 <= bound;
    const uint64_t gm = group_mask(lg), lt = (1ull << (threadIdx.x & 63u)) - 1ull;
    const uint64_t any = __ballot(g0 || g1) & gm, both = __ballot(g0 && g1) & gm;
    if (g0 || g1) {
        const uint32_t p = base + static_cast<uint32_t>(__popcll(any & lt) + __popcll(both & lt));
        const bool sw = g1 && (!g0 || c.h1 < c.h0);  // left child wins ties (trace.h:125)
        const uint32_t near_w = sw ? c.w1 : c.w0, far_w = sw ? c.w0 : c.w1;
        auto put = [&](uint32_t e, uint32_t w) {
            if (e < cap) {
                put_entry<LDS>(s_ray, e >> lg, first + (e & (G - 1u)), w, bound);
            } else if (e - cap < kGroupSpill) {
                spill[e - cap] = w;
            } else {
                raise_status(status, kStatusStackOverflow);
            }
        };
        put(p + (g0 && g1 ? 1u : 0u), near_w);
        if (g0 && g1) put(p, far_w);
    }
    if (hands_on) {  // near_of, in place
        int* below = reinterpret_cast<int*>(&s_bound[(base - 1u) >> lg][first + ((base - 1u) & (G - 1u))]);
        (void)__hip_atomic_fetch_min(below, __float_as_int(bound), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    gr.sp = base + static_cast<uint32_t>(__popcll(any) + __popcll(both));
    gr.from = base;
    gr.run = bound;
    // A tie ends the group's walk (group_best reports it).
    const uint64_t ties = __ballot((r.flags & kRayTie) != 0u);
    if (ties != 0ull && (ties & gm) != 0ull) gr.sp = 0u;
}

// The group's hit on all its lanes (lowest id at the best distance).  Returns
// whether it is a tie.
__device__ __forceinline__ bool group_best(RayState& r, uint32_t lg) {
    const float t = group_min(r.minT, lg, [](float a, float b) { return near_of(a, b); });
    const uint32_t id = group_min(r.minT == t ? r.best : kInvalid, lg, [](uint32_t a, uint32_t b) { return min(a, b); });
    const uint64_t gm = group_mask(lg);
    const uint64_t who = __ballot(r.minT == t && r.best == id) & gm;
    const uint32_t src = static_cast<uint32_t>(__builtin_ctzll(who));
    const float reach = lane_f32(r.bound, src);
    const bool other = (threadIdx.x & 63u) != src && r.best != kInvalid && r.minT < reach;
    const bool tie = (__ballot(other || (r.flags & kRayTie) != 0u) & gm) != 0ull;
    r.minT = t;
    r.best = id;
    r.bu = lane_f32(r.bu, src);
    r.bv = lane_f32(r.bv, src);
    return tie;
}

// Regroups the wave: the groups named by `act` (their first lanes; at most 32)
// become groups of 2^lgn lanes, in order.  Every named group is movable (a lane
// that walked alone has no bounds in its stack: all that it tested comes before
// all of it).  Returns the first lane of the group this lane's new group was, or 64 when there is none
// for it; the caller moves its own per-ray values from that lane.
template <int LDS, int COLS>
__device__ __forceinline__ uint32_t regroup(RayState& r, Group& g, uint32_t lgn, uint64_t act,
                                            uint32_t (*s_ray)[COLS]) {
    constexpr uint32_t R = kGroupRows<LDS>;
    const uint32_t lg = g.lg;
    const uint32_t lane = threadIdx.x & 63u, wcol = threadIdx.x - lane;
    const uint32_t gn = lane >> lgn, jn = lane & ((1u << lgn) - 1u);
    uint32_t own = 64u, i = 0u;
    for (uint64_t m = act; m != 0ull; m &= m - 1ull, ++i)
        if (gn == i) own = static_cast<uint32_t>(__builtin_ctzll(m));
    const uint32_t src = own < 64u ? own : lane;
    const uint32_t moved = lane_u32(g.sp, src);
    const uint32_t n = own < 64u ? moved : 0u;
    const float alone = lane_f32(r.bound, src);
    // A new lane gets at most M of the entries: LDS words, or R << lg pairs, over
    // at least 2 << lg lanes.
    auto move = [&](auto& ent, auto read, auto word, auto bound) {
        constexpr int M = sizeof ent / sizeof ent[0];
        static_assert(M <= static_cast<int>(R), "the entries fit");
        wave_fence();
#pragma unroll
        for (int q = 0; q < M; ++q) {
            const uint32_t e = jn + (static_cast<uint32_t>(q) << lgn);
            if (e < n) ent[q] = read(e);
        }
        wave_fence();
#pragma unroll
        for (int q = 0; q < M; ++q)
            if (jn + (static_cast<uint32_t>(q) << lgn) < n) put_entry<LDS>(s_ray, q, threadIdx.x, word(ent[q]), bound(ent[q]));
        wave_fence();
    };
    if (lg == 0u) {
        uint32_t ent[LDS / 2];
        move(ent, [&](uint32_t e) { return s_ray[e][wcol + src]; }, [](uint32_t w) { return w; }, [&](uint32_t) { return alone; });
    } else {
        uint2 ent[R / 2];
        move(ent, [&](uint32_t e) { return get_entry<LDS>(s_ray, e >> lg, wcol + src + (e & ((1u << lg) - 1u))); },
             [](uint2 p) { return p.x; }, [](uint2 p) { return __uint_as_float(p.y); });
    }
    // A lane's own best goes with it; the group's further lanes hold none.
    const uint32_t bsrc = own < 64u ? (jn < (1u << lg) ? src + jn : src) : lane;
    r.o = lane_v3(r.o, src);
    r.d = lane_v3(r.d, src);
    r.dinv = lane_v3(r.dinv, src);
    r.finite = lane_u32(r.finite ? 1u : 0u, src) != 0u;
    r.minT = lane_f32(r.minT, bsrc);
    r.best = lane_u32(r.best, bsrc);
    r.bu = lane_f32(r.bu, bsrc);
    r.bv = lane_f32(r.bv, bsrc);
    r.bound = lane_f32(r.bound, bsrc);
    r.flags = lane_u32(r.flags, bsrc);
    if (jn >= (1u << lg)) {
        r.minT = r.bound = kMinTInit;
        r.best = kInvalid;
        r.flags &= kRayExact;
    }
    g.sp = n;
    g.lg = lgn;
    g.from = kInvalid;
    return own;
}

// Lanes per group (log2) that spread `count` rays (1..64) over a wave.
__device__ __forceinline__ uint32_t group_log(uint32_t count) {
    return count <= 1u ? 6u : 5u - (31u - static_cast<uint32_t>(__builtin_clz(count - 1u)));
}

// Traces the wave's groups to their ends: `active` groups (stacks in LDS), the
// ray's index in `ray` (equal on all lanes of a group).  Once half the groups
// have ended the rest are given their lanes.
template <int LDS, int COLS, class Load, class Store>
__device__ __forceinline__ void group_trace(const float4* __restrict__ nodes, const float4* __restrict__ tris,
                                            RayState& r, Group& g, bool active, uint32_t ray,
                                            uint32_t (*s_ray)[COLS], uint32_t* spill, uint32_t* status, Load load,
                                            Store store) {
    for (;;) {
        const bool lead = (threadIdx.x & ((1u << g.lg) - 1u)) == 0u;
        const uint64_t act = __ballot(active && lead);
        if (act == 0ull) return;
        const uint32_t lgn = group_log(static_cast<uint32_t>(__popcll(act)));
        if (lgn > g.lg && __ballot(active && !group_movable<LDS>(g)) == 0ull) {
            const uint32_t own = regroup<LDS>(r, g, lgn, act, s_ray);
            ray = lane_u32(ray, own & 63u);
            active = own < 64u;
        }
        group_round<LDS>(nodes, tris, r, g, s_ray, spill, status);
        const bool ended = active && g.sp == 0u;
        if (__ballot(ended) != 0ull) {
            RayState f = r;
            const bool tie = group_best(f, g.lg);
            if (ended) {
                if (tie) {
                    V3 o, d;
                    uint32_t single;
                    group_start<LDS>(r, load(ray, o, d, single), kRayExact, g, s_ray);
                } else {
                    if ((threadIdx.x & ((1u << g.lg) - 1u)) == 0u) store(ray, final_hit(f));
                    active = false;
                }
            }
        }
    }
}

// The end of a persistent loop: the wave's active lanes (at most kTailLanes,
// each with fewer than LDS deferred nodes) go on as groups.  16M shell rays on
// the 871,200-triangle mesh: 870 us without, 921 / 866 / 862 us from 8 / 16 /
// 32 lanes on; 2M camera rays on the 2.88M-triangle hair ball 1,219 us
// without, 1,407 / 1,279 / 1,217.
constexpr uint32_t kTailLanes = 32;
static_assert(kTailLanes <= 32, "regroup takes at most 32 groups");

template <int LDS, int COLS, class Load, class Store>
__device__ __forceinline__ void group_tail(const float4* __restrict__ nodes, const float4* __restrict__ tris,
                                           RayState& r, uint32_t pend, bool active, uint32_t ray,
                                           uint32_t (*s_ray)[COLS], uint32_t* spill, uint32_t* status, Load load,
                                           Store store) {
    test_pending<LDS>(tris, r, pend, s_ray);
    if (active && (r.flags & kRayTie)) {
        V3 o, d;
        uint32_t single;
        init_ray(r, load(ray, o, d, single), kRayExact);
    }
    const bool walking = active && r.word != kInvalid;
    if (walking) s_ray[r.sp][threadIdx.x] = r.word;
    if (active && !walking) store(ray, final_hit(r));
    Group g{walking ? static_cast<uint32_t>(r.sp) + 1u : 0u, 0u, kInvalid, kMinTInit};
    group_trace<LDS>(nodes, tris, r, g, walking, ray, s_ray, spill, status, load, store);
}

// A launch of few rays: wave w traces rays [w << (6 - lg), ...) with 2^lg lanes
// each from the start, without a queue.
template <int LDS, int COLS, class Load, class Store>
__device__ __forceinline__ void grouped_trace(const float4* __restrict__ nodes, const float4* __restrict__ tris,
                                              uint32_t nrays, uint32_t lg, uint32_t flags, uint32_t* status,
                                              uint32_t (*s_ray)[COLS], Load load, Store store) {
    uint32_t spill[kSpillMax<LDS>];
    keep_in_memory(spill);
    const uint32_t ray = (blockIdx.x * static_cast<uint32_t>(COLS) + threadIdx.x) >> lg;
    const bool lead = (threadIdx.x & ((1u << lg) - 1u)) == 0u;
    RayState r;
    r.o = r.d = v3(0.0f, 0.0f, 0.0f);
    init_ray(r, 0u, 0u);
    Group g{0u, lg, kInvalid, kMinTInit};
    bool active = false;
    if (ray < nrays) {
        uint32_t single = kInvalid;
        const uint32_t root = load(ray, r.o, r.d, single);
        if (root == kInvalid) {
            TraceCount cnt{0, 0, 0, 0};
            const TraceHit h = trace_single<false>(tris, single, r.o, r.d, cnt);
            if (lead) store(ray, h);
        } else {
            group_start<LDS>(r, root, flags, g, s_ray);
            active = true;
        }
    }
    group_trace<LDS>(nodes, tris, r, g, active, ray, s_ray, spill, status, load, store);
}

// Lanes per ray (log2) of a launch of `nrays` rays on `lanes` lanes: as many as
// there are lanes for, at most 2^kGroupMax; 0: one lane per ray, persistent.
// Measured: 2,000 rays in a 4,096-triangle soup 58 us with one lane per ray, 26
// with up to 8, 23 with up to 16, 22 with up to 32; 131,072 rays (4 lanes) after a
// rebuild of 2^20 triangles 448 -> 291 us; eight 65,536-path frames in a row 3,650
// -> 1,520 us.  At 16 the wider rounds already find too few nodes to go further.
constexpr uint32_t kGroupMax = 4;
inline uint32_t launch_group(uint64_t nrays, uint64_t lanes) {
    uint32_t lg = 0;
    const uint64_t most = lanes < (1ull << 31) ? lanes : 1ull << 31;  // thread indices are 32-bit
    while (lg < kGroupMax && (nrays << (lg + 1)) <= most) ++lg;
    return lg;
}
// Workgroups of such a launch.
inline uint32_t grouped_blocks(uint64_t nrays, uint32_t lg) {
    return static_cast<uint32_t>(((nrays << lg) + kPersistThreads - 1) / kPersistThreads);
}

// Ray hand-out.  The rays [0, nrays) are cut into pools, and the pools dealt to
// nq slices (nq <= 64, about one per 16K rays; slice q has pools q, q + nq, ...),
// each with its own counter 256 bytes from the next: one address sustains only
// about 90 M returning atomics/s on MI355X, so a single counter caps how small
// the pools can be, and large pools leave waves unevenly loaded at the end.  A
// wave starts on slice (wave index mod nq), takes pools from it and, once it is
// used up, moves on to the next slice that is neither marked in a 64-bit mask of
// used-up slices nor found used up by its own probes.  A slice is marked by the
// one wave that takes its last pool; the mask only saves probes.  A wave stops
// when every slice is marked or found used up.  Counters and mask live in one
// queue block of kQueueWords words that the caller zeroes (zero_queue) before
// the launch.
// Dealing pools keeps the rays in flight together in the caller's order, so that
// neighbours of an image share their nodes in the caches: with slices of
// contiguous rays, 64 places of an image at a time, 10^6 camera rays on the
// 871,200-triangle mesh took 365 us (234), 700,000 on a hair ball of 50,000
// triangles 162 (117), 2,073,600 on one of 2.88M 1,215 (1,170), 4M in a soup 920
// (858); 16M shell rays in no order 865 (857).  (Both sides measured with culling
// by the best distance alone, which camera rays walk 2-3 % faster.)
constexpr uint32_t kQueueSlices = 64;
constexpr uint32_t kQueueStride = 64;  // words between counters (256 bytes)
constexpr uint32_t kQueueMask = kQueueSlices * kQueueStride;  // word offset of the mask
constexpr uint32_t kQueueWords = kQueueMask + 64;
constexpr uint32_t kSliceRays = 16384;

// Pools of nrays rays, and those of slice q.
__device__ __forceinline__ uint32_t pool_count(uint32_t nrays, uint32_t pool) {
    return nrays / pool + (nrays % pool != 0u ? 1u : 0u);
}
__device__ __forceinline__ uint32_t slice_pools(uint32_t pools, uint32_t nq, uint32_t q) {
    return pools > q ? (pools - 1u - q) / nq + 1u : 0u;
}

__device__ __forceinline__ uint32_t queue_slices(uint32_t nrays) {
    return min(kQueueSlices, max(1u, nrays / kSliceRays));
}


// Zeroes the counters and the mask of `levels` consecutive queue blocks with
// the threads of one workgroup.
__device__ __forceinline__ void zero_queue(uint32_t* __restrict__ queue, uint32_t levels) {
    const uint32_t per = kQueueSlices + 2;
    for (uint32_t i = threadIdx.x; i < levels * per; i += blockDim.x) {
        const uint32_t lvl = i / per, k = i % per;
        queue[lvl * kQueueWords + (k < kQueueSlices ? k * kQueueStride : kQueueMask + (k - kQueueSlices))] = 0u;
    }
}

// Persistent closest-hit loop over rays [0, nrays), handed out in per-wave
// pools from the queue block `queue` (see above): pool_large rays (tuned,
// 256 by default) when there are at least four per lane of the grid, else 64
// so that a short queue still spreads over every wave.  Idle lanes are
// refilled when fewer than `refill` (1..64) lanes of the wave are busy.
// load(i, o, d) fetches ray i; store(i, hit) writes its result.  load returns
// the ray's root node's word, or kInvalid for a scene without one (fewer
// than two triangles); then `single` names its one triangle (or kInvalid) and
// the ray is answered at once without entering the loop.
constexpr uint32_t kRayPoolSmall = 64;

// The pool size a launch uses, from the tuned one.
inline uint32_t pool_for(uint32_t pool) { return std::max(kRayPoolSmall, pool); }

template <bool COUNT, int LDS, class Load, class Store>
__device__ __forceinline__ void persistent_trace(const float4* __restrict__ nodes,
                                                 const float4* __restrict__ tris, uint32_t nrays,
                                                 uint32_t* __restrict__ queue, uint32_t* status,
                                                 uint32_t refill, uint32_t pool_large, uint32_t flags,
                                                 uint32_t (*s_ray)[kPersistThreads], Load load, Store store,
                                                 TraceCount& cnt) {
    // Waves past one per kRayPoolSmall rays leave at once: every wave that
    // stays drains the queue with the others, and on a short queue (a late
    // render level, a cache frame's training levels) the extra waves would
    // only add returning atomics on its few slice counters.
    const uint32_t wave_id = __builtin_amdgcn_readfirstlane(blockIdx.x * (blockDim.x / 64u) + threadIdx.x / 64u);
    if (wave_id > 0u && static_cast<uint64_t>(wave_id) * kRayPoolSmall >= nrays) return;
    uint32_t spill[kSpillMax<LDS>];
    keep_in_memory(spill);
    const int lane = threadIdx.x & 63;
    const uint64_t lt = (1ull << lane) - 1ull;
    RayState r;
    bool active = false;
    uint32_t ray = 0, pend = 0;
    uint32_t pool_next = 0, pool_end = 0;  // wave-uniform
    bool drained = false;                  // wave-uniform: no rays left to hand out
    const uint32_t pool =
        nrays / 4u >= gridDim.x * blockDim.x ? pool_large : kRayPoolSmall;
    const uint32_t nq = queue_slices(nrays);
    const uint32_t pools = pool_count(nrays, pool);
    const uint64_t all = nq == 64u ? ~0ull : (1ull << nq) - 1ull;
    uint64_t* mask = reinterpret_cast<uint64_t*>(queue + kQueueMask);
    // Wave-uniform state is read through readfirstlane so that it lives in
    // scalar registers (the compiler cannot tell that threadIdx.x / 64 is
    // uniform over a wave).
    uint32_t q = wave_id % nq;
    uint32_t ties = 0;     // wave-uniform (note_ties)
    uint64_t seen = ~all;  // wave-uniform: slices this wave found used up
    bool used_up = false;  // wave-uniform: the refill loop found slice q used up
    for (;;) {
        const uint64_t busy = __ballot(active);
        if (!drained && static_cast<uint32_t>(__popcll(busy)) < refill) {
            uint64_t idle = ~busy;
            while (idle != 0ull) {
                if (pool_next >= pool_end) {
                    const uint32_t len = slice_pools(pools, nq, q);
                    uint32_t base = 0;
                    if (lane == 0) {
                        base = atomicAdd(queue + q * kQueueStride, 1u);
                        // Only the slice's last pool marks it:
                        // one atomic per slice (every wave marking the slices
                        // it finds used up would serialise on the mask).
                        if (base + 1u == len) atomicOr(mask, 1ull << q);
                    }
                    base = __builtin_amdgcn_readfirstlane(base);
                    if (base >= len) {
                        used_up = true;
                        break;
                    }
                    pool_next = (base * nq + q) * pool;
                    pool_end = pool_next + min(pool, nrays - pool_next);
                    ties >>= 1;
                }
                const uint32_t avail = pool_end - pool_next;
                const uint32_t rank = static_cast<uint32_t>(__popcll(idle & lt));
                const bool take = ((idle >> lane) & 1ull) && rank < avail;
                const uint32_t took = min(static_cast<uint32_t>(__popcll(idle)), avail);
                if (take) {
                    ray = pool_next + rank;
                    uint32_t single = kInvalid;
                    const uint32_t root = load(ray, r.o, r.d, single);
                    if (root == kInvalid) {
                        store(ray, trace_single<COUNT>(tris, single, r.o, r.d, cnt));
                    } else {
                        init_ray(r, root, flags);
                        active = true;
                    }
                }
                pool_next += took;
                idle = ~__ballot(active);
            }
            if (used_up) {
                // Slice q is used up: move to the next slice not known to be
                // used up (kept out of the refill loop above, which stays
                // short).  Every visit here adds a slice to `seen`, so after
                // at most nq of them the wave has a slice with rays or knows
                // that all are used up.
                used_up = false;
                seen |= 1ull << q;
                uint32_t lo = 0, hi = 0;
                if (lane == 0) {
                    const uint64_t m = __hip_atomic_load(mask, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    lo = static_cast<uint32_t>(m);
                    hi = static_cast<uint32_t>(m >> 32);
                }
                lo = __builtin_amdgcn_readfirstlane(lo);
                hi = __builtin_amdgcn_readfirstlane(hi);
                const uint64_t open = ~(seen | (static_cast<uint64_t>(hi) << 32) | lo);
                if (open == 0ull) {
                    drained = true;
                } else {
                    const uint64_t above = q < 63u ? open & (~0ull << (q + 1u)) : 0ull;
                    q = static_cast<uint32_t>(__builtin_ctzll(above ? above : open));
                }
            }
        }
        // Once no slice has rays left the wave ends with groups (group_trace)
        // as soon as kTailLanes rays or fewer are left, all with their
        // deferred nodes in LDS.
        if (drained) {
            const uint64_t left = __ballot(active);
            if (left == 0ull) break;
            if (!COUNT && static_cast<uint32_t>(__popcll(left)) <= kTailLanes && __ballot(active && r.sp >= LDS) == 0ull) {
                group_tail<LDS>(nodes, tris, r, pend, active, ray, s_ray, spill, status, load, store);
                break;
            }
        }
        bool ended;
        if constexpr (COUNT) {  // the reference's order of visits and tests, which the counts describe
            ended = active && !(r.finite ? visit_step<true, LDS, true>(nodes, tris, r, s_ray, spill, cnt, status)
                                         : visit_step<true, LDS, false>(nodes, tris, r, s_ray, spill, cnt, status));
        } else {
            ended = walk_wave<LDS>(nodes, tris, r, pend, active, s_ray, spill, status);
        }
        note_ties(ended && (r.flags & kRayTie), ties, flags);
        if (ended) {
            if (r.flags & kRayTie) {
                V3 o, d;
                uint32_t single;
                init_ray(r, load(ray, o, d, single), kRayExact);
            } else {
                store(ray, final_hit(r));
                active = false;
            }
        }
    }
}

// ---- root filter ---------------------------------------------------------
//
// A batch of rays that start outside the scene's box (the closest-hit
// microbench's shell rays) mostly leaves after the root visit.  In the
// persistent loop above such a ray takes a lane through a refill and one
// visit while its neighbours walk deep paths, so most of the wave's issue
// slots go to lanes that do nothing.  The filtered variant first runs the
// root visit of 64 fresh rays at once on every lane of the wave (busy lanes
// keep their own ray's state in other registers), answers the rays that end
// there, and queues the rest ("survivors") in a per-wave LDS ring; idle
// lanes take survivors from the ring and trace them from the root as above.
// Results are the same bits: a ray that ends at the root visit ends exactly
// as the full traversal would, and a survivor is traced in full.

constexpr uint32_t kSurvCap = 128;  // survivor ring entries per wave
// Lanes are refilled from the ring already when fewer than this many are busy:
// with a survivor ready for every idle lane, or no more rays to filter, that
// costs no filter round.  (Filter rounds wait for the launch's `refill`: with 48
// for both, 16M shell rays, which mostly end in the filter, took 1 % longer.)
// 2.88M-triangle hair ball, 2,073,600 camera rays: 1,393 us without, 1,262 at 48,
// 1,217 at 56; 16M shell rays on the 871,200-triangle mesh 854, 867 and 862.
constexpr uint32_t kReadyRefill = 56;

// The root visit alone (visit_step's decisions without the stack): leaf
// children fold into the best hit; returns whether an internal child is to
// be visited.
template <bool FINITE>
__device__ __forceinline__ bool root_visit(const float4* __restrict__ nodes, const float4* __restrict__ tris,
                                           RayState& r) {
    const bool in0 = (r.word & 1u) != 0, in1 = (r.word & 2u) != 0;
    TraceCount cnt;
    const Children c = test_children<false, FINITE>(nodes, tris, r, cnt);
    return (in0 && c.h0 <= r.minT) || (in1 && c.h1 <= r.minT);
}

// persistent_trace with the root filter (no counting).  s_surv: this wave's
// kSurvCap-entry ring in LDS.  The hand-out protocol (pools from slice
// counters, used-up mask, `seen`) is persistent_trace's; a wave stops once
// every slice is used up, its ring is empty and no lane is busy.
template <int LDS, class Load, class Store>
__device__ __forceinline__ void persistent_trace_filtered(const float4* __restrict__ nodes,
                                                          const float4* __restrict__ tris, uint32_t nrays,
                                                          uint32_t* __restrict__ queue, uint32_t* status,
                                                          uint32_t refill, uint32_t pool_large, uint32_t flags,
                                                          uint32_t (*s_ray)[kPersistThreads],
                                                          uint32_t* __restrict__ s_surv, Load load, Store store) {
    const uint32_t wave_id = __builtin_amdgcn_readfirstlane(blockIdx.x * (blockDim.x / 64u) + threadIdx.x / 64u);
    if (wave_id > 0u && static_cast<uint64_t>(wave_id) * kRayPoolSmall >= nrays) return;
    uint32_t spill[kSpillMax<LDS>];
    keep_in_memory(spill);
    TraceCount cnt{0, 0, 0, 0};
    const int lane = threadIdx.x & 63;
    const uint64_t lt = (1ull << lane) - 1ull;
    RayState r;
    bool active = false;
    uint32_t ray = 0, pend = 0;
    uint32_t pool_next = 0, pool_end = 0;  // wave-uniform
    bool drained = false;                  // wave-uniform: no rays left to hand out
    uint32_t qhead = 0, qtail = 0;         // wave-uniform: survivor ring positions
    const uint32_t pool =
        nrays / 4u >= gridDim.x * blockDim.x ? pool_large : kRayPoolSmall;
    const uint32_t nq = queue_slices(nrays);
    const uint32_t pools = pool_count(nrays, pool);
    const uint64_t all = nq == 64u ? ~0ull : (1ull << nq) - 1ull;
    uint64_t* mask = reinterpret_cast<uint64_t*>(queue + kQueueMask);
    uint32_t q = wave_id % nq;
    uint32_t ties = 0;
    uint64_t seen = ~all;
    for (;;) {
        const uint32_t nbusy = static_cast<uint32_t>(__popcll(__ballot(active)));
        const uint32_t ready = qtail - qhead;
        if (nbusy < (ready + nbusy >= 64u || drained ? max(refill, kReadyRefill) : refill) && (!drained || ready != 0u)) {
            // Filter rounds until the ring can fill every idle lane (or the
            // rays run out).  Each pass either consumes pool rays, takes a
            // new pool, or finds a slice used up (at most nq times).
            while (!drained && qtail - qhead < 64u - nbusy && qtail - qhead <= kSurvCap - 64u) {
                if (pool_next >= pool_end) {
                    const uint32_t len = slice_pools(pools, nq, q);
                    uint32_t base = 0;
                    if (lane == 0) {
                        base = atomicAdd(queue + q * kQueueStride, 1u);
                        if (base + 1u == len) atomicOr(mask, 1ull << q);
                    }
                    base = __builtin_amdgcn_readfirstlane(base);
                    if (base >= len) {
                        seen |= 1ull << q;
                        uint32_t lo = 0, hi = 0;
                        if (lane == 0) {
                            const uint64_t m = __hip_atomic_load(mask, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                            lo = static_cast<uint32_t>(m);
                            hi = static_cast<uint32_t>(m >> 32);
                        }
                        lo = __builtin_amdgcn_readfirstlane(lo);
                        hi = __builtin_amdgcn_readfirstlane(hi);
                        const uint64_t open = ~(seen | (static_cast<uint64_t>(hi) << 32) | lo);
                        if (open == 0ull) {
                            drained = true;
                        } else {
                            const uint64_t above = q < 63u ? open & (~0ull << (q + 1u)) : 0ull;
                            q = static_cast<uint32_t>(__builtin_ctzll(above ? above : open));
                        }
                        continue;
                    }
                    pool_next = (base * nq + q) * pool;
                    pool_end = pool_next + min(pool, nrays - pool_next);
                    ties >>= 1;
                }
                const uint32_t avail = min(64u, pool_end - pool_next);
                const uint32_t fr = pool_next + static_cast<uint32_t>(lane);
                bool surv = false;
                if (static_cast<uint32_t>(lane) < avail) {
                    RayState f;
                    uint32_t single = kInvalid;
                    const uint32_t root = load(fr, f.o, f.d, single);
                    if (root == kInvalid) {
                        store(fr, trace_single<false>(tris, single, f.o, f.d, cnt));
                    } else {
                        init_ray(f, root, flags);
                        surv = f.finite ? root_visit<true>(nodes, tris, f) : root_visit<false>(nodes, tris, f);
                        if (!surv) store(fr, final_hit(f));
                    }
                }
                const uint64_t sm = __ballot(surv);
                if (surv) s_surv[(qtail + static_cast<uint32_t>(__popcll(sm & lt))) & (kSurvCap - 1u)] = fr;
                qtail += static_cast<uint32_t>(__popcll(sm));
                pool_next += avail;
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            // Idle lanes take survivors, in ring order.
            const uint64_t idle = ~__ballot(active);
            const uint32_t qn = qtail - qhead;
            const uint32_t rank = static_cast<uint32_t>(__popcll(idle & lt));
            if (((idle >> lane) & 1ull) && rank < qn) {
                ray = s_surv[(qhead + rank) & (kSurvCap - 1u)];
                uint32_t single = kInvalid;
                const uint32_t root = load(ray, r.o, r.d, single);
                init_ray(r, root, flags);
                active = true;
            }
            qhead += min(static_cast<uint32_t>(__popcll(idle)), qn);
        }
        if (drained && qtail == qhead) {  // as in persistent_trace
            const uint64_t left = __ballot(active);
            if (left == 0ull) break;
            if (static_cast<uint32_t>(__popcll(left)) <= kTailLanes && __ballot(active && r.sp >= LDS) == 0ull) {
                group_tail<LDS>(nodes, tris, r, pend, active, ray, s_ray, spill, status, load, store);
                break;
            }
        }
        const bool ended = walk_wave<LDS>(nodes, tris, r, pend, active, s_ray, spill, status);
        note_ties(ended && (r.flags & kRayTie), ties, flags);
        if (ended) {
            if (r.flags & kRayTie) {
                V3 o, d;
                uint32_t single;
                init_ray(r, load(ray, o, d, single), kRayExact);
            } else {
                store(ray, final_hit(r));
                active = false;
            }
        }
    }
}

}  // namespace pt
