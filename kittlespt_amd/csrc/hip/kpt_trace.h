// kpt_trace.h — two-level BVH2 traversal for gfx950 (device code).
//
// Semantics are those of TLAS::intersect / TLAS::intersectP (tlas.cu:8-125)
// with BLAS2::intersect / intersectP (blas.cuh:50-188), restructured for the
// GPU:
//   * one loop and one stack for both levels; a stack entry carries a level
//     bit, so the BLAS of a TLAS leaf is traversed to completion before the
//     next TLAS entry is popped (LIFO), exactly as the nested reference calls;
//   * the nearer child is kept in a register ("current entry") instead of
//     being pushed and popped at once, and only the farther sibling goes on
//     the stack; the visiting order is the reference's (it pushes the farther
//     child first and pops the nearer one next);
//   * the per-lane stack lives in LDS ([entry][lane] layout: lanes of a wave
//     hit distinct banks) with a private-memory (scratch) spill region for
//     entries beyond the LDS depth, instead of the reference's fixed 16-entry
//     register array that overflows on deep trees;
//   * the BLAS is entered with tmax = min(tmax, closest-so-far).  The reference
//     starts every BLAS with the original tmax and a local closest of +inf;
//     nodes this extra bound skips have a slab entry at or beyond the
//     closest hit, so in exact arithmetic every triangle under them is too,
//     and TLAS::intersect keeps a hit only if strictly closer; the nodes that
//     remain are visited in the reference's order, so the closest hit
//     (including which of two equal-distance hits wins) is the same.  In
//     float the argument has one gap: a triangle whose rounded distance
//     falls below the rounded slab entry of its own box, with another
//     instance's hit in between.  Overlapping coplanar instances a few ulps
//     apart (flat boxes, ties on most rays) never showed it: the oracle's
//     bounded mode equals its reference mode on 600,000 such rays, and these
//     kernels equal the reference mode on the same rays;
//   * any-hit needs no ordering: its result is "some reachable triangle is
//     hit", which does not depend on the visiting order; it visits the
//     nearer child first, which finds occluders close to the origin sooner;
//   * a node is represented by a 32-bit entry (below) kept in its parent's
//     NodePair, so an interior step is one 64-byte line and nothing is decoded.
//
// What bounds it and what that decided (1000 instances, 1.24 M triangles,
// 1920x1080 camera rays and their bounces).  With one loop in which each lane
// ran its own kind of step, a vector instruction had 18 (camera rays) or 9
// (paths) of 64 lanes at work.  So a wave runs one kind of step at a time
// (Trav::round), and the triangles of its leaves are spread over all its lanes
// (Trav::leaves), half of a ray's work and the half whose lanes were fewest.
// Now 44 (camera rays) and 32 (paths) lanes are, and the camera rays take 0.68
// of the instructions; at four cycles each they fill 0.8 of the SIMDs' cycles,
// while a wave waits for 60 % of its own: instructions and latency together.
// Waiting for more lanes to reach the chosen kind costs more than it fills:
// passes at 8, 4, 2 and 1 lanes at leaves and instances took 1458, 1260, 1204
// and 1125 us for a million incoherent rays.  Interior steps come four to a
// round (a round of one: 1590 us against 1458 for two, 1173 for four at two
// lanes).  Node pairs instead of two-level 192-byte records: a third of the
// footprint and of the cache accesses, and 64 registers instead of 96 (8 waves
// per SIMD instead of 5; a few more spilled cost up to twice the time).
// Closest-hit launch alone on the GPU 2.60 -> 1.74 ms, a million incoherent
// rays 2.09 -> 1.11 ms, fifty thousand any-hit rays 124 -> 70 us.
// Traversal is a state machine (init / round) so persistent kernels can refill
// a lane with a new ray, and park a lane's, between rounds.
#pragma once
#include "kpt_vec.h"
#include "../common/kpt_device_types.h"

namespace kpt {

constexpr int TRACE_BLOCK = 256;      // threads per workgroup of the fixed-shape trace kernels
constexpr int LDS_STACK = 16;         // stack entries per lane held in LDS (fixed-shape kernels)
constexpr int STACK_TOTAL = 128;      // entries per lane, LDS and private together (and one that marks the end);
                                      // a push beyond overflows
// The wavefront's persistent kernels take their LDS depth and workgroup size
// from the tuning knobs (dynamic LDS of depth x workgroup words); the private
// spill array is sized for the shallowest LDS part, so the total capacity is
// STACK_TOTAL whatever the depth.
constexpr int LDS_STACK_MIN = 8;
constexpr int LDS_STACK_MAX = 32;
constexpr int SPILL_STACK = STACK_TOTAL + 1 - LDS_STACK_MIN;
constexpr uint32_t TLAS_BIT = 0x80000000u;
struct Ray {
    v3 o, d, inv;
};
KD Ray make_ray(v3 o, v3 d) { Ray r; r.o = o; r.d = d; r.inv = 1.0f / d; return r; }

struct Hit {
    float t;
    int32_t slot;   // triangle slot (-1 = miss)
    int32_t inst;
    float u, v;
};

struct TraceCounts {
    uint32_t interior, leaf, tri, entries, tlas;
};

// Bounds3f::intersectP, bounds.cuh:38-57
KD bool slab(const float4& lo, const float4& hi, const Ray& r, float tmin, float tmax, float* tenter) {
    float t0x = (lo.x - r.o.x) * r.inv.x, t0y = (lo.y - r.o.y) * r.inv.y, t0z = (lo.z - r.o.z) * r.inv.z;
    float t1x = (hi.x - r.o.x) * r.inv.x, t1y = (hi.y - r.o.y) * r.inv.y, t1z = (hi.z - r.o.z) * r.inv.z;
    float ex = fminf_(t0x, t1x), ey = fminf_(t0y, t1y), ez = fminf_(t0z, t1z);
    float xx = fmaxf_(t0x, t1x), xy = fmaxf_(t0y, t1y), xz = fmaxf_(t0z, t1z);
    float te = fmaxf_(fmaxf_(ex, ey), ez);
    float tx = fminf_(fminf_(xx, xy), xz);
    *tenter = te;
    return (te <= tx) && (tx >= tmin) && (te <= tmax);
}

// The slab's entry and exit distances alone (slab above, without its tests).
KD void slab_range(const float4& lo, const float4& hi, const Ray& r, float* tenter, float* texit) {
    float t0x = (lo.x - r.o.x) * r.inv.x, t0y = (lo.y - r.o.y) * r.inv.y, t0z = (lo.z - r.o.z) * r.inv.z;
    float t1x = (hi.x - r.o.x) * r.inv.x, t1y = (hi.y - r.o.y) * r.inv.y, t1z = (hi.z - r.o.z) * r.inv.z;
    *tenter = fmaxf_(fmaxf_(fminf_(t0x, t1x), fminf_(t0y, t1y)), fminf_(t0z, t1z));
    *texit = fminf_(fminf_(fmaxf_(t0x, t1x), fmaxf_(t0y, t1y)), fmaxf_(t0z, t1z));
}

KD void load_node(const Node* nodes, uint32_t i, float4* lo, float4* hi) {
    const float4* p = reinterpret_cast<const float4*>(nodes + i);
    *lo = p[0];
    *hi = p[1];
}

// Object-space ray: Ray::transform (ray.cuh:25-29) with the full 4-term rows.
KD Ray object_ray(const InstTrav& it, const Ray& w) {
    v3 o = mk3(it.r0[0] * w.o.x + it.r0[1] * w.o.y + it.r0[2] * w.o.z + it.r0[3] * 1.0f,
               it.r1[0] * w.o.x + it.r1[1] * w.o.y + it.r1[2] * w.o.z + it.r1[3] * 1.0f,
               it.r2[0] * w.o.x + it.r2[1] * w.o.y + it.r2[2] * w.o.z + it.r2[3] * 1.0f);
    v3 d = mk3(it.r0[0] * w.d.x + it.r0[1] * w.d.y + it.r0[2] * w.d.z + it.r0[3] * 0.0f,
               it.r1[0] * w.d.x + it.r1[1] * w.d.y + it.r1[2] * w.d.z + it.r1[3] * 0.0f,
               it.r2[0] * w.d.x + it.r2[1] * w.d.y + it.r2[2] * w.d.z + it.r2[3] * 0.0f);
    return make_ray(o, d);
}

// Triangle::intersect (triangle.cuh:66-102) on a slot's precomputed edges
// (a = v0, b = v1 - v0, c = v2 - v0).  The reference divides by the
// determinant first and tests u, v and t on the quotients; here the hardware
// reciprocal (1 ulp) rejects what lies outside by more than its error, and
// only a triangle that may pass pays for the IEEE division and the reference's
// own tests.  A NaN passes every one of these comparisons on to the exact
// tests, and u > 1 is left to u + v > 1 (v is not below -1e-30).
__device__ __forceinline__ bool triangle(const float4& a, const float4& b, const float4& c, v3 o, v3 d, float tmin,
                                         float tmax, float* t_out, float* u_out, float* v_out) {
    const float EPS = 1.0e-5f;
    const v3 e1 = mk3(b.x, b.y, b.z), e2 = mk3(c.x, c.y, c.z);
    const v3 pvec = cross(d, e2);
    const float det = dot(e1, pvec);
    const v3 tvec = o - mk3(a.x, a.y, a.z);
    const float un = dot(tvec, pvec);
    const v3 q = cross(tvec, e1);
    const float vn = dot(d, q);
    const float tn = dot(e2, q);
    const float r = __builtin_amdgcn_rcpf(det);
    const float ua = r * un, va = r * vn, ta = r * tn;
    const float OUT = 1.00001f, NEG = -1.0e-30f;
    bool hit = false;
    if (!(__builtin_fabsf(det) < EPS || fminf_(fminf_(ua, va), ta) < NEG || ua + va > OUT || ta > tmax * OUT)) {
        const float inv = 1.0f / det;
        const float u = inv * un;
        const float v = inv * vn;
        const float t = inv * tn;
        hit = !(u < 0.0f || u > 1.0f || v < 0.0f || u + v > 1.0f) && t > EPS && t < tmax && t > tmin;
        *t_out = t; *u_out = u; *v_out = v;
    }
    return hit;
}

// Lane k's value (k uniform), in every lane.
__device__ __forceinline__ float lane_of(float x, int k) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), k));
}

// Where a lane's stack lives: its first LDS word, the word stride between
// entries (a power of two: the workgroup's lanes, so the lanes of a wave hit
// distinct banks) and the number of LDS entries (LDS_STACK_MIN..LDS_STACK_MAX,
// or LDS_STACK for the fixed-shape kernels); all but the pointer are uniform.
struct StackShape {
    uint32_t* lds;
    int stride;
    int depth;
};

typedef __attribute__((address_space(3))) uint32_t lds_u32;   // a pointer that is known to be LDS

// Per-lane stack: LDS part [depth][stride] + a private spill array owned by
// the caller (kept outside the traversal state so the state itself stays in
// registers).  The top is an LDS byte address moved by the stride, so a push
// or pop is one add and one LDS access; the lanes' first words lie within one
// stride, so one uniform address tells for all of them whether an entry is in
// LDS.  Entry 0 is ENTRY_IDLE: a query that pops it has ended, and no pop
// looks for an empty stack.
struct LaneStack {
    uint32_t top;       // LDS byte address of the next free entry
    uint32_t* spill;    // private array of SPILL_STACK entries
    uint32_t base;      // uniform: LDS byte address of lane 0's entry 0
    uint32_t step;      // uniform: bytes between entries
    uint32_t limit;     // uniform: LDS byte address past the LDS part
    int shift;          // uniform: log2(step)
    // entries below the address (entry 0 included); the lane's own offset is less than a step
    KD int index(uint32_t address) const { return (int)((address - base) >> shift); }
    KD int deep(uint32_t address) const { return (int)((address - limit) >> shift); }
    __device__ __forceinline__ static lds_u32* at_address(uint32_t a) { return (lds_u32*)(uintptr_t)a; }
    // A push on a full stack moves the top all the same and nothing more: the
    // caller ends the query, and the top tells of it from then on.
    KD bool overflow() const { return index(top) > STACK_TOTAL + 1; }
    __device__ __forceinline__ void push(uint32_t e) {
        if (top < limit) *at_address(top) = e;
        else if (index(top) <= STACK_TOTAL) spill[deep(top)] = e;
        top += step;
    }
    __device__ __forceinline__ uint32_t pop() {
        top -= step;
        return top < limit ? *at_address(top) : spill[deep(top)];
    }
    // the entries above entry 0: their number, and the i-th one read or
    // written in place (a parked trace's copy)
    KD int size() const { return index(top) - 1; }
    KD uint32_t address(int i) const { return top + ((uint32_t)(i - size()) << shift); }
    __device__ __forceinline__ uint32_t get(int i) const {
        const uint32_t a = address(i);
        return a < limit ? *at_address(a) : spill[deep(a)];
    }
    __device__ __forceinline__ void reset(const StackShape& sh, uint32_t* spill_) {
        // stride and depth are the same for every lane: read them as such, so
        // they stay in scalar registers wherever the traversal runs
        const uint32_t own = (uint32_t)(uintptr_t)(lds_u32*)sh.lds;
        step = 4u * (uint32_t)__builtin_amdgcn_readfirstlane(sh.stride);
        shift = __builtin_ctz(step);
        base = __builtin_amdgcn_readfirstlane(own - 4u * ((uint32_t)threadIdx.x & ((step >> 2) - 1u)));
        limit = base + (uint32_t)__builtin_amdgcn_readfirstlane(sh.depth) * step;
        spill = spill_;
        *at_address(own) = 0xFFFFFFFFu;
        top = own + step;
    }
};

// ---- entries.  A BVH2 node is represented by what the traversal needs to
// process it without loading the node itself; a NodePair holds its two
// children's boxes and entries:
//   interior BLAS node:  index of its children's NodePair
//   interior TLAS node:  TLAS_BIT | index of its children's NodePair
//   BLAS leaf:           LEAF_BIT | count << 23 | first slot   (count < 64, first + count <= 2^23)
//   larger BLAS leaf:    BIG_BIT | node index (its header is loaded)
//   TLAS leaf:           TLAS_BIT | LEAF_BIT | instance
//   nothing left:        ENTRY_IDLE (also an empty BLAS's root entry)
//   the stack's top:     ENTRY_POP (within a round only)
constexpr uint32_t LEAF_BIT = 0x40000000u;
constexpr uint32_t BIG_BIT = 0x20000000u;
constexpr uint32_t ENTRY_PAYLOAD = 0x1FFFFFFFu;
constexpr uint32_t ENTRY_IDLE = 0xFFFFFFFFu;
constexpr uint32_t ENTRY_POP = 0xFFFFFFFEu;

KD uint32_t bits_u(float f) { return __builtin_bit_cast(uint32_t, f); }

// Entry of a BLAS node given its index and header words; first_pair: the
// index of the BLAS pair 0 in the pair array (the TLAS's pairs come first).
KD uint32_t blas_entry(uint32_t idx, uint32_t a, uint32_t b, uint32_t first_pair) {
    if (b == 0u) return first_pair + (a >> 1);
    if (b < 64u && a + b <= (1u << 23)) return LEAF_BIT | (b << 23) | a;
    return BIG_BIT | idx;
}
// Entry of a TLAS node given its header words (pair layout).
KD uint32_t tlas_entry(uint32_t a, uint32_t b) {
    return a != 0u ? (TLAS_BIT | (a >> 1)) : (TLAS_BIT | LEAF_BIT | b);
}

// The pair of two sibling nodes: tlas_pair of the TLAS's pair layout,
// blas_pair of BLAS nodes 2q and 2q + 1.
KD NodePair node_pair(const Node& n0, uint32_t e0, const Node& n1, uint32_t e1) {
    NodePair p;
    for (int k = 0; k < 3; ++k) {
        p.lo0[k] = n0.lo[k]; p.hi0[k] = n0.hi[k];
        p.lo1[k] = n1.lo[k]; p.hi1[k] = n1.hi[k];
    }
    p.e0 = e0; p.e1 = e1; p.pad0 = 0u; p.pad1 = 0u;
    return p;
}
KD NodePair tlas_pair(const Node& n0, const Node& n1) {
    return node_pair(n0, tlas_entry(n0.a, n0.b), n1, tlas_entry(n1.a, n1.b));
}
KD NodePair blas_pair(const Node& n0, const Node& n1, uint32_t q, uint32_t first_pair) {
    return node_pair(n0, blas_entry(2u * q, n0.a, n0.b, first_pair), n1,
                     blas_entry(2u * q + 1u, n1.a, n1.b, first_pair));
}

// The least float above x (x itself for +inf and NaN): te < next_up(b) is
// te <= b, except that te = +inf never passes.
KD float next_up(float x) {
    const uint32_t u = bits_u(x);
    if (!(x < __builtin_inff())) return x;
    return __builtin_bit_cast(float, x == 0.0f ? 1u : ((u >> 31) ? u - 1u : u + 1u));
}

constexpr int INNER_RUN = 4;   // interior steps of a round
constexpr int WIDE_LEAF = 64;  // triangles from which the whole wave tests one lane's leaf

// One lane's query: the closest hit, any hit, or either as the lane says.
enum TravMode : int { TRAV_CLOSEST = 0, TRAV_ANY = 1, TRAV_EITHER = 2 };
template <int MODE>
struct Trav {
    Ray w, o;           // the world ray; the current level's ray
    float tmin;
    float bound;        // a hit's distance has to be below this: tmax, then the closest hit so far
    float enter;        // a box's entry distance has to be below this (TRAV_ANY: at most bound)
    int32_t slot, inst; // the hit (slot -1: none)
    float u, v;
    int32_t cur_inst;
    uint32_t cur;       // the entry to process next (ENTRY_IDLE: finished)
    bool fresh;         // counting: cur is a leaf that has not been counted
    bool lane_any;      // TRAV_EITHER: this lane's query is for any hit
    LaneStack st;

    KD bool is_any() const { return MODE == TRAV_ANY || (MODE == TRAV_EITHER && lane_any); }

    KD bool busy() const { return cur != ENTRY_IDLE; }
    KD Hit hit() const {
        Hit h;
        h.t = slot >= 0 ? bound : __builtin_inff();
        h.slot = slot; h.inst = inst; h.u = u; h.v = v;
        return h;
    }
    KD bool any() const { return slot >= 0; }
    KD void idle() { cur = ENTRY_IDLE; slot = -1; }

    // TLAS::intersect entry: empty TLAS or a miss of the root box ends the
    // query at once (tlas.cu:62-69).
    __device__ __forceinline__ void init(const SceneView& S, const Ray& ray, float t0, float t1, const StackShape& sh,
                                         uint32_t* spill) {
        w = ray; o = ray; tmin = t0; bound = t1; enter = next_up(t1);
        slot = -1; inst = -1; u = 0.0f; v = 0.0f;
        cur_inst = -1;
        cur = ENTRY_IDLE;
        fresh = true;
        st.reset(sh, spill);
        if (S.tlas_root < 0) return;
        float4 rlo, rhi;
        load_node(S.tlas_nodes, 0, &rlo, &rhi);
        float te;
        if (!slab(rlo, rhi, w, t0, t1, &te)) return;
        cur = tlas_entry(bits_u(rlo.w), bits_u(rhi.w));
    }

    // A lane's step leaves ENTRY_POP where the stack's top is next; an interior
    // TLAS node is entered with the world ray again.  (The steps below are
    // written as one-sided updates with one common pop, so that the state is
    // updated in its registers: two-sided branches made the compiler copy it
    // at every merge, about 40 moves a round.)
    __device__ __forceinline__ void pop_next() {
        bool back = false;
        if (cur == ENTRY_POP) {
            cur = st.pop();
            fresh = true;
            back = (cur & (TLAS_BIT | LEAF_BIT)) == TLAS_BIT;
        }
        if (__builtin_amdgcn_ballot_w64(back) != 0ull) {   // uniform
            o.o.x = back ? w.o.x : o.o.x; o.o.y = back ? w.o.y : o.o.y; o.o.z = back ? w.o.z : o.o.z;
            o.d.x = back ? w.d.x : o.d.x; o.d.y = back ? w.d.y : o.d.y; o.d.z = back ? w.d.z : o.d.z;
            o.inv.x = back ? w.inv.x : o.inv.x; o.inv.y = back ? w.inv.y : o.inv.y; o.inv.z = back ? w.inv.z : o.inv.z;
        }
    }

    // Interior node: both children's boxes against the current ray; the
    // nearer one is next, the farther one on the stack.
    template <bool COUNT>
    __device__ __forceinline__ void inner(const SceneView& S, TraceCounts* cnt) {
        if (!(cur & (LEAF_BIT | BIG_BIT))) {
            const float4* p = reinterpret_cast<const float4*>(S.pairs + (cur & ENTRY_PAYLOAD));
            const float4 l1 = p[0], h1 = p[1], l2 = p[2], h2 = p[3];
            if (COUNT) { if (cur & TLAS_BIT) cnt->tlas++; else cnt->interior++; }
            float c1, c2, x1, x2;
            slab_range(l1, h1, o, &c1, &x1);
            slab_range(l2, h2, o, &c2, &x2);
            const bool k1 = c1 <= x1 && x1 >= tmin && (MODE == TRAV_ANY ? c1 <= bound : c1 < enter);
            const bool k2 = c2 <= x2 && x2 >= tmin && (MODE == TRAV_ANY ? c2 <= bound : c2 < enter);
            const uint32_t e1 = bits_u(l1.w), e2 = bits_u(l2.w);
            const bool second = k2 && (!k1 || c1 > c2);
            cur = second ? e2 : e1;
            cur = (k1 || k2) ? cur : ENTRY_POP;
            fresh = true;
            if (k1 && k2) {
                st.push(second ? e1 : e2);
                if (st.top > st.limit && st.overflow()) cur = ENTRY_IDLE;
            }
        }
        pop_next();
    }

    // TLAS leaf: the instance's BLAS, with the ray in object space.
    template <bool COUNT>
    __device__ __forceinline__ void instance(const SceneView& S, TraceCounts* cnt) {
        if ((cur & (TLAS_BIT | LEAF_BIT | BIG_BIT)) == (TLAS_BIT | LEAF_BIT)) {
            if (COUNT) { cnt->tlas++; cnt->entries++; }
            cur_inst = (int32_t)(cur & ENTRY_PAYLOAD);
            const InstTrav it = S.inst_trav[cur_inst];
            o = object_ray(it, w);
            cur = it.root_entry == ENTRY_IDLE ? ENTRY_POP : it.root_entry;
            fresh = true;
        }
    }

    // BLAS leaves of the wave's nt lanes in ml: g = 64 / nt triangles of each,
    // one per lane of the wave.  Lane k tests triangle k % g of the (k / g)-th
    // of them with that lane's ray; finished lanes and lanes at other nodes
    // work along, so the tests fill the wave however few its leaves are.  The
    // hits are handed back one by one in lane order, which is slot order within
    // a leaf, under the strict comparison a lane testing alone would make: the
    // same hit, ties included.
    template <bool COUNT>
    __device__ __forceinline__ void leaves(const SceneView& S, TraceCounts* cnt, uint64_t ml, int nt) {
        const int lane = (int)__lane_id();
        const bool owner = (ml >> lane) & 1ull;
        const int g = __builtin_amdgcn_readfirstlane((int)(64.01f * __builtin_amdgcn_rcpf((float)nt)));
        const int inv = __builtin_amdgcn_readfirstlane((int)(4096.0f * __builtin_amdgcn_rcpf((float)g))) + 1;
        const int r = (lane * inv) >> 12, j = lane - r * g;   // lane / g and lane % g: exact for lane < 64, g <= 64
        // lane r of `list`: the r-th owner
        const uint32_t below = __builtin_amdgcn_mbcnt_hi((uint32_t)(ml >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)ml, 0u));
        const int place = owner ? (int)below : nt + lane - (int)below;
        const int list = __builtin_amdgcn_ds_permute(4 * place, lane);
        const int from = 4 * __builtin_amdgcn_ds_bpermute(4 * r, list);
        auto get = [from](float x) { return __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(from, __builtin_bit_cast(int, x))); };
        const uint32_t e = (uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)cur);
        const v3 ro = mk3(get(o.o.x), get(o.o.y), get(o.o.z)), rd = mk3(get(o.d.x), get(o.d.y), get(o.d.z));
        const float t0 = get(tmin), t1 = get(bound);
        const int s = (int)(e & 0x7FFFFFu) + j;
        bool hit = false;
        float t = 0.0f, hu = 0.0f, hv = 0.0f;
        if (r < nt && j < (int)((e >> 23) & 0x3Fu)) {
            const float4* p = reinterpret_cast<const float4*>(S.tris + s);
            hit = triangle(p[0], p[1], p[2], ro, rd, t0, t1, &t, &hu, &hv);
        }
        const int n = (int)((cur >> 23) & 0x3Fu);
        if (COUNT && owner) {
            if (fresh) cnt->leaf++;
            fresh = false;
            cnt->tri += (uint32_t)(n < g ? n : g);
        }
        if (owner) cur = n > g ? cur + (uint32_t)g - ((uint32_t)g << 23) : ENTRY_POP;
        for (uint64_t m = __builtin_amdgcn_ballot_w64(hit); m != 0ull; m &= m - 1ull) {   // uniform
            const int k = __builtin_ctzll(m);
            const int to = __builtin_amdgcn_readlane(from, k) >> 2;
            const float ht = lane_of(t, k);
            if (COUNT && lane == to && is_any() && slot < 0)   // as a lane alone would have stopped there
                cnt->tri -= (uint32_t)((n < g ? n : g) - 1 - __builtin_amdgcn_readlane(j, k));
            const bool mine = lane == to && ht < bound;
            slot = mine ? __builtin_amdgcn_readlane(s, k) : slot;
            bound = mine ? ht : bound;
            if (MODE != TRAV_ANY) {
                inst = mine ? cur_inst : inst;
                u = mine ? lane_of(hu, k) : u;
                v = mine ? lane_of(hv, k) : v;
                enter = mine ? ht : enter;
            }
            if (MODE != TRAV_CLOSEST) cur = mine && is_any() ? ENTRY_IDLE : cur;
        }
    }

    // A smaller leaf whose slots lie past an entry's 2^23: its header, then all
    // its triangles.
    template <bool COUNT>
    __device__ __forceinline__ void big_leaf(const SceneView& S, TraceCounts* cnt) {
        if ((cur & (TLAS_BIT | LEAF_BIT | BIG_BIT)) == BIG_BIT) {
            float4 lo, hi;
            load_node(S.blas_nodes, cur & ENTRY_PAYLOAD, &lo, &hi);
            if (COUNT) cnt->leaf++;
            const uint32_t first = bits_u(lo.w), n = bits_u(hi.w);
            for (uint32_t j = 0; j < n && !(is_any() && slot >= 0); ++j) {
                const float4* p = reinterpret_cast<const float4*>(S.tris + first + j);
                if (COUNT) cnt->tri++;
                float t, hu, hv;
                if (triangle(p[0], p[1], p[2], o.o, o.d, tmin, bound, &t, &hu, &hv)) {
                    slot = (int32_t)(first + j); inst = cur_inst; u = hu; v = hv;
                    bound = t; enter = t;
                }
            }
            cur = (is_any() && slot >= 0) ? ENTRY_IDLE : ENTRY_POP;
        }
    }

    // Lane k's leaf of WIDE_LEAF or more triangles (k uniform), 64 of them at a
    // time, one per lane of the wave.  Lanes are in slot order: the first of the
    // nearest hits is the one that a lane testing alone would keep.  The ray is
    // uniform, in scalar registers.  With each lane at its own leaf (big_leaf)
    // few lanes were at one together: 200,000 rays through leaves of 9000
    // triangles ran 9.0e9 vector instructions with 12.6 lanes at work, so 2.1e9
    // with 64.  Through leaves of 160, 890 and 21,900: 970 -> 344, 6000 -> 1190
    // and 201,200 -> 66,600 us.  Kernels that meet none are up to 1 % slower for
    // its registers (64 views 226.0 -> 227.7 ms).
    template <bool COUNT>
    __device__ __forceinline__ void wide_leaf(const SceneView& S, TraceCounts* cnt, int k) {
        const bool mine = (int)__lane_id() == k;
        float4 lo, hi;
        load_node(S.blas_nodes, (uint32_t)__builtin_amdgcn_readlane((int)cur, k) & ENTRY_PAYLOAD, &lo, &hi);
        const uint32_t first = (uint32_t)__builtin_amdgcn_readfirstlane((int)bits_u(lo.w));
        const uint32_t n = (uint32_t)__builtin_amdgcn_readfirstlane((int)bits_u(hi.w));
        const v3 ro = mk3(lane_of(o.o.x, k), lane_of(o.o.y, k), lane_of(o.o.z, k));
        const v3 rd = mk3(lane_of(o.d.x, k), lane_of(o.d.y, k), lane_of(o.d.z, k));
        const float t0 = lane_of(tmin, k);
        float t1 = lane_of(bound, k);
        const bool stop = MODE == TRAV_ANY || (MODE == TRAV_EITHER && __builtin_amdgcn_readlane((int)lane_any, k) != 0);
        if (COUNT && mine) cnt->leaf++;
        for (uint32_t i = 0; i < n; i += 64u) {
            const uint32_t s = first + i + (uint32_t)__lane_id();
            bool hit = false;
            float t = 0.0f, hu = 0.0f, hv = 0.0f;
            if (s < first + n) {
                const float4* p = reinterpret_cast<const float4*>(S.tris + s);
                hit = triangle(p[0], p[1], p[2], ro, rd, t0, t1, &t, &hu, &hv);
            }
            uint64_t m = __builtin_amdgcn_ballot_w64(hit);
            if (COUNT && mine) cnt->tri += stop && m != 0ull ? (uint32_t)__builtin_ctzll(m) + 1u : (n - i < 64u ? n - i : 64u);
            while (m != 0ull) {   // uniform
                const int q = __builtin_ctzll(m);
                t1 = lane_of(t, q);
                slot = mine ? (int32_t)(first + i) + q : slot;
                bound = mine ? t1 : bound;
                if (MODE != TRAV_ANY) {
                    inst = mine ? cur_inst : inst;
                    u = mine ? lane_of(hu, q) : u;
                    v = mine ? lane_of(hv, q) : v;
                    enter = mine ? t1 : enter;
                }
                m = __builtin_amdgcn_ballot_w64(hit && t < t1);
                if (stop) { m = 0ull; i = n - 64u; }   // n >= 64: the last pass
            }
        }
        cur = mine ? (stop && slot >= 0 ? ENTRY_IDLE : ENTRY_POP) : cur;
    }

    // One round of the wave, called with all its lanes active (finished ones
    // help with the triangles): a pass over its leaves, one over its instances,
    // then INNER_RUN interior steps.
    template <bool COUNT>
    __device__ __forceinline__ void round(const SceneView& S, TraceCounts* cnt) {
        const uint32_t kind = cur & (TLAS_BIT | LEAF_BIT | BIG_BIT);
        const uint64_t ml = __builtin_amdgcn_ballot_w64(kind == LEAF_BIT);
        if (ml != 0ull) {
            leaves<COUNT>(S, cnt, ml, __builtin_popcountll(ml));
            pop_next();
        } else if (__builtin_amdgcn_ballot_w64(kind == (TLAS_BIT | LEAF_BIT)) != 0ull) {
            instance<COUNT>(S, cnt);
            pop_next();
        } else if (__builtin_amdgcn_ballot_w64(!(cur & (LEAF_BIT | BIG_BIT))) != 0ull) {
#pragma unroll
            for (int k = 0; k < INNER_RUN; ++k) inner<COUNT>(S, cnt);
        } else {
            bool many = false;
            if (kind == BIG_BIT) {
                float4 lo, hi;
                load_node(S.blas_nodes, cur & ENTRY_PAYLOAD, &lo, &hi);
                many = bits_u(hi.w) >= (uint32_t)WIDE_LEAF;
            }
            uint64_t m = __builtin_amdgcn_ballot_w64(many);
            if (m == 0ull) big_leaf<COUNT>(S, cnt);
            for (; m != 0ull; m &= m - 1ull) wide_leaf<COUNT>(S, cnt, __builtin_ctzll(m));
            pop_next();
        }
    }

    // To the end of every lane's query (all lanes of the wave active).
    template <bool COUNT>
    __device__ __forceinline__ void run(const SceneView& S, TraceCounts* cnt) {
        while (__builtin_amdgcn_ballot_w64(busy()) != 0ull) round<COUNT>(S, cnt);
    }
};
typedef Trav<TRAV_CLOSEST> ClosestTrav;
typedef Trav<TRAV_ANY> AnyTrav;
typedef Trav<TRAV_EITHER> EitherTrav;

// XCD-aware workgroup swizzle: the dispatcher hands consecutive workgroup ids
// to the 8 XCDs round-robin; remap so each XCD owns a contiguous run of tiles
// (neighbouring tiles share BVH nodes in that XCD's L2).
KD uint32_t xcd_swizzle(uint32_t bid, uint32_t nblocks) {
    const uint32_t X = 8;
    uint32_t per = nblocks / X;
    if (per == 0 || bid >= per * X) return bid;
    return (bid % X) * per + (bid / X);
}

}  // namespace kpt
