// Closest-hit traversal as a per-lane step machine, run by persistent waves
// that refill idle lanes with new rays.
//
// A lane's next step is one of four kinds, each one 64-byte fetch plus the
// arithmetic on it: a four-wide node visit (decode and slab-test its
// quantized child boxes, order the hits by entry distance), one triangle of
// the lane's current leaf, entering an instance (its inverse transform and
// BVH) or leaving one after a hit (its model transform, for the world-space
// t).  The walk is bound by vector instruction issue, and a wave pays for a
// kind's instructions whether one of its lanes or all 64 are of that kind:
// with every kind run in every iteration the 4M-triangle room took 253
// instructions per ray (now 172), about five times what its steps are with all
// lanes busy.  So an iteration
// runs ONE kind, the one that most lanes wait for (persistent_walk), and
// the other lanes keep their state; what a lane does, and in which order,
// does not depend on it.  A hit leaf child becomes the lane's leaf range
// (the nearest child first, farther ones wait on the stack like inner
// nodes).  A lane whose ray finishes takes the next ray from its wave's
// chunk of the ray list, so the wave's SIMD lanes stay busy instead of
// idling behind the wave's longest ray.  The two levels of a scene --
// instance hierarchy (TLAS) and mesh hierarchy (BLAS) -- are walked in the
// same loop: entering an instance transforms the ray into mesh space
// (sp_RayIntersectScene, src/sp_scene.cpp:263-276) and the mesh walk
// continues on the same stack.
//
// Measured against all kinds per iteration, per pass: 1M-triangle box scene
// at 512x512 2397 -> 1757 us, 4M-triangle room at 1080p 5443 -> 4415,
// 1M-triangle room with shadow rays 3979 -> 2784, 256x256 frame 361 -> 200,
// 64x64 tile 110 -> 74; mesh rays: 2^21 on 500k triangles 664 -> 513.
//
// Stack: the top entries of each lane live in LDS (4 or 8 KB per wave);
// deeper entries spill to a global array (rare: the builder bounds
// tree depth, and a closest-hit walk holds at most three pending children
// per wide level).
#pragma once

#include "spg_internal.h"

namespace spg {

// Rays a wave takes from the shared counter with one atomic, at most (a
// short ray list is divided evenly among the waves): same-address atomics
// serialize in L2, so the mesh walk at 2^21 rays takes 744 us with 64 (and 16
// waves per CU) against 530 with 128 (and 12).  The scene walk is the same
// within 3%: box 1771 -> 1757 us, room with shadow rays 2861 -> 2784, 1080p
// room 4386 -> 4415.
constexpr uint32_t kSceneChunk = 128, kMeshChunk = 128;
// The weights of the step kinds when a wave chooses the kind to run: a lane
// that waits for a rare kind costs as much as one that waits for a node, but
// the node step is the longest (about 150 instructions against 60 to 90),
// and a rare kind that waits until it has the most lanes waits for long.
// Box at 512x512, room at 1080p and room with shadow rays, us per call: equal
// weights 2182, 5540, 3688; 1 2 2 2 2111, 5348, 3470; 1 3 3 3 2139, 5438,
// 3541; 1 2 4 6 2107, 5428, 3494; 2 3 4 5 2091, 5319, 3461; these 2104, 5384,
// 3492, so the weights have to differ but within 1.5% it does not matter how.
// Mesh rays (2^21 on 500k triangles): 1 1 554, 2 3 530, 1 3 524, 1 2 524.
constexpr int kNodeWeight = 1, kTriangleWeight = 2, kEnterWeight = 3, kFinishWeight = 4;

// Node, triangle and stack-spill arrays are reached through pointers read
// from memory (mesh and scene tables), so the compiler cannot prove them
// global and would emit flat loads, which also hold the LDS wait counter
// and serialize with the LDS stack.  These loads name the global address
// space explicitly (a native vector type, so no HIP vector constructor
// takes the address back to the generic space).
typedef float f4v __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(1))) f4v gf4v;
typedef __attribute__((address_space(1))) int gint;
typedef __attribute__((address_space(3))) int lint;

__device__ __forceinline__ float4 ld_g4(const float4 *p)
{
    f4v v = *(gf4v *)p;
    return make_float4(v.x, v.y, v.z, v.w);
}

typedef float f2v __attribute__((ext_vector_type(2)));
typedef const __attribute__((address_space(1))) f2v gf2v;
typedef const __attribute__((address_space(1))) float gf1;

__device__ __forceinline__ float2 ld_g2(const float4 *p)
{
    f2v v = *(gf2v *)p;
    return make_float2(v.x, v.y);
}

__device__ __forceinline__ float ld_g1(const float4 *p) { return *(gf1 *)p; }

__device__ __forceinline__ uint32_t d_leaf_first(int32_t r)
{
    return ((uint32_t)~r) >> 3;
}
__device__ __forceinline__ uint32_t d_leaf_count(int32_t r)
{
    return (((uint32_t)~r) & 7u) + 1u;
}

struct Hit
{
    float t, u, v;
    uint32_t prim;
};

struct SceneHit
{
    float t, u, v;
    uint32_t inst, prim;
};

struct Counts
{
    uint32_t box, tlasBox, tri, mesh;
};

template <int kShort>
struct LaneStack
{
    lint *lds;       // this wave's LDS block, entry i of lane l at lds[i*64 + l]
    gint *spill;     // entry i >= kShort at spill[(i-kShort)*stride + gl]
    uint32_t stride; // lanes in the grid
    uint32_t gl;     // this lane's index in the grid
    uint32_t lane;
    __device__ __forceinline__ void write(int i, int v)
    {
        if (i < kShort) lds[i * 64 + lane] = v;
        else spill[(size_t)(i - kShort) * stride + gl] = v;
    }
    // Entries i, i + 1, i + 2; only the first n are live (the others are
    // above the stack top, so what they hold does not matter and the LDS
    // case writes all three without a branch).
    __device__ __forceinline__ void write3(int i, int n, int v0, int v1, int v2)
    {
        if (__ballot(i + 3 > kShort) == 0ull)
        {
            lint *at = lds + i * 64 + lane;
            at[0] = v0;
            at[64] = v1;
            at[128] = v2;
        }
        else
        {
            if (n > 0) write(i, v0);
            if (n > 1) write(i + 1, v1);
            if (n > 2) write(i + 2, v2);
        }
    }
    __device__ __forceinline__ int read(int i)
    {
        int v;
        if (__ballot(i >= kShort) == 0ull) v = lds[i * 64 + lane];
        else if (i < kShort) v = lds[i * 64 + lane];
        else v = spill[(size_t)(i - kShort) * stride + gl];
        return v;
    }
};

// The instance level of one scene as a lane sees it (batched launches mix
// scenes within a wave).
struct SceneView
{
    const float4 *tlasNodes;
    const DevInstance *inst;
};

__device__ __forceinline__ SceneView scene_view(const DevScene &S)
{
    return SceneView{S.tlasNodes, S.inst};
}

struct Trav
{
    v3 o, inv;                 // ray of the current level (world, or mesh space)
    v3 ld;                     // mesh-space direction
    v3 wo, wd, winv;           // world ray
    const float4 *nodes;       // records of the current level (a mesh's: nodes,
                               // then triangles)
    float tc;                  // t cull of the current level: the best hit's
                               // bound with the slack
    Hit h;                     // best hit in the current mesh
    SceneHit out;              // best hit in the scene
    int32_t cur;               // the lane's next step: a node (>= 0), a leaf
                               // (< 0: triangles in a mesh, an instance in
                               // the instance hierarchy) or kFinishStep / kNoStep
    int sp, spBase;            // stack entries; where the mesh's begin (-1:
                               // in the instance hierarchy)
    uint32_t inst;             // the instance walked
    bool mm, mmW;              // the current level's / the world ray is finite
    bool anyHit;               // occlusion query: stop at the first instance
                               // hit with a positive world t
};

// Values of Trav::cur that are not references (node indices stay below
// 2^28).
constexpr int32_t kFinishStep = 0x7FFFFFFD;  // leave the instance with its hit
constexpr int32_t kNoStep = 0x7FFFFFFC;      // no walk: idle or complete
constexpr uint32_t kFirstStepCode = 0x7FFFFFFC;

// Moller-Trumbore on one fetched triangle record (a.xyz, e1.x) (e1.yz,
// e2.xy) (e2.z, prim, n.xy) (n.z, ...) with n = cross(e1, e2) stored
// (src/ray_intersection.cpp:156-190).  Returns whether the hit c beats
// `best`: t > 0 and smaller (src/sp_scene.cpp:189-193); equal t goes to the
// lower triangle index so the result does not depend on the visit order.
__device__ __forceinline__ bool triangle_candidate(float4 t0, float4 t1, float4 t2,
                                                   float4 t3, v3 o, v3 d,
                                                   const Hit &best, Hit &c)
{
    v3 a{t0.x, t0.y, t0.z}, e1v{t0.w, t1.x, t1.y}, e2v{t1.z, t1.w, t2.x};
    v3 n{t2.z, t2.w, t3.x};
    c.prim = __float_as_uint(t2.y);
    c.u = c.v = 0.0f;
    c.t = mt_test_n(o, d, a, e1v, e2v, n, &c.u, &c.v);
    return c.t > 0.0f && (c.t < best.t || (c.t == best.t && c.prim < best.prim));
}

__device__ __forceinline__ m34 rows3(float4 a, float4 b, float4 c)
{
    return m34{{{a.x, a.y, a.z, a.w}, {b.x, b.y, b.z, b.w}, {c.x, c.y, c.z, c.w}}};
}

// The t cull in the instance hierarchy.
__device__ __forceinline__ float world_cull(float t)
{
    return t > 0.0f ? t * kCullSlack : INFINITY;
}

// What the lanes of a step (`act`) do after it: a lane with `need` has
// nothing to descend into; it leaves a finished mesh walk (by a step of its
// own when it found a hit, at once without one), then pops; with an empty
// stack its walk is complete.  Any other lane goes on with `next`.
//
// The fetch and its arithmetic sit in branches on `act`; the state is
// written through selects after them, in straight code that every lane runs:
// written inside nested divergent branches, each value would need a second
// register at every join and be copied into it on the way.
template <bool kTwoLevel, int kShort>
__device__ __forceinline__ void trav_advance(const SceneView &sv, Trav &s,
                                             LaneStack<kShort> &st, bool act, bool need,
                                             int32_t next)
{
    need = need && act;
    bool fin = false;
    if (kTwoLevel)
    {
        const bool end = need && s.sp <= s.spBase;
        const bool hit = s.h.prim != SPG_MISS;
        fin = end && hit;
        const bool leave = end && !hit;
        const float wt = world_cull(s.out.t);
        s.o = v3{leave ? s.wo.x : s.o.x, leave ? s.wo.y : s.o.y, leave ? s.wo.z : s.o.z};
        s.inv = v3{leave ? s.winv.x : s.inv.x, leave ? s.winv.y : s.inv.y,
                   leave ? s.winv.z : s.inv.z};
        s.mm = leave ? s.mmW : s.mm;
        s.nodes = leave ? sv.tlasNodes : s.nodes;
        s.tc = leave ? wt : s.tc;
        s.spBase = leave ? -1 : s.spBase;
    }
    const bool pop = need && !fin && s.sp != 0;
    int v = 0;
    if (pop) v = st.read(s.sp - 1);
    s.sp -= pop ? 1 : 0;
    const int32_t popped = fin ? kFinishStep : pop ? v : kNoStep;
    s.cur = !act ? s.cur : need ? popped : next;
}

// The four bytes of a word as halves of value q 2^-24 (subnormal halves):
// bytes 0, 1 and bytes 2, 3.
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ h2 halves_lo(uint32_t w)
{
    return __builtin_bit_cast(h2, __builtin_amdgcn_perm(0u, w, 0x0C010C00u));
}
__device__ __forceinline__ h2 halves_hi(uint32_t w)
{
    return __builtin_bit_cast(h2, __builtin_amdgcn_perm(0u, w, 0x0C030C02u));
}

// v_min_f64 / v_max_f64 of two numbers (fmin and fmax would first quiet
// operands that cannot be NaN here).
__device__ __forceinline__ double min_f64(double a, double b)
{
    double r;
    asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ double max_f64(double a, double b)
{
    double r;
    asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

// The sort key of a missed or absent child: above every entry distance.
constexpr uint32_t kMissKey = 0x7FE00000u;

// A hit child's key: the entry distance's bits with the sign cleared
// (-0 = +0) and the two low bits replaced by the child slot, so keys are
// distinct and near-ties go to the lower slot; a missed or absent child gets
// the largest key.
__device__ __forceinline__ uint32_t child_key(int k, bool hit, float e)
{
    return hit ? ((__float_as_uint(e) & 0x7FFFFFFCu) | (uint32_t)k) : kMissKey;
}

// The child keys of a node for a ray that step_node's fast form does not
// cover (rare; the node is read again so that its words stay out of the
// registers of the common path).
__device__ __forceinline__ void slow_keys(const float4 *src, bool mm, v3 o, v3 inv, float tc,
                                          uint32_t (&key)[4])
{
    asm volatile("" : "+v"(src));
    const float4 A = ld_g4(src), B = ld_g4(src + 1), C = ld_g4(src + 2);
    const float2 D = ld_g2(src + 3);
    const uint32_t eb = __float_as_uint(A.w);
    const float sx = __uint_as_float((eb & 0xFFu) << 23);
    const float sy = __uint_as_float(((eb >> 8) & 0xFFu) << 23);
    const float sz = __uint_as_float(((eb >> 16) & 0xFFu) << 23);
    const uint32_t q[6] = {__float_as_uint(C.x), __float_as_uint(C.y), __float_as_uint(C.z),
                           __float_as_uint(C.w), __float_as_uint(D.x), __float_as_uint(D.y)};
    const int32_t ref[4] = {__float_as_int(B.x), __float_as_int(B.y), __float_as_int(B.z),
                            __float_as_int(B.w)};
    const v3 a{sx * inv.x, sy * inv.y, sz * inv.z};
    const v3 b{(A.x - o.x) * inv.x, (A.y - o.y) * inv.y, (A.z - o.z) * inv.z};
    const bool fold = mm && finite3(a) && finite3(b);
    const bool px = inv.x > 0.0f, py = inv.y > 0.0f, pz = inv.z > 0.0f;
#pragma unroll
    for (int k = 0; k < 4; ++k)
    {
        auto dq = [&](int f, float sc, float p) {
            return fmaf((float)((q[f] >> (8 * k)) & 0xFFu), sc, p);
        };
        float e;
        bool h;
        if (fold)
            // only a 2^24 overflows: the same distances, unscaled
            h = slab_hit_t(dq(px ? 0 : 3, a.x, b.x), dq(py ? 1 : 4, a.y, b.y),
                           dq(pz ? 2 : 5, a.z, b.z), dq(px ? 3 : 0, a.x, b.x),
                           dq(py ? 4 : 1, a.y, b.y), dq(pz ? 5 : 2, a.z, b.z), &e);
        else
            // a non-finite origin, inverse direction or per-axis factor (an
            // axis-parallel ray, or s inv overflowing): the reference's
            // compare-and-select form on the decoded box
            h = slab_hit(dq(0, sx, A.x), dq(1, sy, A.y), dq(2, sz, A.z), dq(3, sx, A.x),
                         dq(4, sy, A.y), dq(5, sz, A.z), o, inv, &e);
        key[k] = child_key(k, h && e <= tc && ref[k] != kEmptyChild, e);
    }
}

// One node visit: decode and slab-test the children, the nearest hit one is
// the next step and the others go to the stack.
template <bool kCount, bool kTwoLevel, int kShort>
__device__ __forceinline__ void step_node(const SceneView &sv, Trav &s,
                                          LaneStack<kShort> &st, Counts &cnt, bool act)
{
    int npush = 0;
    int32_t push0 = 0, push1 = 0, push2 = 0, next = kNoStep;
    bool none = false;
    if (act)
    {
        const float4 *src = s.nodes + 4 * (size_t)(uint32_t)s.cur;
        const float4 A = ld_g4(src), B = ld_g4(src + 1), C = ld_g4(src + 2);
        const float2 D = ld_g2(src + 3);
        const v3 o = s.o, inv = s.inv;
        const float tc = s.tc;
        // A: origin p and scale exponents; B: child references; C, D: the
        // child boxes, one field of all four children per 32-bit word.  A
        // coordinate decodes to p + q * s: q * s is exact (8-bit integer
        // times a power of two), so the FMA rounds the same sum once.
        const uint32_t eb = __float_as_uint(A.w);
        const float sx = __uint_as_float((eb & 0xFFu) << 23);
        const float sy = __uint_as_float(((eb >> 8) & 0xFFu) << 23);
        const float sz = __uint_as_float(((eb >> 16) & 0xFFu) << 23);
        const uint32_t q0 = __float_as_uint(C.x), q1 = __float_as_uint(C.y),
                       q2 = __float_as_uint(C.z), q3 = __float_as_uint(C.w),
                       q4 = __float_as_uint(D.x), q5 = __float_as_uint(D.y);
        int32_t ref[4] = {__float_as_int(B.x), __float_as_int(B.y), __float_as_int(B.z),
                          __float_as_int(B.w)};
        uint32_t key[4];
        // a plane at p + q s (q the 8-bit field) is crossed at
        // t = (p + q s - o) inv = q (s inv) + (p - o) inv: per node and axis
        // a = s inv (exact: s is a power of two) and b = (p - o) inv, then
        // one FMA per plane.  The byte q is spread into a half whose bits read
        // as the subnormal q 2^-24, so the multiply-add that widens a half
        // operand takes it without a conversion: (q 2^-24) (a 2^24) + b, the
        // same product and rounding.
        const float ax = sx * inv.x, ay = sy * inv.y, az = sz * inv.z;
        const float bx = (A.x - o.x) * inv.x, by = (A.y - o.y) * inv.y,
                    bz = (A.z - o.z) * inv.z;
        const float cx24 = ax * 16777216.0f, cy24 = ay * 16777216.0f, cz24 = az * 16777216.0f;
        // finite factors: the IEEE maximum keeps a NaN (v_maximum3; v_max3
        // would drop it), which an infinite direction gives where p - o
        // overflows, 0 times infinity
        auto mx = [](float x, float y) { return __builtin_elementwise_maximum(x, y); };
        const float big = mx(mx(mx(fabsf(cx24), fabsf(cy24)), mx(fabsf(cz24), fabsf(bx))),
                             mx(fabsf(by), fabsf(bz)));
        const bool fast = s.mm && big < INFINITY;
        // per axis the near plane is the lo field where inv > 0 (a
        // positive a makes t increase with q) and the hi field where
        // inv < 0, so choosing the fields once per node orders each
        // axis's two distances
        const bool px = inv.x > 0.0f, py = inv.y > 0.0f, pz = inv.z > 0.0f;
        const uint32_t nx = px ? q0 : q3, fx = px ? q3 : q0;
        const uint32_t ny = py ? q1 : q4, fy = py ? q4 : q1;
        const uint32_t nz = pz ? q2 : q5, fz = pz ? q5 : q2;
        {
            const h2 nx0 = halves_lo(nx), nx1 = halves_hi(nx), fx0 = halves_lo(fx),
                     fx1 = halves_hi(fx), ny0 = halves_lo(ny), ny1 = halves_hi(ny),
                     fy0 = halves_lo(fy), fy1 = halves_hi(fy), nz0 = halves_lo(nz),
                     nz1 = halves_hi(nz), fz0 = halves_lo(fz), fz1 = halves_hi(fz);
#pragma unroll
            for (int k = 0; k < 4; ++k)
            {
                const int i = k & 1;
                auto pl = [&](h2 l, h2 h, float c, float b) {
                    return fmaf((float)(k < 2 ? l[i] : h[i]), c, b);
                };
                float e;
                bool h = slab_hit_t(pl(nx0, nx1, cx24, bx), pl(ny0, ny1, cy24, by),
                                    pl(nz0, nz1, cz24, bz), pl(fx0, fx1, cx24, bx),
                                    pl(fy0, fy1, cy24, by), pl(fz0, fz1, cz24, bz), &e);
                key[k] = child_key(k, h & (e <= tc) & (ref[k] != kEmptyChild), e);
            }
        }
        if (!fast) slow_keys(src, s.mm, o, inv, tc, key);
        if (kCount)
        {
            uint32_t present = 0;
#pragma unroll
            for (int k = 0; k < 4; ++k) present += ref[k] != kEmptyChild ? 1u : 0u;
            if (!kTwoLevel || s.spBase >= 0) cnt.box += present;
            else cnt.tlasBox += present;
        }
        // sort (key, reference) pairs by key: five compare-exchanges.  A pair is
        // one 64-bit word, key above reference; as a double it is positive and
        // finite (keys stay below 0x7FF00000), so the double minimum and maximum
        // order the words as integers, subnormals included, in two operations
        // per exchange instead of a compare and four selects.
        double pr[4];
#pragma unroll
        for (int k = 0; k < 4; ++k)
            pr[k] = __longlong_as_double(
                (long long)(((uint64_t)key[k] << 32) | (uint32_t)ref[k]));
        auto cx = [&](int a, int b) {
            const double lo = min_f64(pr[a], pr[b]), hi = max_f64(pr[a], pr[b]);
            pr[a] = lo;
            pr[b] = hi;
        };
        cx(0, 1);
        cx(2, 3);
        cx(0, 2);
        cx(1, 3);
        cx(1, 2);
        auto miss = [&](int k) { return __double2hiint(pr[k]) == (int)kMissKey; };
        auto refOf = [&](int k) { return (int32_t)__double2loint(pr[k]); };
        // the nearest is next; the others wait on the stack, the nearest
        // of them on top: slot 3 at sp, slot 2 above it, slot 1 on top
        const bool v1 = !miss(1), v2 = !miss(2), v3 = !miss(3);
        npush = (v1 ? 1 : 0) + (v2 ? 1 : 0) + (v3 ? 1 : 0);
        push0 = v3 ? refOf(3) : v2 ? refOf(2) : refOf(1);
        push1 = v3 ? refOf(2) : refOf(1);
        push2 = refOf(1);
        next = refOf(0);
        none = miss(0);
    }
    if (__ballot(npush != 0) != 0ull) st.write3(s.sp, npush, push0, push1, push2);
    s.sp += npush;
    trav_advance<kTwoLevel>(sv, s, st, act, none, next);
}

// One triangle of the lane's leaf; after the last one the lane pops.
template <bool kCount, bool kTwoLevel, int kShort>
__device__ __forceinline__ void step_triangle(const SceneView &sv, Trav &s,
                                              LaneStack<kShort> &st, Counts &cnt, bool act)
{
    Hit c{0.0f, 0.0f, 0.0f, 0u};
    bool take = false;
    if (act)
    {
        const float4 *src = s.nodes + 4 * (size_t)d_leaf_first(s.cur);
        const float4 A = ld_g4(src), B = ld_g4(src + 1), C = ld_g4(src + 2);
        const float4 D = make_float4(ld_g1(src + 3), 0.0f, 0.0f, 0.0f);
        take = triangle_candidate(A, B, C, D, s.o, s.ld, s.h, c);
    }
    s.h.t = take ? c.t : s.h.t;
    s.h.u = take ? c.u : s.h.u;
    s.h.v = take ? c.v : s.h.v;
    s.h.prim = take ? c.prim : s.h.prim;
    const float ts = c.t * kCullSlack;
    s.tc = take && ts < s.tc ? ts : s.tc;
    if (kCount) cnt.tri += act ? 1u : 0u;
    // ~cur = first * 8 + (count - 1): the next triangle is first + 1,
    // count - 1, which is ~cur + 7
    trav_advance<kTwoLevel>(sv, s, st, act, d_leaf_count(s.cur) == 1u,
                            (int32_t)((uint32_t)s.cur - 7u));
}

// Entering instance (leaf): o' = M^-1 o, d' = norm(M^-1 d)
// (src/sp_scene.cpp:272-276); the mesh walk starts at its root above the
// current stack.
template <bool kCount>
__device__ __forceinline__ void step_enter(const SceneView &sv, Trav &s, Counts &cnt, bool act)
{
    if (act)
    {
        s.inst = d_leaf_first(s.cur);
        const float4 *src = reinterpret_cast<const float4 *>(sv.inst + s.inst) + 3;
        const float4 A = ld_g4(src), B = ld_g4(src + 1), C = ld_g4(src + 2), D = ld_g4(src + 3);
        const m34 I = rows3(A, B, C);
        s.o = xform_point(I, s.wo);
        s.ld = normalize(xform_vector(I, s.wd));
        s.inv = inverse(s.ld);
        s.mm = finite3(s.o) && finite3(s.inv);
        s.tc = s.out.t > 0.0f ? s.out.t * D.x * kCullSlack : INFINITY;
        s.nodes = reinterpret_cast<const float4 *>(
            ((uint64_t)__float_as_uint(D.w) << 32) | __float_as_uint(D.z));
        s.h.t = INFINITY;
        s.h.prim = SPG_MISS;
        s.spBase = s.sp;
        s.cur = 0;
        if (kCount) cnt.mesh += 1u;
    }
}

// Leaving an instance with a hit: world t = dot(M (o' + t' d') - o, d), the
// closest world hit wins (src/sp_scene.cpp:296-322), equal t goes to the
// lower instance index.
template <int kShort>
__device__ __forceinline__ void step_finish(const SceneView &sv, Trav &s,
                                            LaneStack<kShort> &st, bool act)
{
    float tw = 0.0f;
    if (act)
    {
        const float4 *src = reinterpret_cast<const float4 *>(sv.inst + s.inst);
        const float4 A = ld_g4(src), B = ld_g4(src + 1), C = ld_g4(src + 2);
        const v3 lh = s.o + s.ld * s.h.t;
        const v3 wh = xform_point(rows3(A, B, C), lh);
        tw = dot(wh - s.wo, s.wd);
    }
    // an occlusion query takes the first instance hit at a positive
    // world t (what k_resolve_shadow counts as a blocker) and stops;
    // a hit whose world t rounds to <= 0 neither stops nor blocks
    const bool closer = tw < s.out.t || s.out.t < 0.0f ||
                        (tw == s.out.t && s.inst < s.out.inst);
    const bool better = act && (s.anyHit ? tw > 0.0f : closer);
    s.out.t = better ? tw : s.out.t;
    s.out.u = better ? s.h.u : s.out.u;
    s.out.v = better ? s.h.v : s.out.v;
    s.out.inst = better ? s.inst : s.out.inst;
    s.out.prim = better ? s.h.prim : s.out.prim;
    s.h.prim = act ? SPG_MISS : s.h.prim;
    // an occlusion query that found a blocker is complete
    trav_advance<true>(sv, s, st, act, !(s.anyHit && better), kNoStep);
}

__device__ __forceinline__ void trav_begin_scene(const SceneView &sv, Trav &s, v3 o, v3 d)
{
    s.o = s.wo = o;
    s.wd = d;
    s.inv = s.winv = inverse(d);
    s.mm = s.mmW = finite3(o) && finite3(s.inv);
    s.nodes = sv.tlasNodes;
    s.tc = INFINITY;
    s.anyHit = false;
    s.out = SceneHit{-1.0f, 0.0f, 0.0f, SPG_MISS, SPG_MISS};
    s.sp = 0;
    s.spBase = -1;
    s.cur = 0;
}

__device__ __forceinline__ void trav_begin_mesh(const DevMesh &M, Trav &s, v3 o,
                                                v3 d)
{
    s.o = o;
    s.ld = d;
    s.inv = inverse(d);
    s.mm = finite3(o) && finite3(s.inv);
    s.nodes = M.nodes;
    s.tc = INFINITY;
    s.h = Hit{INFINITY, 0.0f, 0.0f, SPG_MISS};
    s.sp = 0;
    s.cur = 0;
}

// The rays of a persistent launch in chunks, handed to its waves.  A wave's
// first chunk is the one at its own position, the further ones come from the
// counter (zero on entry), so a launch whose rays fit its waves makes no
// atomic at all and in the others no wave starts by waiting for one
// (same-address atomics take 11 ns each: 56 us for 5120 waves that start
// together).
struct WorkSource
{
    uint32_t *counter;
    uint32_t waves;
    WorkChunks work;
    bool first;
    __device__ __forceinline__ WorkSource(uint32_t *c, uint32_t rays, uint32_t w,
                                          uint32_t maxChunk)
        : counter(c), waves(w), work(rays, w, maxChunk), first(true)
    {
    }
    // The wave's next chunk as rays [lo, hi); false: none left (every
    // further call says so too).  Wave-uniform.
    __device__ __forceinline__ bool next(uint32_t lane, uint32_t &lo, uint32_t &hi)
    {
        uint32_t j = blockIdx.x;
        if (!first)
        {
            uint32_t k = 0;
            if (waves < work.chunks && lane == 0) k = atomicAdd(counter, 1u);
            // wave-uniform (a scalar register), so the loop's exit is
            // uniform and the compiler keeps no per-lane copies of the
            // lane state across it
            j = waves + __builtin_amdgcn_readfirstlane(k);
        }
        first = false;
        const bool some = j < work.chunks;
        lo = some ? work.begin(j) : 0u;
        hi = some ? work.end(j) : 0u;
        return some;
    }
};

// Persistent driver: the launch's waves walk rays [0, n), refilling a wave's
// idle lanes once `refill` (1..64, wave-uniform) of them wait.  begin(ray, s)
// starts a ray and returns false if it needs no walk; store(ray, s) writes
// the result of a completed walk (at the refill that reuses its lane, so the
// stores of several rays share one pass).  Must be called by every lane of a
// one-wave block.
template <bool kCount, bool kTwoLevel, int kShort, uint32_t kChunk, class Begin,
          class Store>
__device__ __forceinline__ void persistent_walk(SceneView &sv, uint32_t n,
                                                uint32_t *counter, int *spill,
                                                uint32_t refill, Begin begin,
                                                Store store, Counts &cnt,
                                                uint32_t &rays)
{
    static_assert(kShort >= kMinShortStack, "the spill area holds every deeper entry");
    const uint32_t want = walk_waves(n), waves = want < gridDim.x ? want : gridDim.x;
    if (blockIdx.x >= waves) return;
    __shared__ int lds[kShort * 64];
    const uint32_t lane = threadIdx.x;
    LaneStack<kShort> st{(lint *)lds, (gint *)spill, gridDim.x * 64u,
                         blockIdx.x * 64u + lane, lane};
    const unsigned long long below = (1ull << lane) - 1ull;
    WorkSource work(counter, n, waves, kChunk);
    uint32_t chunkNext = 0, chunkEnd = 0;
    bool exhausted = n == 0u;
    uint32_t ray = SPG_MISS;
    // a lane that never gets a ray still runs the steps' straight code: its
    // state has to be defined (above all the stack pointer, since every lane
    // writes the slots above its own top)
    Trav s{};
    s.cur = kNoStep;
    s.spBase = -1;
    for (;;)
    {
        const unsigned long long idleMask = __ballot(s.cur == kNoStep);
        const uint32_t idle = (uint32_t)__popcll(idleMask);
        const bool more = !(exhausted && chunkNext >= chunkEnd);
        if (idle == 64u || (idle >= refill && more))
        {
            if (s.cur == kNoStep && ray != SPG_MISS)
            {
                store(ray, s);
                ray = SPG_MISS;
                rays++;
            }
            if (!more) break;  // every lane is idle
            if (chunkNext >= chunkEnd) exhausted = !work.next(lane, chunkNext, chunkEnd);
            const uint32_t avail = chunkEnd - chunkNext;
            const uint32_t rank = (uint32_t)__popcll(idleMask & below);
            if (s.cur == kNoStep && rank < avail)
            {
                ray = chunkNext + rank;
                if (!begin(ray, s)) s.cur = kNoStep;
            }
            chunkNext += idle < avail ? idle : avail;
        }
        // The kind of step this iteration runs: the lanes of each kind are
        // counted and the largest weighted count wins; the other lanes wait.
        const bool isNode = (uint32_t)s.cur < kFirstStepCode;
        const unsigned long long mNode = __ballot(isNode);
        const unsigned long long mLeaf = __ballot(s.cur < 0);
        if (kTwoLevel)
        {
            const unsigned long long mIn = __ballot(s.spBase >= 0);
            const unsigned long long mFin = __ballot(s.cur == kFinishStep);
            const int wNode = __popcll(mNode) * kNodeWeight,
                      wTri = __popcll(mLeaf & mIn) * kTriangleWeight,
                      wEnter = __popcll(mLeaf & ~mIn) * kEnterWeight,
                      wFin = __popcll(mFin) * kFinishWeight;
            if (wNode >= wTri && wNode >= wEnter && wNode >= wFin)
                step_node<kCount, true>(sv, s, st, cnt, isNode);
            else if (wTri >= wEnter && wTri >= wFin)
                step_triangle<kCount, true>(sv, s, st, cnt, s.cur < 0 && s.spBase >= 0);
            else if (wEnter >= wFin)
                step_enter<kCount>(sv, s, cnt, s.cur < 0 && s.spBase < 0);
            else
                step_finish(sv, s, st, s.cur == kFinishStep);
        }
        else
        {
            if (__popcll(mNode) * kNodeWeight >= __popcll(mLeaf) * kTriangleWeight)
                step_node<kCount, false>(sv, s, st, cnt, isNode);
            else
                step_triangle<kCount, false>(sv, s, st, cnt, s.cur < 0);
        }
    }
}

}  // namespace spg
