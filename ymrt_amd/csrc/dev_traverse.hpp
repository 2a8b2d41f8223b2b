// dev_traverse.hpp -- two-level wide-BVH traversal for gfx950.
//
// Restates the queries of src/ShadingUtilities.cuh:
//   closest hit  TraceRay            (310-431) incl. the +-2 ulp nearby-hit list
//   any hit      BVHTraverseShadow   (563-635), boundary instances skipped
//   boundaries   TraceVolume         (434-559), only boundary instances
// over a 4-wide tree (one 128-B node per visit, children visited nearest
// first, far children pushed on a per-lane stack in LDS laid out
// [slot][lane] so the 64 lanes of a wave hit 64 distinct banks).  The
// triangle test is the reference's watertight shear test
// (src/ShadingUtilities.cuh:54-134) evaluated in the same operation order with
// contraction off, so t and barycentrics are the reference's floats.  Box
// tests use (b - o) * (1/d) like src/BoundingBox.h:119-155 and scale every
// far distance by 1 + 2*gamma(3), which keeps them conservative.
#pragma once

#include <cstddef>

#include "dev_scene.hpp"

namespace ym {

enum : int { kModeAll = 0, kModeSkipBoundary = 1, kModeBoundaryOnly = 2 };
constexpr int kNearbyCap = 4;

struct RayPre {
    f3 o, d, inv;
    int kx, ky, kz;
    float sx, sy, sz;
    // visit_node: byte offset of the near planes within an axis' (lo, hi)
    // pair, and whether a reciprocal is infinite (a zero direction component)
    uint32_t near_x, near_y, near_z;
    bool flat;

    // what the reciprocals alone decide
    YM_HD void set_planes()
    {
        near_x = (f2u(inv.x) >> 27) & 16u;
        near_y = (f2u(inv.y) >> 27) & 16u;
        near_z = (f2u(inv.z) >> 27) & 16u;
        flat = fmaxf(fmaxf(fabsf(inv.x), fabsf(inv.y)), fabsf(inv.z)) == INFINITY;
    }
};

YM_HD RayPre make_pre(f3 o, f3 d)
{
    RayPre r;
    r.o = o;
    r.d = d;
    r.inv = f3{1.f / d.x, 1.f / d.y, 1.f / d.z};
    f3 a = abs3(d);
    int kz = 0;
    if (a.y > comp(a, kz)) kz = 1;
    if (a.z > comp(a, kz)) kz = 2;
    int kx = kz + 1;
    if (kx == 3) kx = 0;
    int ky = kx + 1;
    if (ky == 3) ky = 0;
    r.kx = kx;
    r.ky = ky;
    r.kz = kz;
    float dx = comp(d, kx), dy = comp(d, ky), dz = comp(d, kz);
    r.sx = -dx / dz;
    r.sy = -dy / dz;
    r.sz = comp(r.inv, kz);  // 1 / dz
    r.set_planes();
    return r;
}

struct TriHit {
    float t, e0, e1, e2, inv;
};

// Returns true when the sheared plane crossing lies inside the triangle and
// the denominator is non-zero; t is not range-checked.
YM_HD bool tri_test(const RayPre &r, f3 q0, f3 q1, f3 q2, TriHit &h)
{
    f3 p0 = q0 - r.o, p1 = q1 - r.o, p2 = q2 - r.o;
    f3 a{comp(p0, r.kx), comp(p0, r.ky), comp(p0, r.kz)};
    f3 b{comp(p1, r.kx), comp(p1, r.ky), comp(p1, r.kz)};
    f3 c{comp(p2, r.kx), comp(p2, r.ky), comp(p2, r.kz)};
    a.x += r.sx * a.z;
    a.y += r.sy * a.z;
    b.x += r.sx * b.z;
    b.y += r.sy * b.z;
    c.x += r.sx * c.z;
    c.y += r.sy * c.z;
    float e0 = b.x * c.y - b.y * c.x;
    float e1 = c.x * a.y - c.y * a.x;
    float e2 = a.x * b.y - a.y * b.x;
    if ((e0 < 0 || e1 < 0 || e2 < 0) && (e0 > 0 || e1 > 0 || e2 > 0)) return false;
    float den = e0 + e1 + e2;
    if (den == 0) return false;
    a.z *= r.sz;
    b.z *= r.sz;
    c.z *= r.sz;
    float inv = 1.0f / den;
    float t = e0 * a.z + e1 * b.z + e2 * c.z;
    t *= inv;
    h.t = t;
    h.e0 = e0;
    h.e1 = e1;
    h.e2 = e2;
    h.inv = inv;
    return true;
}

YM_HD bool tri_back(f3 q0, f3 q1, f3 q2, f3 d)
{
    f3 gn = normalize(cross(q1 - q0, q2 - q0));
    return dot(gn, d) > 0.0f;
}

// IntersectSphereObject (src/ShadingUtilities.cuh:219-275) in object space.
// The reference divides the roots by 2.0 * a in double precision and rounds
// to float; for a quotient of two floats that equals the correctly rounded
// float quotient (53 >= 2 * 24 + 2 bits), which is what float division gives
// here (2a is exact).  ex_* describe the first root at or beyond tmin whether
// or not it is accepted (the nearby-hit bookkeeping needs it); on acceptance
// t, the hit point on the sphere and the back-face flag are returned.
struct SphereTest {
    bool ex_hit;
    float ex_t;
    int ex_back;
    float t;
    f3 p;
    int back;
};

YM_HD bool sphere_test(f3 o, f3 d, float radius, float tmin, float tmax, SphereTest &r)
{
    r.ex_hit = false;
    const float a = d.x * d.x + d.y * d.y + d.z * d.z;
    const float b = 2.0f * (d.x * o.x + d.y * o.y + d.z * o.z);
    const float c = o.x * o.x + o.y * o.y + o.z * o.z - radius * radius;
    const float disc = b * b - 4.0f * a * c;
    if (disc < 0) return false;
    const float sq = sqrtf(disc);
    const float t1 = (-b - sq) / (2.0f * a);
    const float t2 = (-b + sq) / (2.0f * a);
    r.ex_hit = true;
    r.ex_t = t1 >= tmin ? t1 : t2;
    r.ex_back = dot(d, normalize(o + d * r.ex_t)) > 0.0f;
    if (t1 > tmax || t2 < tmin) return false;
    float t = t1;
    if (t < tmin) {
        t = t2;
        if (t > tmax) return false;
    }
    f3 po = o + d * t;
    const float dist = length(po);
    po = dist > kFloatEpsilon ? (po * radius) / dist : s3(0.0f);
    r.t = t;
    r.p = po;
    r.back = dot(d, po / radius) > 0.0f;
    return true;
}

// Length of column c of an affine map's linear part: the scale an instance
// applies along object axis c.
YM_HD float sphere_axis_scale(const Affine &m, int c)
{
    return sqrtf(m.r[c] * m.r[c] + m.r[4 + c] * m.r[4 + c] + m.r[8 + c] * m.r[8 + c]);
}

// FetchGeometryNormal (src/ShadingUtilities.cuh:878-951): world position with
// its rounding-error bound and the normalised geometric normal of a hit.  For
// a sphere (b0, b1, b2) is the object-space hit point.
YM_HD void hit_geometry(const DevScene &sc, uint32_t inst, uint32_t tri, float b0, float b1, float b2, f3 &p,
                        f3 &perr, f3 &ng)
{
    const DevInstance &in = sc.instances[inst];
    if (in.flags & kInstSphere) {
        const float radius = gmax(in.radius, kFloatEpsilon);
        p = f3{b0, b1, b2};
        perr = error_gamma(5) * abs3(p);
        ng = p / radius;
    } else {
        const ShadeTri &st = sc.shade[in.shade_base + tri];
        const f3 p0{st.p[0], st.p[1], st.p[2]}, p1{st.p[3], st.p[4], st.p[5]}, p2{st.p[6], st.p[7], st.p[8]};
        const float xs = fabsf(p0.x * b0) + fabsf(p1.x * b1) + fabsf(p2.x * b2);
        const float ys = fabsf(p0.y * b0) + fabsf(p1.y * b1) + fabsf(p2.y * b2);
        const float zs = fabsf(p0.z * b0) + fabsf(p1.z * b1) + fabsf(p2.z * b2);
        p = p0 * b0 + p1 * b1 + p2 * b2;
        perr = error_gamma(7) * f3{xs, ys, zs};
        ng = cross(p1 - p0, p2 - p0);
    }
    p = xf_position(in.o2w, p, &perr);
    ng = normalize(xf_transpose_vector(in.w2o, ng));
}

struct Query {
    f3 o, d;
    float tmin, tmax;
    uint32_t last_inst, last_tri;
};

struct Hit {
    float t;
    uint32_t inst, tri;
    float b0, b1, b2;
    int back;  // spheres; a triangle's comes from resolve_backs
};

// Whether the ray (world direction d) meets triangle tri of instance inst
// from behind.
YM_HD int tri_hit_back(const DevScene &sc, uint32_t inst, uint32_t tri, f3 d)
{
    const DevInstance &in = sc.instances[inst];
    const ShadeTri &st = sc.shade[in.shade_base + tri];
    return tri_back(f3{st.p[0], st.p[1], st.p[2]}, f3{st.p[3], st.p[4], st.p[5]}, f3{st.p[6], st.p[7], st.p[8]},
                    xf_dir(in.w2o, d));
}

// Per-lane scratch for one traversal: the stack and the nearby list, in LDS
// laid out [slot][lane].  With kWindow > 0 only the top kWindow stack entries
// live in LDS (a ring indexed by depth); an entry pushed deeper than that
// evicts the entry kWindow below it to a global spill area laid out
// [depth - kWindow][thread], and popping restores it.  Most traversals never
// leave the window, so the spill area costs nothing but its allocation while
// the small window lets more waves share a CU's LDS.
//
// With kPreSlots, the world-space ray setup (reciprocal direction, shear
// constants and axis) is parked in LDS [kPreSlots][kBlock] when a traversal
// enters an instance and read back when it leaves, instead of being
// recomputed with five divisions.
//
// With kDeep > 0 the deeper entries go to a private array of kDeep instead of
// the spill area (for kernels that own no memory).  The kernel declares the
// array beside this struct: an array indexed at run time inside it would keep
// the whole struct in private memory, and every step would load its pointers
// and the lane from there.
constexpr int kPreSlots = 7;
template <int kBlock, int kWindow = 0, bool kPreLds = false, int kDeep = 0>
struct LaneScratch {
    static constexpr int kLanes = kBlock;
    static constexpr bool kParkPre = kPreLds;
    uint32_t *stack;        // [kWindow or kStack][kBlock]
    uint32_t *nb_prim;      // [kNearbyCap][kBlock]
    float *nb_t;
    int *nb_back;           // during a traversal the crossing's code (Traversal::ex_code), after
                            // resolve_backs the side
    int lane;
    uint32_t *spill;        // global [kMaxSpill][spill_stride], unused when kWindow == 0
    uint32_t spill_stride, spill_index;
    float *pre_park = nullptr;  // LDS [kPreSlots][kBlock] when kPreLds
    uint32_t *deep = nullptr;   // private [kDeep]

    YM_HD void park_pre(const RayPre &r)
    {
        float *q = pre_park + lane;
        q[0 * kBlock] = r.inv.x;
        q[1 * kBlock] = r.inv.y;
        q[2 * kBlock] = r.inv.z;
        q[3 * kBlock] = r.sx;
        q[4 * kBlock] = r.sy;
        q[5 * kBlock] = r.sz;
        q[6 * kBlock] = __builtin_bit_cast(float, r.kz);
    }
    // the parked setup of the ray (o, d)
    YM_HD RayPre unpark_pre(f3 o, f3 d) const
    {
        const float *q = pre_park + lane;
        RayPre r;
        r.o = o;
        r.d = d;
        r.inv = f3{q[0 * kBlock], q[1 * kBlock], q[2 * kBlock]};
        r.sx = q[3 * kBlock];
        r.sy = q[4 * kBlock];
        r.sz = q[5 * kBlock];
        r.kz = __builtin_bit_cast(int, q[6 * kBlock]);
        r.kx = r.kz + 1 == 3 ? 0 : r.kz + 1;
        r.ky = r.kx + 1 == 3 ? 0 : r.kx + 1;
        r.set_planes();
        return r;
    }

    static constexpr int kWindowSize = kWindow;
    YM_HD int nbi(int i) const { return i * kBlock + lane; }
    // Three entries at depths sp, sp+1, sp+2 with no spill bookkeeping: only
    // for sp + 3 <= kWindow (or the full stack when kWindow == 0), where those
    // depths are free slots of their own.
    YM_HD void put3(int sp, uint32_t a, uint32_t b, uint32_t c)
    {
        stack[sp * kBlock + lane] = a;
        stack[(sp + 1) * kBlock + lane] = b;
        stack[(sp + 2) * kBlock + lane] = c;
    }
    YM_HD void push(int sp, uint32_t v)
    {
        if constexpr (kWindow == 0) {
            stack[sp * kBlock + lane] = v;
        } else {
            static_assert((kWindow & (kWindow - 1)) == 0, "window must be a power of two");
            const int w = (sp & (kWindow - 1)) * kBlock + lane;
            if (sp >= kWindow) {
                if constexpr (kDeep > 0) deep[sp - kWindow] = stack[w];
                else gstore(spill + (size_t)(sp - kWindow) * spill_stride + spill_index, stack[w]);
            }
            stack[w] = v;
        }
    }
    // sp is the depth of the entry being popped (already decremented)
    YM_HD uint32_t pop(int sp)
    {
        if constexpr (kWindow == 0) {
            return stack[sp * kBlock + lane];
        } else {
            const int w = (sp & (kWindow - 1)) * kBlock + lane;
            const uint32_t v = stack[w];
            if (sp >= kWindow) {
                if constexpr (kDeep > 0) stack[w] = deep[sp - kWindow];
                else stack[w] = gload(spill + (size_t)(sp - kWindow) * spill_stride + spill_index);
            }
            return v;
        }
    }
};

// What the steps of a traversal read, apart from its start and results.  A
// kernel that reads its scene from device memory copies it first: a step
// would otherwise reload the pointers, which its own stores might change as
// far as the compiler can tell, before each of its loads (interior, 64 spp:
// 792 -> 780 ms).
struct TravScene {
    const WNode *nodes;
    const float4 *tris;
    const DevInstance *instances;
    YM_HD explicit TravScene(const DevScene &sc) : nodes(sc.nodes), tris(sc.tris), instances(sc.instances) {}
};

struct TraceCounters {
    uint32_t nodes, tris;
};

// compare-exchange as selects (no branch, no exec-mask changes)
#define YM_SORT2(ka, va, kb, vb)                      \
    do {                                              \
        const bool sw_ = kb < ka;                     \
        const float lo_ = sw_ ? kb : ka;              \
        const float hi_ = sw_ ? ka : kb;              \
        const uint32_t vlo_ = sw_ ? vb : va;          \
        const uint32_t vhi_ = sw_ ? va : vb;          \
        ka = lo_;                                     \
        kb = hi_;                                     \
        va = vlo_;                                    \
        vb = vhi_;                                    \
    } while (0)

// Resumable traversal: init() then step() until it returns something other
// than kTravContinue.  One step visits one wide node, one instance leaf (an
// instance entry or a sphere) or one triangle leaf, then pops the
// next entry, so a caller can interleave rays (a lane that finishes can
// start another ray while the rest of its wave traverses).
// kSphere: the scene has sphere instances (their test is compiled in only
// then; it costs registers in the traversal loop).
constexpr int kTravContinue = 0, kTravHit = 1, kTravMiss = 2, kTravOverflow = -1;

// Which side of a triangle a ray meets takes a normalised normal (about 70
// instructions), and a traversal with the nearby list would need it for every
// triangle the ray crosses, in steps where few lanes of the wave are at a
// leaf.  A traversal keeps the triangle's id instead, and resolve_backs works
// out the sides of its results once, when many lanes have one.
//
// The state holds no flags where a value says the same (hit.inst, cur_inst,
// ex_t): a per-lane flag is an exec-wide mask in two scalar registers that
// every join of divergent paths merges (38 spilled scalar registers in the
// closest-hit kernel with five flags, 1 without).
template <int kMode, bool kAny, bool kNearby, bool kCount, bool kSphere, int kStack>
struct Traversal {
    Query q;
    RayPre pre;
    Hit hit;                  // hit.inst kEmpty: nothing hit so far
    float tbest;
    uint32_t node, cur_inst;  // cur_inst: the instance the ray has entered, or kEmpty
    int sp, nb_count;
    // nearby list: the instance whose crossings are being collected, entered
    // or linked (kEmpty: none), its nearest crossing, hit or not, and the side
    // code of its last tested one.  A linked mesh's subtree is traversed in
    // one piece like an entered one, so its crossings end where another
    // instance's begin.
    uint32_t near_inst;
    float ex_t;
    int ex_code;
    float tub, tlb;

    YM_HD bool in_blas() const { return cur_inst != kEmpty; }
    // side of a crossing, until resolve_backs: a triangle's id, or a sphere's
    // side itself under the leaf bit
    YM_HD static int sphere_code(int back) { return (int)(kLeafBit | (uint32_t)back); }
    YM_HD int hit_code() const { return kSphere && hit.tri == kEmpty ? sphere_code(hit.back) : (int)hit.tri; }

    YM_HD int init(const DevScene &sc, const Query &query)
    {
        const uint32_t root = kMode == kModeAll ? sc.tlas_root
                              : kMode == kModeSkipBoundary ? sc.tlas_root_solid
                                                           : sc.tlas_root_boundary;
        q = query;
        hit.inst = kEmpty;
        nb_count = 0;
        if (sc.instance_count == 0 || root == kSentinel) return kTravMiss;
        pre = make_pre(q.o, q.d);
        tbest = q.tmax;
        cur_inst = kEmpty;
        near_inst = kEmpty;
        ex_t = INFINITY;
        ex_code = 0;
        tub = 0.0f;
        tlb = 0.0f;
        sp = 0;
        node = root;
        return kTravContinue;
    }

    // Starts collecting the crossings of instance `inst` (kEmpty: of none)
    // and settles those of the one before: the nearby-list update at the end
    // of an instance (TraceRay's per-instance block,
    // src/ShadingUtilities.cuh:357-393).
    template <typename LS>
    YM_HD void nearby_open(LS &ls, uint32_t inst)
    {
        if (near_inst == kEmpty) {
        } else if (hit.inst == near_inst) {
            tub = next_float_up(next_float_up(tbest));
            tlb = next_float_down(next_float_down(tbest));
            int w = 0;
            for (int i = 0; i < nb_count; ++i) {
                const float ti = ls.nb_t[ls.nbi(i)];
                if (ti > tlb && ti < tub) {
                    ls.nb_t[ls.nbi(w)] = ti;
                    ls.nb_prim[ls.nbi(w)] = ls.nb_prim[ls.nbi(i)];
                    ls.nb_back[ls.nbi(w)] = ls.nb_back[ls.nbi(i)];
                    ++w;
                }
            }
            nb_count = w;
            if (nb_count < kNearbyCap) {
                ls.nb_prim[ls.nbi(nb_count)] = near_inst;
                ls.nb_t[ls.nbi(nb_count)] = tbest;
                ls.nb_back[ls.nbi(nb_count)] = hit_code();
                ++nb_count;
            }
        } else if (hit.inst != kEmpty && ex_t > tlb && ex_t < tub) {
            if (nb_count < kNearbyCap) {
                ls.nb_prim[ls.nbi(nb_count)] = near_inst;
                ls.nb_t[ls.nbi(nb_count)] = ex_t;
                ls.nb_back[ls.nbi(nb_count)] = ex_code;
                ++nb_count;
            }
        }
        near_inst = inst;
        ex_t = INFINITY;
    }

    // The sides of the hit and of the nearby list's entries, once the
    // traversal has ended with a hit.
    template <typename LS>
    YM_HD void resolve_backs(const DevScene &sc, LS &ls)
    {
        if (kNearby) nearby_open(ls, kEmpty);
        const bool sphere = kSphere && hit.tri == kEmpty;
        if (!sphere) hit.back = tri_hit_back(sc, hit.inst, hit.tri, q.d);
        if (kNearby) {
            for (int i = 0; i < nb_count; ++i) {
                const uint32_t inst = ls.nb_prim[ls.nbi(i)];
                const int code = ls.nb_back[ls.nbi(i)];
                int back = hit.back;
                if (inst != hit.inst)
                    back = kSphere && (code & (int)kLeafBit) ? code & 1 : tri_hit_back(sc, inst, (uint32_t)code, q.d);
                ls.nb_back[ls.nbi(i)] = back;
            }
        }
    }

    // leaving an instance: back to world space
    template <typename LS>
    YM_HD void leave_instance(LS &ls)
    {
        if constexpr (LS::kParkPre)
            pre = ls.unpark_pre(q.o, q.d);
        else
            pre = make_pre(q.o, q.d);
        if (kNearby) nearby_open(ls, kEmpty);
        cur_inst = kEmpty;
    }

    // Pops the next entry.  kThrough: a sentinel is handled on the spot
    // (leave the instance, pop again); otherwise it is left in node for the
    // next step.
    template <bool kThrough, typename LS>
    YM_HD int pop(LS &ls)
    {
        for (;;) {
            if (sp == 0) return hit.inst != kEmpty ? kTravHit : kTravMiss;
            node = ls.pop(--sp);
            if (!kThrough || node != kSentinel) return kTravContinue;
            leave_instance(ls);
        }
    }

    // One wide-node visit (node is an inner node): pushes the far children
    // that are hit and moves to the nearest, or pops.  Without kThrough it
    // never changes the ray setup, so a loop of visits keeps it in place.
    // The loads follow the ray's signs: each axis' near planes come from its
    // lo or hi half, so a slab test needs no minimum and maximum per axis, and
    // an empty child (bounds +inf, -inf) misses by itself.  A ray with an
    // infinite reciprocal (a zero direction component) lying in a box face
    // has 0 * inf there; for those lanes both products of the axis go through
    // minimum and maximum, which rejects the box unless it is flat.  Traversal
    // is bound by instruction issue: 20 instructions per child instead of 32,
    // with the deferred sides and the flags taken out, took the closest-hit
    // kernel of the interior at 1080p and 1 spp from 1088 to 890 us per pass,
    // the shadow kernel from 556 to 510, and the 64-spp frame from 950 to 879 ms.
    template <bool kThrough, typename SC, typename LS>
    YM_HD int visit_node(const SC &sc, LS &ls, TraceCounters &cnt)
    {
        {
            const char *n = reinterpret_cast<const char *>(sc.nodes + node);
            const char *nx = n + pre.near_x, *ny = n + pre.near_y, *nz = n + pre.near_z;
            const char *fx = n - pre.near_x, *fy = n - pre.near_y, *fz = n - pre.near_z;
            const float4 ax = gload(reinterpret_cast<const float4 *>(nx + offsetof(WNode, lo_x)));
            const float4 bx = gload(reinterpret_cast<const float4 *>(fx + offsetof(WNode, hi_x)));
            const float4 ay = gload(reinterpret_cast<const float4 *>(ny + offsetof(WNode, lo_y)));
            const float4 by = gload(reinterpret_cast<const float4 *>(fy + offsetof(WNode, hi_y)));
            const float4 az = gload(reinterpret_cast<const float4 *>(nz + offsetof(WNode, lo_z)));
            const float4 bz = gload(reinterpret_cast<const float4 *>(fz + offsetof(WNode, hi_z)));
            const uint4 ch = gload(reinterpret_cast<const uint4 *>(n + offsetof(WNode, child)));
            if (kCount) cnt.nodes++;
            constexpr float kRobust = 1.0f + 2.0f * error_gamma(3);
            float k0, k1, k2, k3;
#define YM_SLAB(K, AX, BX, AY, BY, AZ, BZ)                                                        \
    {                                                                                             \
        const float x0 = (AX - pre.o.x) * pre.inv.x, x1 = (BX - pre.o.x) * pre.inv.x;             \
        const float y0 = (AY - pre.o.y) * pre.inv.y, y1 = (BY - pre.o.y) * pre.inv.y;             \
        const float z0 = (AZ - pre.o.z) * pre.inv.z, z1 = (BZ - pre.o.z) * pre.inv.z;             \
        const float tn = fmaxf(fmaxf(x0, y0), z0);                                                \
        const float tf = fminf(fminf(x1, y1), z1) * kRobust;                                      \
        const float t0 = fmaxf(tn, 0.0f);                                                         \
        const bool h = (tf > t0) & (tn <= tbest);                                                 \
        K = h ? t0 : INFINITY;                                                                    \
    }
#define YM_SLAB_FLAT(K, AX, BX, AY, BY, AZ, BZ, C)                                                \
    {                                                                                             \
        const float x0 = (AX - pre.o.x) * pre.inv.x, x1 = (BX - pre.o.x) * pre.inv.x;             \
        const float y0 = (AY - pre.o.y) * pre.inv.y, y1 = (BY - pre.o.y) * pre.inv.y;             \
        const float z0 = (AZ - pre.o.z) * pre.inv.z, z1 = (BZ - pre.o.z) * pre.inv.z;             \
        const float tn = fmaxf(fmaxf(fminf(x0, x1), fminf(y0, y1)), fminf(z0, z1));               \
        const float tf = fminf(fminf(fmaxf(x0, x1), fmaxf(y0, y1)), fmaxf(z0, z1)) * kRobust;     \
        const float t0 = fmaxf(tn, 0.0f);                                                         \
        const bool h = (C != kSentinel) & (tf > t0) & (tn <= tbest);                              \
        K = h ? t0 : INFINITY;                                                                    \
    }
            if (pre.flat) {
                YM_SLAB_FLAT(k0, ax.x, bx.x, ay.x, by.x, az.x, bz.x, ch.x)
                YM_SLAB_FLAT(k1, ax.y, bx.y, ay.y, by.y, az.y, bz.y, ch.y)
                YM_SLAB_FLAT(k2, ax.z, bx.z, ay.z, by.z, az.z, bz.z, ch.z)
                YM_SLAB_FLAT(k3, ax.w, bx.w, ay.w, by.w, az.w, bz.w, ch.w)
            } else {
                YM_SLAB(k0, ax.x, bx.x, ay.x, by.x, az.x, bz.x)
                YM_SLAB(k1, ax.y, bx.y, ay.y, by.y, az.y, bz.y)
                YM_SLAB(k2, ax.z, bx.z, ay.z, by.z, az.z, bz.z)
                YM_SLAB(k3, ax.w, bx.w, ay.w, by.w, az.w, bz.w)
            }
#undef YM_SLAB
#undef YM_SLAB_FLAT
            uint32_t v0 = ch.x, v1 = ch.y, v2 = ch.z, v3 = ch.w;
            YM_SORT2(k0, v0, k1, v1);
            YM_SORT2(k2, v2, k3, v3);
            YM_SORT2(k0, v0, k2, v2);
            YM_SORT2(k1, v1, k3, v3);
            YM_SORT2(k1, v1, k2, v2);
            if (k0 != INFINITY) {
                const int need = (k1 != INFINITY) + (k2 != INFINITY) + (k3 != INFINITY);
                constexpr int kFast = LS::kWindowSize > 0 ? LS::kWindowSize : kStack;
                if (sp + 3 <= kFast) {
                    // missed children sort last: the hit ones go far to near,
                    // the slots past them are written but stay above the top
                    const uint32_t s0 = need == 3 ? v3 : (need == 2 ? v2 : v1);
                    const uint32_t s1 = need == 3 ? v2 : v1;
                    ls.put3(sp, s0, s1, v1);
                    sp += need;
                } else {
                    if (sp + need > kStack) return kTravOverflow;
                    if (k3 != INFINITY) ls.push(sp++, v3);
                    if (k2 != INFINITY) ls.push(sp++, v2);
                    if (k1 != INFINITY) ls.push(sp++, v1);
                }
                node = v0;
                return kTravContinue;
            }
        }
        return pop<kThrough>(ls);
    }

    template <typename SC, typename LS>
    YM_HD int step(const SC &sc, LS &ls, TraceCounters &cnt)
    {
        if (node == kSentinel) {
            leave_instance(ls);
            return pop<true>(ls);
        }
        if (!(node & kLeafBit)) {
            return visit_node<true>(sc, ls, cnt);
        } else if (leaf_is_instance(node)) {
            // top-level leaf: an instance to enter
            const uint32_t ii = leaf_first(node);
            const DevInstance in = gload(sc.instances + ii);
            bool take = true;
            if (kMode == kModeSkipBoundary) take = !(in.flags & kInstBoundary);
            if (kMode == kModeBoundaryOnly) take = (in.flags & kInstBoundary) != 0;
            if (kNearby && take) nearby_open(ls, ii);
            if (kSphere && take && (in.flags & kInstSphere)) {
                SphereTest st;
                const bool acc = sphere_test(xf_point(in.w2o, q.o), xf_dir(in.w2o, q.d), in.radius, q.tmin, tbest, st);
                if (kCount) cnt.tris++;
                if (acc) {
                    tbest = st.t;
                    hit.t = st.t;
                    hit.inst = ii;
                    hit.tri = kEmpty;
                    if (!kAny) {
                        hit.b0 = st.p.x;
                        hit.b1 = st.p.y;
                        hit.b2 = st.p.z;
                        hit.back = st.back;
                    }
                    if (kAny) return kTravHit;
                }
                if (kNearby) {
                    ex_t = st.ex_hit ? st.ex_t : INFINITY;
                    ex_code = sphere_code(st.ex_back);
                    nearby_open(ls, kEmpty);
                }
            } else if (take) {
                if (sp + 1 > kStack) return kTravOverflow;
                ls.push(sp++, kSentinel);
                if constexpr (LS::kParkPre) ls.park_pre(pre);
                pre = make_pre(xf_point(in.w2o, q.o), xf_dir(in.w2o, q.d));
                cur_inst = ii;
                node = in.blas_root;
                return kTravContinue;
            }
        } else {
            const uint32_t first = leaf_first(node), count = leaf_count(node);
            for (uint32_t k = 0; k < count; ++k) {
                const float4 *tp = sc.tris + 3u * (first + k);
                const float4 w0 = gload(tp), w1 = gload(tp + 1), w2 = gload(tp + 2);
                const uint32_t tri = f2u(w0.w);
                const uint32_t inst = in_blas() ? cur_inst : f2u(w1.w);
                if (kNearby && inst != near_inst) nearby_open(ls, inst);
                if (kCount) cnt.tris++;
                const f3 q0{w0.x, w0.y, w0.z}, q1{w1.x, w1.y, w1.z}, q2{w2.x, w2.y, w2.z};
                TriHit th;
                // the triangle the ray left: q.last_* are kEmpty without one,
                // which neither an instance nor a triangle id is
                const bool left = inst == q.last_inst && tri == q.last_tri;
                if (!tri_test(pre, q0, q1, q2, th) || left) continue;
                if (kNearby && th.t >= q.tmin) {
                    ex_t = gmin(ex_t, th.t);
                    ex_code = (int)tri;
                }
                if (th.t < q.tmin || th.t > tbest) continue;
                tbest = th.t;
                hit.t = th.t;
                hit.inst = inst;
                hit.tri = tri;
                if (!kAny) {
                    hit.b0 = th.e0 * th.inv;
                    hit.b1 = th.e1 * th.inv;
                    hit.b2 = th.e2 * th.inv;
                }
                if (kAny) return kTravHit;
            }
        }
        return pop<true>(ls);
    }
};

// Traversal steps of the wave's continuing lanes (r == kTravContinue).
// Node visits and leaf tests are two long code paths; while at least
// kInnerFirst lanes are at wide nodes, only those lanes step, so each path
// runs with a fuller wave instead of both running under partial masks; with
// fewer at nodes every lane steps, so no lane waits for long.  kLoop: the
// node visits run as a loop of their own until fewer than kInnerFirst lanes
// are at nodes (the ray setup then stays in place, which saves register
// copies per visit); faster for closest-hit rays, slower for shadow rays,
// which end at their first hit.  Measured best on the interior frame:
// kInnerFirst 16 with the loop (closest hit), 24 without (shadow rays); 8
// and 32 were slower for both.
template <int kInnerFirst, bool kLoop, class TV, class SC, class LS>
__device__ __forceinline__ void wave_step(TV &tv, int &r, const SC &sc, LS &ls, TraceCounters &tc)
{
    if constexpr (kLoop) {
        for (;;) {
            const bool at_node = r == kTravContinue && !(tv.node & kLeafBit);
            if (__popcll(__ballot(at_node)) < kInnerFirst) break;
            if (at_node) r = tv.template visit_node<false>(sc, ls, tc);
        }
        if (r == kTravContinue) r = tv.step(sc, ls, tc);
    } else {
        const bool leaf = (tv.node & kLeafBit) != 0;
        const uint64_t inner = __ballot(r == kTravContinue && !leaf);
        if (r == kTravContinue && (!leaf || __popcll(inner) < kInnerFirst)) r = tv.step(sc, ls, tc);
    }
}

// Returns 1 on hit, 0 on miss, -1 on stack overflow (the ray is abandoned).
template <int kMode, bool kAny, bool kNearby, bool kCount, bool kSphere, int kStack, typename LS>
YM_HD int traverse(const DevScene &sc, const Query &q, Hit &hit, int &nb_count, LS &ls, TraceCounters &cnt)
{
    Traversal<kMode, kAny, kNearby, kCount, kSphere, kStack> tv;
    int r = tv.init(sc, q);
    while (r == kTravContinue) r = tv.step(sc, ls, cnt);
    if (!kAny && r == kTravHit) tv.resolve_backs(sc, ls);
    hit = tv.hit;
    nb_count = tv.nb_count;
    return r == kTravHit ? 1 : (r == kTravMiss ? 0 : -1);
}

#undef YM_SORT2

}  // namespace ym
