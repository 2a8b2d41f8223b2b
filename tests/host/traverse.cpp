// The library's traversal (dev_traverse.hpp) and tree builder (bvh.hpp)
// compiled for the host, for scenes of one mesh under one instance: the tree
// is the one that the library builds for such a scene, so hits, any-hit flags
// and visit counts have to equal the GPU's bit for bit.  TEST CODE ONLY.
#include <algorithm>
#include <cstring>
#include <memory>
#include <vector>

#include "../../ymrt_amd/csrc/buffers.hpp"
#include "../../ymrt_amd/csrc/bvh.hpp"
#include "../../ymrt_amd/csrc/dev_traverse.hpp"

using namespace ym;

namespace {

constexpr int kHostStack = 96;  // the library's deepest stack

struct Mesh {
    std::vector<WNode> nodes;
    std::vector<float4> tris;
    std::vector<ShadeTri> shade;
    DevInstance in{};
    DevScene sc{};
    uint32_t max_stack = 0;
};

// kRing: a window of 16 entries with the deeper ones apart and the parked ray
// setup, as the kernels keep them; otherwise one plain stack.
template <bool kRing>
struct Scratch;
template <>
struct Scratch<false> {
    uint32_t stack[kHostStack];
    LaneScratch<1> ls{stack, nullptr, nullptr, nullptr, 0, nullptr, 0, 0};
};
template <>
struct Scratch<true> {
    uint32_t stack[16], deep[kHostStack - 16];
    float park[kPreSlots];
    LaneScratch<1, 16, true, kHostStack - 16> ls{stack, nullptr, nullptr, nullptr, 0, nullptr, 0, 0, park, deep};
};

Query query(const float *r)
{
    Query q;
    q.o = f3{r[0], r[1], r[2]};
    q.tmin = r[3];
    q.d = f3{r[4], r[5], r[6]};
    q.tmax = r[7];
    q.last_inst = q.last_tri = kEmpty;
    return q;
}

// deepest: the most stack entries a ray of the call held at once
template <bool kAny, bool kRing>
void trace(const Mesh &m, const float *rays, uint32_t n, uint32_t *out, uint32_t *visits, int *deepest)
{
    auto s = std::make_unique<Scratch<kRing>>();
    for (uint32_t i = 0; i < n; ++i) {
        Traversal<kAny ? kModeSkipBoundary : kModeAll, kAny, false, true, false, kHostStack> tv;
        TraceCounters cnt{0, 0};
        int r = tv.init(m.sc, query(rays + 8 * (size_t)i));
        while (r == kTravContinue) {
            r = tv.step(m.sc, s->ls, cnt);
            *deepest = std::max(*deepest, tv.sp);
        }
        if (kAny) {
            out[i] = r == kTravHit;
        } else {
            if (r == kTravHit) tv.resolve_backs(m.sc, s->ls);
            const uint32_t miss[4] = {f2u(kTMax), kEmpty, kEmpty, 0u};
            const uint32_t hit[4] = {f2u(tv.hit.t), tv.hit.tri, tv.hit.inst, (uint32_t)tv.hit.back};
            std::memcpy(out + 4 * (size_t)i, r == kTravHit ? hit : miss, sizeof(hit));
        }
        visits[2 * (size_t)i] = cnt.nodes;
        visits[2 * (size_t)i + 1] = cnt.tris;
    }
}

}  // namespace

extern "C" {

// pos: the corners of n triangles; w2o: three rows of four, identity to link
// the mesh into the top-level tree as the library does.
void *ht_mesh(const float *pos, uint32_t n, const float *w2o)
{
    auto *m = new Mesh;
    std::vector<BuildPrim> prims(n);
    m->shade.resize(n);
    for (uint32_t t = 0; t < n; ++t) {
        const float *p = pos + 9 * (size_t)t;
        std::memcpy(m->shade[t].p, p, sizeof(m->shade[t].p));
        for (int k = 0; k < 3; ++k) prims[t].box.grow(p + 3 * k);
        prims[t].box.fix();
        for (int a = 0; a < 3; ++a) prims[t].c[a] = 0.5f * (prims[t].box.lo[a] + prims[t].box.hi[a]);
        prims[t].id = t;
    }
    BinaryBuilder builder(prims, 4);
    const std::vector<BinNode> bin = builder.build();
    uint32_t depth = 0;
    m->in.blas_root = collapse_wide(bin, m->nodes, 0, &depth);
    m->max_stack = 3 * depth + 2;
    std::memcpy(&m->in.w2o, w2o, sizeof(float) * 12);
    bool identity = true;
    for (int k = 0; k < 12; ++k) identity = identity && w2o[k] == (k % 5 == 0 ? 1.0f : 0.0f);
    for (const BuildPrim &b : prims) {
        const float *p = m->shade[b.id].p;
        m->tris.push_back(make_float4(p[0], p[1], p[2], u2f(b.id)));
        m->tris.push_back(make_float4(p[3], p[4], p[5], u2f(identity ? 0u : kEmpty)));
        m->tris.push_back(make_float4(p[6], p[7], p[8], 0.0f));
    }
    m->sc.nodes = m->nodes.data();
    m->sc.tris = m->tris.data();
    m->sc.shade = m->shade.data();
    m->sc.instances = &m->in;
    m->sc.instance_count = 1;
    m->sc.tlas_root = m->sc.tlas_root_solid = identity ? m->in.blas_root : instance_code(0);
    m->sc.tlas_root_boundary = kSentinel;
    return m;
}

void ht_free(void *m) { delete static_cast<Mesh *>(m); }
uint32_t ht_max_stack(void *m) { return static_cast<Mesh *>(m)->max_stack; }
uint32_t ht_node_count(void *m) { return (uint32_t)static_cast<Mesh *>(m)->nodes.size(); }
const void *ht_nodes(void *m) { return static_cast<Mesh *>(m)->nodes.data(); }

// out: hits (4 words per ray) or any-hit flags; visits: 2 words per ray.
// Returns the most stack entries held at once.
int ht_trace(void *mesh, const float *rays, uint32_t n, int any, int ring, uint32_t *out, uint32_t *visits)
{
    const Mesh &m = *static_cast<Mesh *>(mesh);
    int deepest = 0;
    if (any && ring) trace<true, true>(m, rays, n, out, visits, &deepest);
    else if (any) trace<true, false>(m, rays, n, out, visits, &deepest);
    else if (ring) trace<false, true>(m, rays, n, out, visits, &deepest);
    else trace<false, false>(m, rays, n, out, visits, &deepest);
    return deepest;
}

// One visit_node of ray i at nodes[i].  out[4 * i]: the codes that it goes on
// to, in order (the node it moves to, then the stack from its top), and
// kSentinel past them.  park: the ray's setup goes through the parked form
// first, as after an instance.
void ht_visit(const void *nodes, const float *rays, uint32_t n, int park, uint32_t *out)
{
    auto s = std::make_unique<Scratch<true>>();
    for (uint32_t i = 0; i < n; ++i) {
        DevScene sc{};
        sc.nodes = static_cast<const WNode *>(nodes) + i;
        sc.instance_count = 1;
        Traversal<kModeAll, false, false, false, false, kHostStack> tv;
        TraceCounters cnt{0, 0};
        tv.init(sc, query(rays + 8 * (size_t)i));
        if (park) {
            s->ls.park_pre(tv.pre);
            tv.pre = s->ls.unpark_pre(tv.q.o, tv.q.d);
        }
        uint32_t *o = out + 4 * (size_t)i;
        std::fill(o, o + 4, kSentinel);
        if (tv.visit_node<false>(sc, s->ls, cnt) != kTravContinue) continue;
        *o++ = tv.node;
        while (tv.sp > 0) *o++ = s->ls.pop(--tv.sp);
    }
}

uint64_t ht_path_bytes() { return path_bytes(); }
}
