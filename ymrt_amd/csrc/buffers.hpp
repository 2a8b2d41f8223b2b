// buffers.hpp -- path-state buffers of the frame drivers (render.cpp, batch.cpp).
#pragma once

#include <algorithm>
#include <vector>

#include "internal.hpp"
#include "pt.hpp"

namespace ym {

// Pass counters per chunk slot.
constexpr size_t kCountersPerSlot = (size_t)(kMaxPasses + 2) * kCtrStride;

struct RenderBuffers {
    uint32_t cap = 0;
    // the adjoint's replay pass: its own pass counters, statistics and slot
    uint32_t *adj_counters = nullptr;
    unsigned long long *adj_stats = nullptr;
    FrameSlot *adj_slot = nullptr;
    PathState ps{};
    std::vector<void *> allocs;
    uint32_t *counters = nullptr;
    unsigned long long *stats = nullptr;
    FrameSlot *slots = nullptr;  // device table of the chunks a launch serves
    std::vector<hipEvent_t> events;
    size_t event_next = 0;

    ~RenderBuffers()
    {
        for (void *p : allocs) (void)hipFree(p);
        for (hipEvent_t e : events) (void)hipEventDestroy(e);
    }
};

template <typename T>
inline int alloc(RenderBuffers *rb, T **p, size_t count)
{
    void *m = nullptr;
    YM_HIP(hipMalloc(&m, sizeof(T) * std::max<size_t>(count, 1)));
    rb->allocs.push_back(m);
    *p = static_cast<T *>(m);
    return YMRT_OK;
}

// Lays out the path state of n paths (and the pass counters and statistics)
// through get(pointer, count), which allocates or carves each array.  A batch
// shares the path state among up to `slots` frame chunks: pass counters and
// compaction counts per slot, statistics per frame (stat_sets).
template <typename Get>
inline int layout_buffers(RenderBuffers &rb, size_t n, uint32_t spill_threads, Get &&get, uint32_t slots = 1,
                          uint32_t stat_sets = 1)
{
    PathState &ps = rb.ps;
    int rc = 0;
    rc |= get(ps.ray, n * 2);
    rc |= get(ps.bs, n * 2);
    rc |= get(ps.acc, n * 2);
    rc |= get(ps.xhdr, n);
    rc |= get(ps.xrec, n * kMaxBoundaryRecord);
    rc |= get(ps.hit, n * 2);
    rc |= get(ps.nb, n * 4);
    rc |= get(ps.sh, n * kShadowSlots * 4);
    rc |= get(ps.sh_flags, n);
    rc |= get(ps.out, n);
    rc |= get(ps.queue[0], n);
    rc |= get(ps.queue[1], n);
    rc |= get(ps.q_hit, n);
    rc |= get(ps.q_hit_vol, n);
    rc |= get(ps.q_hit_diffuse, n);
    rc |= get(ps.q_hit_metal, n);
    rc |= get(ps.q_medium, n);
    rc |= get(ps.flag, n);
    rc |= get(ps.ccount, 4 * (n / kCompactSpan + 1) * slots);
    rc |= get(ps.q_shadow, n);
    rc |= get(ps.q_transmit, n);
    rc |= get(ps.spill, (size_t)(kMaxStackDepth - kStackWindow) * spill_threads);
    rc |= get(ps.first_hit, n);
    rc |= get(rb.counters, kCountersPerSlot * slots);
    rc |= get(rb.stats, (size_t)kStatCount * stat_sets);
    rc |= get(rb.slots, (size_t)slots);
    ps.spill_threads = spill_threads;
    return rc;
}

// Device memory that each path of a frame chunk takes (rounded up), with what
// the adjoint's replay adds when it first runs.
inline uint64_t path_bytes()
{
    auto total = [](size_t n) {
        RenderBuffers sizes;  // owns nothing: only the layout is computed
        size_t bytes = 0;
        layout_buffers(sizes, n, 0, [&](auto *&p, size_t count) {
            bytes += sizeof(*p) * count;
            return 0;
        });
        return bytes;
    };
    constexpr size_t n = (size_t)kCompactSpan * 256;
    return (total(n) - total(0) + n - 1) / n + sizeof(*PathState{}.adj_g);
}

}  // namespace ym
