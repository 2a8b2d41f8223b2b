// kernels_pt.hip -- wavefront path tracing on gfx950.
//
// Stages of one bounce pass (the reference's Ray_generation / Ray_trace /
// Ray_shading kernels, src/Shading.cu:1634-2302, with its inline shadow rays
// split into their own stage):
//   raygen  camera rays for a chunk of (pixel, sample) paths
//   extend  closest hit + homogeneous/grid free-flight sampling, miss -> env
//   shade   surface or volume vertex: NEE light and BSDF/phase samples written
//           as up to two shadow rays, next direction, Russian roulette
//   shadow  any-hit of each shadow ray (+ boundary-walk transmittance when
//           media are on), adds the NEE term in the reference's order
//   resolve per-pixel mean over the samples of the chunk (sample order fixed,
//           so frames are deterministic -- no float atomics)
// Path state lies in HBM in records indexed by the path's slot (PathState);
// queues hold slot ids and are filled per wave64 with a ballot + one atomic per
// fetch of items, or by the compaction of the slots' stage flags.  Every kernel
// deals its queue over its waves from the length in a device counter, so
// launches never need the host to know queue lengths (no host round trip per
// stage).
#include <algorithm>
#include <mutex>
#include <unordered_map>

#include "dev_shade.hpp"
#include "dev_traverse.hpp"
#include "internal.hpp"
#include "pt.hpp"

namespace ym {

constexpr int kBlock = 64;

// ------------------------------------------------------------ wave helpers
__device__ __forceinline__ uint32_t lane_id() { return __lane_id(); }
// a value that all lanes of the wave hold, kept in a scalar register
__device__ __forceinline__ uint32_t uniform(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }

// Items a wave takes per work fetch: up to kSub sub-batches of 64.  Every
// global counter here is touched by all waves of the grid, and device-scope
// atomics on one address serialise across the chip, so a wave of a long queue
// fetches kSub * 64 items at once and publishes each output queue's survivors
// of all sub-batches with one atomic.  Stages with little work per item take
// more per fetch (ray generation 32 sub-batches, free flight 8), where the one
// counter's atomics would otherwise set the pace; the default of 4 measured
// best for the others.  Short queues are dealt in smaller shares (Share).
constexpr int kSub = 4;
constexpr int kRaygenSub = 32, kMediumSub = 8;

// A wave's part of one slot's queue.  The first dealt() items of the queue
// are dealt without atomics: the slot's home waves take grain() items each,
// this wave [first, first_end).  The items past dealt() are fetched from the
// slot's work counter, grain() at a time.  for_slots sets them; dealt and
// grain are read once per fetch and wait in LDS (kShareWords words per wave),
// where they cost the bodies no registers.
constexpr int kShareWords = 5;
// typed as LDS: a generic pointer would hold its 64-bit address in registers
using LdsWord = volatile __attribute__((address_space(3))) uint32_t;
struct Share {
    LdsWord *w;
    uint32_t first, first_end;
    __device__ __forceinline__ uint32_t dealt() const { return __builtin_amdgcn_readfirstlane(w[0]); }
    __device__ __forceinline__ uint32_t grain() const { return __builtin_amdgcn_readfirstlane(w[1]); }
    // the next range of a queue of n items; false when none is left
    __device__ __forceinline__ bool fetch(uint32_t *work, uint32_t n, uint32_t &cur, uint32_t &end) const
    {
        const uint32_t d = dealt();
        if (d >= n) return false;
        const uint32_t g = grain();
        uint32_t got = 0;
        if (__lane_id() == 0) got = atomicAdd(work, g);
        const uint32_t base = d + (uint32_t)__builtin_amdgcn_readfirstlane(got);
        if (base >= n) return false;
        cur = base;
        end = min(base + g, n);
        return true;
    }
};

// Persistent loop over n items (one wave per block): body(i, p, out) handles
// item i < n, sets p (the path slot it appends) and out[q] for each output
// queue q.  stage: LDS of kQueues * kS * 64 words.  Survivors of a fetch's
// sub-batches (at most kS) are staged in LDS and then published with one atomic
// per queue and a coalesced copy.
template <int kQueues, int kS = kSub, typename Body>
__device__ __forceinline__ void run_items(uint32_t *stage, const Share &share, uint32_t *fetch, uint32_t n,
                                          uint32_t *const *counters, uint32_t *const *queues, Body &&body)
{
    constexpr int kQ = kQueues > 0 ? kQueues : 1;
    const uint64_t below = (1ull << lane_id()) - 1ull;
    uint32_t base = share.first, end = share.first_end;
    for (;;) {
        if (base >= end && !share.fetch(fetch, n, base, end)) break;
        uint32_t filled[kQ] = {};
#pragma unroll 1
        for (; base < end; base += kBlock) {
            const uint32_t i = base + lane_id();
            uint32_t p = 0;
            bool out[kQ] = {};
            if (i < end) body(i, p, out);
            static_for<0, kQueues>([&](auto Q) {
                const uint64_t m = __ballot(out[Q()]);
                if (out[Q()]) stage[Q() * kS * kBlock + filled[Q()] + (uint32_t)__popcll(m & below)] = p;
                filled[Q()] += (uint32_t)__popcll(m);
            });
        }
        if constexpr (kQueues > 0) {
            __syncthreads();
            static_for<0, kQueues>([&](auto Q) {
                if (filled[Q()]) {
                    uint32_t dst = 0;
                    if (lane_id() == 0) dst = atomicAdd(counters[Q()], filled[Q()]);
                    dst = __shfl(dst, 0);
                    for (uint32_t j = lane_id(); j < filled[Q()]; j += kBlock)
                        queues[Q()][dst + j] = stage[Q() * kS * kBlock + j];
                }
            });
            __syncthreads();
        }
    }
}

// Lane refill: a kernel that keeps one traversal per lane lets finished lanes
// take new items while the others stay where they are in their trees, once
// kRefillLanes lanes are done.  Ray lengths vary by orders of magnitude, so a
// wave that waited for its slowest ray would run most of its steps with few
// lanes active.  refill() hands the wave's idle lanes the next items of its
// range [cur, end), which starts as its dealt share and is fetched from the
// work counter as it runs dry; it
// returns true on the lanes that took item *item.  Refilling at 32 (extend)
// and 16 (shadow) idle lanes measured fastest on the interior frame (extend:
// 16, 24, 28, 40 and 48 were 1-13 % slower; shadow: 8, 24 and 32 were
// slower or the same).
constexpr int kLaneIdle = 3;  // no ray (beside kTravContinue/Hit/Miss/Overflow)
template <int kRefillLanes>
struct RefillRange {
    const Share &share;
    uint32_t *work;
    uint32_t n;
    uint32_t cur, end;
    bool more;  // the range or the work counter may hold items
    __device__ __forceinline__ RefillRange(const Share &s, uint32_t *w, uint32_t count)
        : share(s), work(w), n(uniform(count)), cur(uniform(s.first)), end(uniform(s.first_end)),
          more(cur < end || s.dealt() < n)
    {
    }
    __device__ __forceinline__ bool refill(bool idle_lane, uint32_t &item)
    {
        const uint64_t below = (1ull << lane_id()) - 1ull;
        bool took = false;
        uint64_t idle = __ballot(idle_lane);
        while (idle && more) {
            if (cur >= end && !share.fetch(work, n, cur, end)) {
                more = false;
                break;
            }
            const uint32_t take = min((uint32_t)__popcll(idle), end - cur);
            if (idle_lane && !took) {
                const uint32_t rank = (uint32_t)__popcll(idle & below);
                if (rank < take) {
                    item = cur + rank;
                    took = true;
                }
            }
            cur = uniform(cur + take);
            idle = __ballot(idle_lane && !took);
        }
        // a queue dealt in full has nothing to fetch
        if (more && cur >= end && share.dealt() >= n) more = false;
        return took;
    }
    // lanes to wait for before the next refill: all of them once the counter
    // is drained, since nothing could refill them
    __device__ __forceinline__ uint32_t want() const { return more ? (uint32_t)kRefillLanes : (uint32_t)kBlock; }
};

__device__ __forceinline__ void wave_add64(unsigned long long *counter, uint32_t v)
{
    // sum v over the wave, one atomic
    uint32_t s = v;
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
    if (lane_id() == 0 && s) atomicAdd(counter, (unsigned long long)s);
}

// ------------------------------------------------------------ adjoint replay
// The replay pass of ymrt_render_adjoint runs the frame's paths a second time
// with the same samples (every random number is keyed by pixel, sample and
// vertex), so each path takes the same vertices and ps.out[p] already holds
// its radiance L_path from the first pass.  A gradient event whose factor
// multiplies every deposit after it adds adj . (L_path - L_now) * w; a term
// of one shadow ray's deposit D adds adj . D * w; adj is the pixel's
// dLoss/dImage over spp.  Sampling pdfs and MIS weights stay fixed.

// Pixel adjoint / spp of path slot p (64-bit slot arithmetic as k_raygen).
__device__ __forceinline__ f3 adj_pixel(const PtParams &prm, uint32_t p)
{
    const uint64_t gp = prm.chunk_base + p;
    const uint32_t spp = (uint32_t)prm.rs.spp;
    const uint64_t vpix = gp / spp;
    const uint32_t tile = (uint32_t)(vpix >> 8), within = (uint32_t)(vpix & 255u);
    const uint32_t ty = tile / prm.tiles_x, tx = tile - ty * prm.tiles_x;
    const uint32_t px = tx * 16u + (within & 15u), py = ty * 16u + (within >> 4);
    const float *a = prm.adj.img + ((size_t)py * prm.rs.width + px) * 3;
    const float inv = 1.0f / (float)spp;
    return f3{a[0] * inv, a[1] * inv, a[2] * inv};
}

// Gradient sums of one wave in a replay kernel: albedo rows and roughness
// entries go to LDS (kAdjLds floats when they fit) and reach global memory
// with one atomic per nonzero entry when the wave's work ends; texels and
// voxels go straight to global memory (their targets are spread out).
// kOn false: nothing is compiled.
template <bool kOn>
struct AdjSums {
    float *lds;
    const AdjParams *A;
    __device__ __forceinline__ void begin()
    {
        if constexpr (kOn) {
            if (A->lds) {
                for (uint32_t i = lane_id(); i < kAdjLds; i += kBlock) lds[i] = 0.0f;
                __syncthreads();
            }
        }
    }
    __device__ __forceinline__ void add(uint32_t i, float v)
    {
        if constexpr (kOn) {
            if (v == 0.0f) return;
            if (A->lds) atomicAdd(&lds[i], v);
            else if (i < A->n_alb * 3u) unsafeAtomicAdd(&A->g_alb[i], v);
            else unsafeAtomicAdd(&A->g_rough[i - A->n_alb * 3u], v);
        }
    }
    __device__ __forceinline__ void albedo(uint32_t row, int c, float v) { add(row * 3u + (uint32_t)c, v); }
    __device__ __forceinline__ void roughness(uint32_t entry, float v) { add(A->n_alb * 3u + entry, v); }
    __device__ __forceinline__ void end()
    {
        if constexpr (kOn) {
            if (A->lds) {
                __syncthreads();
                const uint32_t n = A->n_alb * 3u + A->n_rough;
                for (uint32_t i = lane_id(); i < n; i += kBlock) {
                    const float v = lds[i];
                    if (v == 0.0f) continue;
                    if (i < A->n_alb * 3u) unsafeAtomicAdd(&A->g_alb[i], v);
                    else unsafeAtomicAdd(&A->g_rough[i - A->n_alb * 3u], v);
                }
            }
        }
    }
};

// Density events of the trackers for the target volume's voxel grid: a real
// collision (probability sigma / sigma_m) adds scale * tsig / sigma, a null
// collision or a ratio-tracking step (1 - sigma / sigma_m) adds scale *
// -tsig / (sigma_m - sigma), tsig the target's sigma_t (gray); at most
// `left` events.
struct AdjTrackEvents {
    const DevScene &sc;
    float *g_vox;
    uint32_t vol;
    int grid;
    float tsig, scale;
    uint32_t left;
    int vox;
    __device__ __forceinline__ void note(int v, f3 po)
    {
        if ((uint32_t)v == vol) vox = grid_voxel(sc, grid, po);
    }
    __device__ __forceinline__ void real(float st, float sm)
    {
        (void)sm;
        if (vox >= 0 && st > 0.0f && left) {
            unsafeAtomicAdd(&g_vox[vox], scale * (tsig / st));
            --left;
        }
        vox = -1;
    }
    __device__ __forceinline__ void null(float st, float sm)
    {
        if (vox >= 0 && sm - st > 0.0f && left) {
            unsafeAtomicAdd(&g_vox[vox], scale * (-tsig / (sm - st)));
            --left;
        }
        vox = -1;
    }
};

__device__ __forceinline__ AdjTrackEvents adj_track(const DevScene &sc, const AdjParams &A, float scale,
                                                    uint32_t limit)
{
    const DevVolume &v = sc.volumes[A.vol];
    return AdjTrackEvents{sc, A.g_vox, A.vol, v.grid, v.sigma_t[0], scale, limit, -1};
}

// A shadow ray's transmittance records at most this many events; later ones
// are dropped (the CPU restatement of the adjoint drops the same).
constexpr uint32_t kAdjRayEvents = 1024;

// ------------------------------------------------------------ frame slots
// Multi-frame launches (ymrt_render_batch): one launch of a pass kernel serves
// every frame chunk of a round, each chunk a slot with its own scene,
// settings, counters and part of the path state.  A wave starts at its home
// slot -- the slot whose share of the launch's items holds the wave's index,
// so waves spread over the slots in proportion to their work -- drains it
// with the single-frame body, then visits the others in turn and helps with
// what is left there.  The slot index is wave-uniform, so the slot's fields
// come from scalar loads as kernel arguments do.
__device__ __forceinline__ uint32_t pass_counter(const FrameSlot &f, uint32_t pass, uint32_t k)
{
    return f.prm.counters[pass * kCtrStride + k];
}
__device__ __forceinline__ uint32_t *pass_work(const FrameSlot &f, uint32_t pass, uint32_t k)
{
    return f.prm.counters + pass * kCtrStride + k;
}

// Runs body(f, share) for the slots this wave works on: its home slot first,
// then the others.  count(f): the items queued in slot f; work(f): its work
// counter.  A launch's items are dealt in shares of `grain`:
//   * kMaxGrain when every wave of the grid gets that many: long queues, whose
//     fetch atomics (tens of ns each on one address, one after another across
//     the chip) would set the pace in smaller shares;
//   * down to kMinGrain, one full wave, otherwise, so that a short queue is
//     spread over all the waves the GPU holds: a wave's items run one sub-batch
//     after another, each a chain of dependent loads, and with shares of
//     kMaxGrain a 65536-path launch would occupy 256 of 1024 SIMDs for four
//     such chains.
//     Shares of less than a wave (16 or 32 rays to each traversal wave, on
//     more waves) are slower: the SIMDs then issue more instructions for the
//     same rays (Cornell 256x256 at 1 spp 2.9 and 2.4 ms against 2.1).
// The first share of each home wave is dealt by its index, so a queue that
// one round of shares covers takes no atomics at all; waves without a share
// leave at once.  rot: the grid index of the first wave that takes a share; the
// waves used come back, so that a kernel with several queues can deal each to
// other waves.  Shares of kMaxGrain from one counter against these (measured
// when the traversal kernels still took 16 rays to a wave, which cost Cornell
// 2.9 ms where it now takes 2.1): Cornell 256x256 at 1 spp 6.9 -> 3.1 ms, its
// 512x512 smoke at 16 spp (23 passes, the last of them short) 49 -> 40 ms, the
// interior at 1080p and 1 spp 27.7 -> 24.1 ms, at 64 spp 958 -> 950 ms.
template <uint32_t kMinGrain, uint32_t kMaxGrain, typename Count, typename Work, typename Body>
__device__ __forceinline__ uint32_t for_slots(const FrameSlot *__restrict__ fs, uint32_t nfs, Count count, Work work,
                                              Body body, uint32_t rot = 0)
{
    // words of Share, then what the next slot's deal needs: kept out of
    // registers while a body runs
    __shared__ uint32_t words[kShareWords];
    LdsWord *w = (LdsWord *)words;
    const uint32_t me = blockIdx.x >= rot ? blockIdx.x - rot : blockIdx.x + gridDim.x - rot;
    uint32_t home = 0, waves_used;
    {
        uint32_t total = 0;
        for (uint32_t s = 0; s < nfs; ++s) total += count(fs[s]);
        total = uniform(total);
        if (total == 0) return 0;
        const uint32_t per = total / gridDim.x;
        const uint32_t grain = per >= kMaxGrain ? kMaxGrain : per <= kMinGrain ? kMinGrain : per / kMinGrain * kMinGrain;
        const uint32_t waves = min((total + grain - 1) / grain, gridDim.x);
        if (me >= waves) return waves;
        waves_used = waves;
        // wave w's home is the slot whose items hold item floor(w * total / waves)
        uint32_t before = 0;
        if (nfs > 1) {
            const uint32_t target = (uint32_t)(((uint64_t)me * total) / waves);
            for (uint32_t c; home + 1 < nfs && before + (c = count(fs[home])) <= target; ++home) before += c;
        }
        w[1] = grain;
        w[2] = total;
        w[3] = waves;
        w[4] = before;
    }
    for (uint32_t j = 0; j < nfs; ++j) {
        const uint32_t s = __builtin_amdgcn_readfirstlane(home + j >= nfs ? home + j - nfs : home + j);
        const FrameSlot &f = fs[s];
        const uint32_t n = uniform(count(f));
        const uint32_t before = s == 0 ? 0u : (uint32_t)__builtin_amdgcn_readfirstlane(w[4]);
        w[4] = before + n;
        if (n == 0) continue;
        const uint32_t grain = __builtin_amdgcn_readfirstlane(w[1]);
        const uint32_t waves = __builtin_amdgcn_readfirstlane(w[3]);
        // home waves of slot s: ceil(before * waves / total) up to
        // ceil((before + n) * waves / total)
        uint32_t w0 = 0, w1 = waves;
        if (nfs > 1) {
            const uint32_t total = __builtin_amdgcn_readfirstlane(w[2]);
            w0 = (uint32_t)(((uint64_t)before * waves + total - 1) / total);
            w1 = (uint32_t)(((uint64_t)(before + n) * waves + total - 1) / total);
        }
        const uint32_t dealt = (uint32_t)min((uint64_t)(w1 - w0) * grain, (uint64_t)n);
        w[0] = dealt;
        Share share{w, 0, 0};
        if (j == 0) {
            share.first = min((me - w0) * grain, n);
            share.first_end = min(share.first + grain, n);
        } else if (dealt >= n || dealt + __hip_atomic_load(work(f), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= n) {
            continue;  // nothing left to fetch
        }
        body(f, share);
    }
    return waves_used;
}

// ------------------------------------------------------------ state access
__device__ __forceinline__ f3 xyz(float4 v) { return f3{v.x, v.y, v.z}; }
__device__ __forceinline__ float4 f4(f3 v, float w) { return make_float4(v.x, v.y, v.z, w); }

__device__ __forceinline__ Transfer load_transfer(const PathState &ps, uint32_t p, uint32_t cap)
{
    Transfer t;
    const uint32_t h = ps.xhdr[p];
    t.count = (int)(h & 0xFFu);
    t.max_idx = (int)((h >> 8) & 0xFFu) - 1;
#pragma unroll
    for (int i = 0; i < kMaxBoundaryRecord; ++i) {
        uint4 r = make_uint4(0u, 0u, 0u, 0u);
        if (i < t.count) r = ps.xrec[(size_t)i * cap + p];
        t.rec[i] = CameraRecord{r.x, __uint_as_float(r.y), r.z, (int32_t)r.w};
    }
    return t;
}
__device__ __forceinline__ void store_transfer(const PathState &ps, uint32_t p, uint32_t cap, const Transfer &t)
{
    ps.xhdr[p] = (uint32_t)t.count | ((uint32_t)(t.max_idx + 1) << 8);
#pragma unroll
    for (int i = 0; i < kMaxBoundaryRecord; ++i)
        if (i < t.count)
            ps.xrec[(size_t)i * cap + p] = make_uint4(t.rec[i].prim, __float_as_uint(t.rec[i].ior),
                                                      t.rec[i].priority, (uint32_t)t.rec[i].vol);
}
// hit flags
constexpr uint32_t kHitBack = 1u;
constexpr uint32_t kHitVolume = 2u;

// The nearby list of the path's hit record ha.  A list of one is the hit
// itself (the instance with the closest hit is always on it) and is not kept
// apart.
__device__ __forceinline__ NearbyList load_nearby(const PathState &ps, uint32_t p, uint32_t cap, uint4 ha)
{
    NearbyList nb;
    nb.n = (int)((ha.w >> 4) & 0xFu);
#pragma unroll
    for (int i = 0; i < kNearbyMax; ++i) {
        uint2 e = make_uint2(0u, 0u);
        if (i == 0) e = make_uint2(ha.y | ((ha.w & kHitBack) << 31), ha.x);
        if (i < nb.n && nb.n > 1) e = ps.nb[(size_t)i * cap + p];
        nb.prim[i] = e.x & 0x7FFFFFFFu;
        nb.back[i] = (int)(e.x >> 31);
        nb.t[i] = __uint_as_float(e.y);
    }
    return nb;
}
__device__ __forceinline__ Sampler load_sampler(const PathState &ps, uint32_t p)
{
    const uint4 s = *ps.smp(p);
    Sampler r;
    r.index = (uint64_t)s.x | ((uint64_t)s.y << 32);
    r.dim = s.z;
    r.frame_type = s.w;
    return r;
}
__device__ __forceinline__ void store_sampler(const PathState &ps, uint32_t p, const Sampler &s)
{
    *ps.smp(p) = make_uint4((uint32_t)s.index, (uint32_t)(s.index >> 32), s.dim, s.frame_type);
}

// info word
constexpr uint32_t kInfoNeverScatter = 1u << 8;
constexpr uint32_t kInfoPendingBunch = 1u << 10;
__device__ __forceinline__ int info_depth(uint32_t i) { return (int)(i & 0xFFu); }
__device__ __forceinline__ uint32_t info_vertex(uint32_t i) { return i >> 16; }

// Stage flag kind of a surface hit on a material of shading class cls.
__device__ __forceinline__ uint32_t shade_flag(uint32_t cls)
{
    return cls == kMatDiffuse ? kFlagDiffuse : cls == kMatMetal ? kFlagMetal : kFlagHit;
}

// shadow flags: bits 0-3 shadow ray k recorded (slots 0-1 shape light,
// 2-3 distant light), 4-7 ray k crosses the surface, 8-11 ray k reached the
// light past solid geometry, 12 volume vertex, 13 path ends after this
// shadow stage, 16-23 vertex depth, 24-31 and 14-15 the low and high bits of the
// vertex number (at most kMaxPasses), which keys the random numbers of the
// transmittance stage
constexpr uint32_t kShActiveMask = 0xFu;
constexpr uint32_t kShTransmit0 = 1u << 4;
constexpr uint32_t kShClear0 = 1u << 8;
constexpr uint32_t kShClearMask = 0xFu << 8;
constexpr uint32_t kShVolume = 1u << 12;
constexpr uint32_t kShTerminate = 1u << 13;
constexpr uint32_t kShDepthShift = 16;
static_assert(kMaxPasses < 1024, "a vertex number has ten bits");
__device__ __forceinline__ uint32_t sh_vertex_bits(uint32_t v) { return (v & 0xFFu) << 24 | ((v >> 8) & 3u) << 14; }
__device__ __forceinline__ uint32_t sh_vertex(uint32_t fl) { return fl >> 24 | ((fl >> 14) & 3u) << 8; }

// indirect_light_clamp (src/Shading.cu:61-81).  Its powers use the GPU's
// float powf: the double-precision form (ym_powf) would raise the registers
// of every kernel that deposits radiance, for a setting that is off in the
// measured workloads.
__device__ __forceinline__ f3 light_clamp(const ymrt_render_settings &rs, f3 c, int depth)
{
    if (!(rs.enable_indirect_clamp && depth > 1)) return c;
    if (!(rs.indirect_limit > 0.0f)) return s3(0.0f);
    const float lum = luminance(c);
    if (lum <= 1E-10f) return c;
    const float lim = rs.indirect_limit;
    const float pw = gmin(0.05f + 0.25f * powf(lum / lim, 1.5f), 1.0f);
    const float sf = powf(lim / (lim + lum), pw);
    return c * sf;
}

// ------------------------------------------------------------ raygen
__device__ __forceinline__ void raygen_body(const DevScene &sc, const PtParams &prm, const PathState &ps,
                                            const Share &share)
{
    uint32_t *cnt = prm.counters;  // pass 0 slots
    uint32_t *const ctrs[1] = {cnt + kCtrActive};
    uint32_t *const qs[1] = {ps.queue[0]};
    __shared__ uint32_t stage[kRaygenSub * kBlock];
    run_items<1, kRaygenSub>(stage, share, cnt + kCtrWorkRaygen, prm.chunk_paths, ctrs, qs,
                             [&](uint32_t p, uint32_t &slot, bool(&out)[1]) {
        slot = p;
        ps.flag[p] = 0;
        {
            const uint64_t gp = prm.chunk_base + p;
            const uint32_t spp = (uint32_t)prm.rs.spp;
            const uint64_t vpix = gp / spp;
            const uint32_t s = (uint32_t)(gp - vpix * spp);
            const uint32_t tile = (uint32_t)(vpix >> 8), within = (uint32_t)(vpix & 255u);
            const uint32_t ty = tile / prm.tiles_x, tx = tile - ty * prm.tiles_x;
            const uint32_t px = tx * 16u + (within & 15u), py = ty * 16u + (within >> 4);
            if (px < prm.rs.width && py < prm.rs.height) {
                out[0] = true;
                const uint32_t pixel_index = py * prm.rs.width + px;
                Sampler smp;
                float ox, oy;
                if (prm.rs.sampler_type == YMRT_SAMPLER_HALTON) {
                    smp.index = prm.henum.index(px, py, (uint32_t)((prm.frame - 1) * prm.rs.spp) + s);
                    smp.dim = 2;
                    smp.frame_type = kSamplerHalton;
                    ox = radical_inverse_plain<2>(smp.index);
                    oy = radical_inverse_plain<3>(smp.index);
                    ox = __builtin_fmaf(ox, prm.henum.x_scale, -(float)px);
                    oy = __builtin_fmaf(oy, prm.henum.y_scale, -(float)py);
                    ox = gclamp(ox, 0.000001f, 0.999999f);
                    oy = gclamp(oy, 0.000001f, 0.999999f);
                } else {
                    smp.index = (uint64_t)pixel_index | ((uint64_t)s << 32);
                    smp.dim = 0;
                    smp.frame_type = (uint32_t)(prm.frame - 1) << 1;
                    ox = sampler_next(sc, smp);
                    oy = sampler_next(sc, smp);
                }
                const DevCamera &cam = sc.camera;
                const float nx = ((float)px + ox) / (float)prm.rs.width;
                const float ny = ((float)py + oy) / (float)prm.rs.height;
                const float height = 2.0f * cam.tan_half_fov;
                const float width = height * cam.aspect;
                const f3 dir = normalize(-cam.w + ((nx - 0.5f) * width) * cam.u + ((ny - 0.5f) * height) * cam.v);
                *ps.ray_o(p) = f4(cam.position, __uint_as_float(kEmpty));
                *ps.ray_d(p) = f4(dir, __uint_as_float(kEmpty));
                *ps.beta(p) = make_float4(1.0f, 1.0f, 1.0f, __uint_as_float(1u | kInfoNeverScatter));
                *ps.L(p) = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                store_sampler(ps, p, smp);
                Transfer t;
                t.count = cam.record_count;
                t.max_idx = cam.max_idx;
                for (int i = 0; i < kMaxBoundaryRecord; ++i) t.rec[i] = cam.rec[i];
                store_transfer(ps, p, prm.cap, t);
            }
        }
    });
}


__global__ __launch_bounds__(kBlock) void k_raygen_m(const FrameSlot *__restrict__ fs, uint32_t nfs)
{
    for_slots<kBlock, kBlock * kRaygenSub>(
        fs, nfs, [](const FrameSlot &f) { return f.prm.chunk_paths; },
        [](const FrameSlot &f) { return f.prm.counters + kCtrWorkRaygen; },
        [](const FrameSlot &f, const Share &share) { raygen_body(f.sc, f.prm, f.ps, share); });
}



// ------------------------------------------------------------ extend
// Closest hit for every queued path (Ray_trace_path_tracing,
// src/Shading.cu:1765-1901).  With kMedia, paths that carry medium records
// hand their hit or miss to k_medium, which samples free flight; the others
// resolve misses here and queue surface hits for shading.  Visited wide nodes
// and tested triangles are summed per wave into the frame statistics.
// Each lane keeps its own traversal and is refilled as it finishes
// (RefillRange).

template <bool kNearby, bool kMedia, bool kSphere, int kStack>
__device__ __forceinline__ void extend_body(const DevScene &sc, const PtParams &prm, const PathState &ps, uint32_t pass,
                                            const Share &share)
{
    __shared__ uint32_t stack[kStackWindow * kBlock];
    __shared__ uint32_t nbp[(kNearby ? kNearbyCap : 1) * kBlock];
    __shared__ float nbt[(kNearby ? kNearbyCap : 1) * kBlock];
    __shared__ int nbb[(kNearby ? kNearbyCap : 1) * kBlock];
    __shared__ float pre_park[kPreSlots * kBlock];
    uint32_t *cnt = prm.counters + pass * kCtrStride;
    const uint32_t *qin = ps.queue[pass & 1];
    LaneScratch<kBlock, kStackWindow, true> ls{stack, nbp, nbt, nbb, (int)lane_id(), ps.spill, ps.spill_threads,
                                               blockIdx.x * kBlock + threadIdx.x, pre_park};
    const ymrt_render_settings &rs = prm.rs;
    uint32_t rays = 0, cam_rays = 0;
    TraceCounters tc{0, 0};
    RefillRange<32> rr(share, cnt + kCtrWorkExtend, cnt[kCtrActive]);

    const TravScene ts(sc);
    Traversal<kModeAll, false, kNearby, true, kSphere, kStack> tv;
    uint32_t p = 0;
    int r = kLaneIdle;
    for (;;) {
        uint32_t item = 0;
        if (rr.more && rr.refill(r == kLaneIdle, item)) {
            p = gload(qin + item);
            const float4 o4 = gload(ps.ray_o(p)), d4 = gload(ps.ray_d(p));
            Query q;
            q.o = xyz(o4);
            q.d = xyz(d4);
            q.tmin = kTMin;
            q.tmax = kTMax;
            q.last_inst = __float_as_uint(o4.w);
            q.last_tri = __float_as_uint(d4.w);
            tv.hit.back = 0;
            tv.hit.tri = 0;
            tv.hit.b0 = tv.hit.b1 = tv.hit.b2 = 0.0f;
            r = tv.init(sc, q);
        }
        const uint32_t want = rr.want();
        for (;;) {
            const uint64_t busy = __ballot(r == kTravContinue);
            if (busy == 0 || (uint32_t)(kBlock - __popcll(busy)) >= want) break;
            wave_step<16, true>(tv, r, ts, ls, tc);
        }
        if (r != kTravContinue && r != kLaneIdle) {
            if (r == kTravOverflow) atomicOr(prm.error, 1u);
            const bool hit = r == kTravHit;
            r = kLaneIdle;
            if (hit) tv.resolve_backs(sc, ls);
            uint32_t info = gload(ps.info(p));
            if (info & kInfoPendingBunch) {
                // the boundary bunch of the previous vertex reads that
                // vertex's nearby list, which the writes below replace
                Transfer t = load_transfer(ps, p, prm.cap);
                const NearbyList nb = load_nearby(ps, p, prm.cap, *ps.hit_a(p));
                boundary_bunch(sc, t, nb);
                store_transfer(ps, p, prm.cap, t);
                info &= ~kInfoPendingBunch;
                *ps.info(p) = info;
            }
            rays += 1;
            cam_rays += (info_depth(info) == 1 && (info & kInfoNeverScatter)) ? 1u : 0u;
            const Hit &h = tv.hit;
            if (pass == 0 && prm.aov) ps.first_hit[p] = hit ? h.inst : kEmpty;
            const bool in_medium = kMedia && prm.media && (gload(ps.xhdr + p) & 0xFFu) != 0;
            if (!hit && !in_medium) {
                f3 Lv = xyz(gload(ps.L(p)));
                if (rs.enable_env_light)
                    Lv = Lv + light_clamp(rs, xyz(gload(ps.beta(p))) * background(tv.q.d), info_depth(info));
                gstore(ps.out + p, f4(Lv, 0.0f));
            } else {
                // a path in a medium may have no surface hit (h.inst empty);
                // one outside a medium always has one here
                const uint32_t mat = hit ? gload(&sc.instances[h.inst].material) : kEmpty;
                gstore(ps.flag + p, (pass << kFlagBits) | (in_medium ? kFlagMedium : shade_flag(gload(sc.mat_class + mat))));
                uint32_t flags = h.back ? kHitBack : 0u;
                int nbc = hit ? 1 : 0;  // without the list the hit is its own nearby hit
                if constexpr (kNearby) {
                    if (hit) nbc = tv.nb_count;
                    if (nbc > 1)
                        static_for<0, kNearbyCap>([&](auto K) {
                            if (K() < nbc)
                                gstore(ps.nb + (size_t)K() * prm.cap + p,
                                       make_uint2(nbp[K() * kBlock + lane_id()] |
                                                      ((uint32_t)(nbb[K() * kBlock + lane_id()] != 0) << 31),
                                                  __float_as_uint(nbt[K() * kBlock + lane_id()])));
                        });
                }
                flags |= (uint32_t)nbc << 4;
                gstore(ps.hit_a(p), make_uint4(__float_as_uint(hit ? h.t : kTMax), hit ? h.inst : kEmpty, h.tri, flags));
                gstore(ps.hit_b(p), make_float4(h.b0, h.b1, h.b2, 0.0f));
            }
        }
        if (!rr.more && __ballot(r != kLaneIdle) == 0) break;
    }
    wave_add64(prm.stats + kStatExtension, rays);
    wave_add64(prm.stats + kStatCamera, cam_rays);
    wave_add64(prm.stats + kStatExtendNodes, tc.nodes);
    wave_add64(prm.stats + kStatExtendTris, tc.tris);
}


template <bool kNearby, bool kMedia, bool kSphere, int kStack>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(kSphere ? 1 : 4))) void k_extend_m(const FrameSlot *__restrict__ fs, uint32_t nfs, uint32_t pass)
{
    for_slots<kBlock, kBlock * kSub>(
        fs, nfs, [&](const FrameSlot &f) { return pass_counter(f, pass, kCtrActive); },
        [&](const FrameSlot &f) { return pass_work(f, pass, kCtrWorkExtend); },
        [&](const FrameSlot &f, const Share &share) {
            extend_body<kNearby, kMedia, kSphere, kStack>(f.sc, f.prm, f.ps, pass, share);
        });
}



// ------------------------------------------------------------ compaction
// Gathers the paths flagged for the next stage of this pass (kShade: surface
// and volume shading; otherwise free flight) in slot order: the traversal
// kernels finish paths in no fixed order, and read in slot order the next
// stage's lanes (and neighbouring waves) load neighbouring path-state
// entries together.  A scan of every slot's flag (4 B) costs less than the
// scattered reads it saves.  No atomics: k_compact_count sums the matches of
// each block of kCompactSpan slots, k_compact_scatter writes a block's
// matches at the sum of the counts before it, and the block holding the last
// slot sets the queue lengths.
// kMode: kCompactMedium, kCompactShade (four queues) or kCompactTransmit
enum : int { kCompactMedium = 0, kCompactShade = 1, kCompactTransmit = 2 };
template <int kMode>
struct Compact {
    static constexpr int kQ = kMode == kCompactShade ? 4 : 1;
    __device__ static void match(uint32_t f, uint32_t tag, bool (&m)[kQ])
    {
        if constexpr (kMode == kCompactShade) {
            m[0] = f == (tag | kFlagHit);
            m[1] = f == (tag | kFlagVolume);
            m[2] = f == (tag | kFlagDiffuse);
            m[3] = f == (tag | kFlagMetal);
        } else {
            m[0] = f == (tag | (kMode == kCompactMedium ? kFlagMedium : kFlagTransmit));
        }
    }
};

template <int kMode>
__device__ __forceinline__ void compact_count_body(const PtParams &prm, const PathState &ps, uint32_t pass, uint32_t b)
{
    constexpr int kQ = Compact<kMode>::kQ;
    constexpr uint32_t kWaves = kCompactThreads / kBlock;
    __shared__ uint32_t red[kQ][kWaves];
    const uint32_t n = prm.chunk_paths;
    const uint32_t first = b * kCompactSpan;
    if (first >= n) return;
    const uint32_t last = min(first + kCompactSpan, n);
    const uint32_t tag = pass << kFlagBits;
    uint32_t c[kQ] = {};
    for (uint32_t i = first + threadIdx.x; i < last; i += kCompactThreads) {
        bool m[kQ];
        Compact<kMode>::match(ps.flag[i], tag, m);
        static_for<0, kQ>([&](auto Q) { c[Q()] += m[Q()] ? 1u : 0u; });
    }
    static_for<0, kQ>([&](auto Q) {
        uint32_t v = c[Q()];
        for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
        if (lane_id() == 0) red[Q()][threadIdx.x / kBlock] = v;
    });
    __syncthreads();
    if (threadIdx.x < (uint32_t)kQ) {
        uint32_t v = 0;
        for (uint32_t w = 0; w < kWaves; ++w) v += red[threadIdx.x][w];
        ps.ccount[threadIdx.x * prm.ccount_stride + b] = v;
    }
}


// one row of the grid (blockIdx.y) per slot
template <int kMode>
__global__ __launch_bounds__(kCompactThreads) void k_compact_count_m(const FrameSlot *__restrict__ fs, uint32_t pass)
{
    const FrameSlot &f = fs[blockIdx.y];
    compact_count_body<kMode>(f.prm, f.ps, pass, blockIdx.x);
}

template <int kMode>
__device__ __forceinline__ void compact_scatter_body(const PtParams &prm, const PathState &ps, uint32_t pass,
                                                     uint32_t b)
{
    constexpr int kQ = Compact<kMode>::kQ;
    constexpr uint32_t kWaves = kCompactThreads / kBlock;
    __shared__ uint32_t red[kQ][kWaves];
    __shared__ uint32_t base[kQ];
    uint32_t *cnt = prm.counters + pass * kCtrStride;
    const uint32_t n = prm.chunk_paths;
    const uint32_t first = b * kCompactSpan;
    if (first >= n) return;
    const uint32_t last = min(first + kCompactSpan, n);
    const uint32_t stride = prm.ccount_stride;
    uint32_t *const qs[4] = {kMode == kCompactShade    ? ps.q_hit
                             : kMode == kCompactMedium ? ps.q_medium
                                                       : ps.q_transmit,
                             ps.q_hit_vol, ps.q_hit_diffuse, ps.q_hit_metal};
    const uint32_t ctr[4] = {kMode == kCompactShade ? kCtrHit : kMode == kCompactMedium ? kCtrMedium : kCtrTransmit,
                             kCtrHitVol, kCtrHitDiffuse, kCtrHitMetal};
    const uint32_t tag = pass << kFlagBits;
    const uint32_t wave = threadIdx.x / kBlock;
    const uint64_t below = (1ull << lane_id()) - 1ull;
    // this block's offsets: the counts of the blocks before it, summed by
    // k_compact_scan
    if (threadIdx.x < (uint32_t)kQ) base[threadIdx.x] = ps.ccount[threadIdx.x * stride + b];
    __syncthreads();
    uint32_t off[kQ];
    static_for<0, kQ>([&](auto Q) { off[Q()] = base[Q()]; });
    for (uint32_t t0 = first; t0 < last; t0 += kCompactThreads) {
        const uint32_t i = t0 + threadIdx.x;
        uint32_t p = 0;
        bool m[kQ] = {};
        if (i < last) {
            p = i;
            Compact<kMode>::match(ps.flag[p], tag, m);
        }
        uint32_t rank[kQ];
        __syncthreads();  // red[] of the previous tile has been read
        static_for<0, kQ>([&](auto Q) {
            const uint64_t mask = __ballot(m[Q()]);
            rank[Q()] = (uint32_t)__popcll(mask & below);
            if (lane_id() == 0) red[Q()][wave] = (uint32_t)__popcll(mask);
        });
        __syncthreads();
        static_for<0, kQ>([&](auto Q) {
            uint32_t before = 0, total = 0;
            for (uint32_t w = 0; w < kWaves; ++w) {
                const uint32_t v = red[Q()][w];
                before += w < wave ? v : 0u;
                total += v;
            }
            if (m[Q()]) qs[Q()][off[Q()] + before + rank[Q()]] = p;
            off[Q()] += total;
        });
    }
    if (last == n && threadIdx.x < (uint32_t)kQ) cnt[ctr[threadIdx.x]] = off[threadIdx.x];
}


// The per-block counts of one slot (blockIdx.y; one block per queue) turned
// into their exclusive prefix sums in place, so that each scatter block reads
// its offsets instead of summing the counts of all blocks before it (a sum
// whose total work grows with the square of the block count).
constexpr uint32_t kScanThreads = 1024;
template <int kMode>
__global__ __launch_bounds__(kScanThreads) void k_compact_scan_m(const FrameSlot *__restrict__ fs)
{
    const FrameSlot &f = fs[blockIdx.y];
    constexpr int kQ = Compact<kMode>::kQ;
    constexpr uint32_t kWaves = kScanThreads / kBlock;
    __shared__ uint32_t wsum[kWaves];
    const uint32_t nb = (f.prm.chunk_paths + kCompactSpan - 1) / kCompactSpan;
    const uint32_t stride = f.prm.ccount_stride;
    const uint32_t per = (nb + kScanThreads - 1) / kScanThreads;
    const uint32_t lo = min(threadIdx.x * per, nb), hi = min(lo + per, nb);
    const uint32_t wave = threadIdx.x / kBlock;
    {
        const uint32_t q = blockIdx.x;  // one block per queue
        if (q >= (uint32_t)kQ) return;
        uint32_t *c = f.ps.ccount + (size_t)q * stride;
        uint32_t own = 0;
        for (uint32_t j = lo; j < hi; ++j) own += c[j];
        uint32_t incl = own;
        for (int off = 1; off < kBlock; off <<= 1) {
            const uint32_t y = __shfl_up(incl, off);
            if ((int)lane_id() >= off) incl += y;
        }
        if (lane_id() == kBlock - 1) wsum[wave] = incl;
        __syncthreads();
        uint32_t before = incl - own;
        for (uint32_t w = 0; w < wave; ++w) before += wsum[w];
        for (uint32_t j = lo; j < hi; ++j) {
            const uint32_t v = c[j];
            c[j] = before;
            before += v;
        }
    }
}

// one row of the grid (blockIdx.y) per slot
template <int kMode>
__global__ __launch_bounds__(kCompactThreads) void k_compact_scatter_m(const FrameSlot *__restrict__ fs, uint32_t pass)
{
    const FrameSlot &f = fs[blockIdx.y];
    compact_scatter_body<kMode>(f.prm, f.ps, pass, blockIdx.x);
}

// The whole compaction of short chunks in one launch: a block gathers
// kScanThreads slots and counts the matches before them itself.  The reads
// grow with the number of chunks and with the square of their length, so this
// is for chunks of up to kCompactSmall slots and for launches of which the
// chunks times the square of the longest is at most kCompactReads (32 MB of
// flags read).  There the reads are a few us, while three launches of the
// kernels above take about 23 with the gaps between them.  One launch against
// three, ms per call, 1 spp: Cornell frames of 64x64, 128x128 and 256x256 1.26
// and 1.40, 1.42 and 1.54, 1.65 and 1.72, with a medium (three compactions per
// pass) 3.66 and 4.29, 4.22 and 4.86, 5.03 and 5.48; batches of them with the
// medium, 4 and 16 of 256x256 8.32 and 8.79, 18.2 and 17.4; 64 of 256x256 49.6
// and 44.8; 32 and 64 of 128x128 17.2 and 17.8, 28.2 and 28.1.
constexpr uint32_t kCompactSmall = 65536;
constexpr uint64_t kCompactReads = 1ull << 34;
template <int kMode>
__global__ __launch_bounds__(kScanThreads) void k_compact_small_m(const FrameSlot *__restrict__ fs, uint32_t pass)
{
    const FrameSlot &f = fs[blockIdx.y];
    constexpr int kQ = Compact<kMode>::kQ;
    constexpr uint32_t kWaves = kScanThreads / kBlock;
    __shared__ uint32_t red[2][kQ][kWaves];
    const uint32_t n = f.prm.chunk_paths;
    const uint32_t first = blockIdx.x * kScanThreads;
    if (first >= n) return;
    const uint32_t *flag = f.ps.flag;
    const uint32_t tag = pass << kFlagBits;
    const uint32_t wave = threadIdx.x / kBlock;
    uint32_t c[kQ] = {};
#pragma unroll 8
    for (uint32_t i = threadIdx.x; i < first; i += kScanThreads) {
        bool m[kQ];
        Compact<kMode>::match(flag[i], tag, m);
        static_for<0, kQ>([&](auto Q) { c[Q()] += m[Q()] ? 1u : 0u; });
    }
    const uint32_t i = first + threadIdx.x;
    bool m[kQ] = {};
    if (i < n) Compact<kMode>::match(flag[i], tag, m);
    uint32_t rank[kQ];
    static_for<0, kQ>([&](auto Q) {
        uint32_t v = c[Q()];
        for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
        const uint64_t mask = __ballot(m[Q()]);
        rank[Q()] = (uint32_t)__popcll(mask & ((1ull << lane_id()) - 1ull));
        if (lane_id() == 0) {
            red[0][Q()][wave] = v;
            red[1][Q()][wave] = (uint32_t)__popcll(mask);
        }
    });
    __syncthreads();
    uint32_t *const qs[4] = {kMode == kCompactShade    ? f.ps.q_hit
                             : kMode == kCompactMedium ? f.ps.q_medium
                                                       : f.ps.q_transmit,
                             f.ps.q_hit_vol, f.ps.q_hit_diffuse, f.ps.q_hit_metal};
    const uint32_t ctr[4] = {kMode == kCompactShade ? kCtrHit : kMode == kCompactMedium ? kCtrMedium : kCtrTransmit,
                             kCtrHitVol, kCtrHitDiffuse, kCtrHitMetal};
    uint32_t *cnt = f.prm.counters + pass * kCtrStride;
    static_for<0, kQ>([&](auto Q) {
        uint32_t before = 0, total = 0;
        for (uint32_t w = 0; w < kWaves; ++w) {
            before += red[0][Q()][w] + (w < wave ? red[1][Q()][w] : 0u);
            total += red[0][Q()][w] + red[1][Q()][w];
        }
        if (m[Q()]) qs[Q()][before + rank[Q()]] = i;
        if (first + kScanThreads >= n && threadIdx.x == 0) cnt[ctr[Q()]] = total;
    });
}

// ------------------------------------------------------------ medium
// Free flight through the media of the path's top-priority records
// (SampleVolumeScattering, src/VolumeEval.cuh:217-251, called from
// src/Shading.cu:1800-1840): scattering vertices go to the volume shading
// queue, surviving rays to surface shading or, on a miss, to the environment.
// kHet: 1 the scene has voxel-grid media (delta tracking), 2 texture-density
// media as well (the texture graph evaluator and its LDS stack are compiled
// in); 0 every medium is homogeneous and the tracker is compiled out.
// kAdj (the adjoint's replay): the delta tracker's collisions in the target
// grid volume are density gradient events.  The homogeneous variant is held
// to 5 waves per SIMD (96 VGPRs, no spills): it waits on memory most of the
// time, and the fifth wave measured 1.5 % faster than four.
template <int kHet, bool kAdj = false>
__device__ __forceinline__ void medium_body(const DevScene &sc, const PtParams &prm, const PathState &ps, uint32_t pass,
                                            const Share &share)
{
    constexpr bool kGrid = kHet > 0;
    __shared__ float tex_stk[kHet == 2 ? kTexStack * 3 * kBlock : 1];
    uint32_t *cnt = prm.counters + pass * kCtrStride;
    const uint32_t n = cnt[kCtrMedium];
    const ymrt_render_settings &rs = prm.rs;
    run_items<0, kMediumSub>(nullptr, share, cnt + kCtrWorkMedium, n, nullptr, nullptr, [&](uint32_t i, uint32_t &p, bool(&)[1]) {
        {
            p = ps.q_medium[i];
            const uint4 ha = *ps.hit_a(p);
            const bool hit = ha.y != kEmpty;
            const f3 o = xyz(*ps.ray_o(p)), d = xyz(*ps.ray_d(p));
            const float4 bi = *ps.beta(p);
            f3 beta = xyz(bi);
            bool vol_hit = false;
            float dist = 0.0f;
            const Transfer t = load_transfer(ps, p, prm.cap);
            int vi[kMaxBoundaryRecord];
            const int nv = t.volumes(vi, sc.volume_count);
            if (nv > 0) {
                Sampler smp = load_sampler(ps, p);
                bool het = false;
                if constexpr (kGrid) {
                    static_for<0, kMaxBoundaryRecord>([&](auto K) {
                        if (K() < nv && vol_is_het(sc, vi[K()])) het = true;
                    });
                }
                f3 trw;
                const float tmax = hit ? __uint_as_float(ha.x) : kTMax;
                if constexpr (kGrid && kAdj) {
                    // every later deposit of the path depends on this flight
                    float scale = 0.0f;
                    if (het && prm.adj.vol != kEmpty) {
                        const f3 dl = adj_pixel(prm, p) * (xyz(ps.out[p]) - xyz(*ps.L(p)));
                        scale = dl.x + dl.y + dl.z;
                    }
                    if (scale != 0.0f) {
                        AdjTrackEvents ev = adj_track(sc, prm.adj, scale, 0xFFFFFFFFu);
                        vol_hit = sample_heterogeneous<kHet == 2>(sc, nv, vi, o, d, tmax, trw, dist, smp, tex_stk, ev);
                    } else {
                        vol_hit = het ? sample_heterogeneous<kHet == 2>(sc, nv, vi, o, d, tmax, trw, dist, smp, tex_stk)
                                      : sample_homogeneous(sc, nv, vi, tmax, trw, dist, smp);
                    }
                } else if constexpr (kGrid) {
                    vol_hit = het ? sample_heterogeneous<kHet == 2>(sc, nv, vi, o, d, tmax, trw, dist, smp, tex_stk)
                                  : sample_homogeneous(sc, nv, vi, tmax, trw, dist, smp);
                } else {
                    vol_hit = sample_homogeneous(sc, nv, vi, tmax, trw, dist, smp);
                }
                beta = beta * trw;
                *ps.beta(p) = f4(beta, bi.w);
                store_sampler(ps, p, smp);
            }
            if (vol_hit) {
                ps.flag[p] = (pass << kFlagBits) | kFlagVolume;
                const f3 vpos = o + d * dist;
                *ps.hit_a(p) = make_uint4(ha.x, ha.y, ha.z, ha.w | kHitVolume);
                *ps.hit_b(p) = make_float4(vpos.x, vpos.y, vpos.z, 0.0f);
            } else if (hit) {
                ps.flag[p] = (pass << kFlagBits) | shade_flag(sc.mat_class[sc.instances[ha.y].material]);
            } else {
                f3 Lv = xyz(*ps.L(p));
                if (rs.enable_env_light) Lv = Lv + light_clamp(rs, beta * background(d), info_depth(__float_as_uint(bi.w)));
                ps.out[p] = f4(Lv, 0.0f);
            }
        }
    });
}


template <int kHet, bool kAdj = false>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(kHet ? 1 : 5))) void k_medium_m(const FrameSlot *__restrict__ fs, uint32_t nfs, uint32_t pass)
{
    for_slots<kBlock, kBlock * kMediumSub>(
        fs, nfs, [&](const FrameSlot &f) { return pass_counter(f, pass, kCtrMedium); },
        [&](const FrameSlot &f) { return pass_work(f, pass, kCtrWorkMedium); },
        [&](const FrameSlot &f, const Share &share) { medium_body<kHet, kAdj>(f.sc, f.prm, f.ps, pass, share); });
}



// ------------------------------------------------------------ shade
// Adjoint replay, a surface vertex whose diffuse albedo is the target image
// texture (every material using it is Lambert-only): the albedo is a bilinear
// blend of four texels, so each tap's texel channel c gets dl_c * w / albedo_c
// (a one-channel texture: the sum over the colour channels).
__device__ __forceinline__ void adj_texels(const DevScene &sc, const AdjParams &A, f2 uv, f3 dl)
{
    const DevTexture &t = sc.textures[A.tex];
    const f3 al = image_eval(sc, t, uv);
    uint32_t off[4];
    float w[4];
    image_taps(t, uv, off, w);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        if (!(w[k] > 0.0f)) continue;
        if (t.channels == 1) {
            const float v = (al.x > 0.0f ? dl.x * (w[k] / al.x) : 0.0f) + (al.y > 0.0f ? dl.y * (w[k] / al.y) : 0.0f) +
                            (al.z > 0.0f ? dl.z * (w[k] / al.z) : 0.0f);
            if (v != 0.0f) unsafeAtomicAdd(&A.g_tex[off[k]], v);
        } else {
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const float a = comp(al, c);
                if (!(a > 0.0f)) continue;
                const float v = comp(dl, c) * (w[k] / a);
                if (v != 0.0f) unsafeAtomicAdd(&A.g_tex[off[k] + (uint32_t)c], v);
            }
        }
    }
}

// Records shadow ray k of path p (origin, direction, maximum distance, BSDF or
// phase value, clamped Li, MIS weight) straight to its slot in HBM.  The
// direction is renormalised as the reference's Ray constructor does
// (src/Ray.h:28-29): a light-sample direction is already unit length up to
// rounding, and those last bits decide self-hits of rays that leave a surface
// with no spawn offset.
struct ShadowEmit {
    const PathState &ps;
    uint32_t p;
    uint32_t flags;
    // g: the adjoint replay's d ln f / d r of the ray's BSDF value (0 otherwise)
    __device__ __forceinline__ void emit(int k, f3 orig, f3 dir, float tmax, bool transmit, f3 f, f3 li, float mis,
                                         float g = 0.0f)
    {
        float4 *r = ps.shadow(k, p);
        r[0] = f4(orig, tmax);
        r[1] = f4(normalize(dir), 0.0f);
        r[2] = f4(f, mis);
        r[3] = f4(li, g);
        flags |= (1u << k) | (transmit ? (kShTransmit0 << k) : 0u);
    }
};

// Distance to a shape-light sample, shortened by SHADOW_RAY_CLAMP
// (src/Shading.cu:337).
__device__ __forceinline__ float shadow_tmax(f3 pos, f3 ldir, f3 lpos, f3 lerr, f3 lng)
{
    return length(offset_ray_origin(lpos, lerr, -ldir, lng) - pos) * kShadowRayClamp;
}

// kVolume: volume scattering vertices (Ray_shading_path_tracing's volume branch,
// src/Shading.cu:2070-2130, with EvalVolumeDistantLight 202-290 and
// EvalVolumeShapeLight 419-513); otherwise surface vertices (2132-2302 with
// EvalDistantLight 83-198 and EvalShapeLight 294-417).
// kGraph: the scene has procedural texture nodes or normal / bump maps (the
// variant without them keeps the image-texture fast path only).  kClass:
// kMatDiffuse or kMatMetal shades the hits on materials of that class (their
// own queue) with the lobes the class leaves fixed at compile time, which
// gives the general variant's floats with fewer live registers.  The
// variants without the graph evaluator are held to 168 VGPRs (3 waves per
// SIMD, a few spilled registers): the shading stage waits on dependent
// loads, and the third wave hides more of them than the spills cost (6 %
// faster on the interior frame; 4 waves spill too much).
// kAdj: the adjoint's replay pass (surface vertices): albedo, texel and
// roughness gradient events.
//
// LDS of a shading wave: the output queues' stage, the texture graph's value
// stack and the adjoint's sums.
struct ShadeLds {
    uint32_t *stage;
    float *tex, *adj;
};

template <bool kVolume, bool kGraph, uint32_t kClass = kMatGeneral, bool kAdj = false>
__device__ __forceinline__ void shade_body(const ShadeLds &lds, const DevScene &sc, const PtParams &prm,
                                           const PathState &ps, uint32_t pass, const Share &share)
{
    AdjSums<kAdj> sums{lds.adj, &prm.adj};
    sums.begin();
    uint32_t *cnt = prm.counters + pass * kCtrStride;
    uint32_t *cnt_next = prm.counters + (pass + 1) * kCtrStride;
    constexpr bool kDiffuse = kClass == kMatDiffuse, kMetal = kClass == kMatMetal;
    const uint32_t n = cnt[kVolume ? kCtrHitVol : kDiffuse ? kCtrHitDiffuse : kMetal ? kCtrHitMetal : kCtrHit];
    const uint32_t *q = kVolume ? ps.q_hit_vol : kDiffuse ? ps.q_hit_diffuse : kMetal ? ps.q_hit_metal : ps.q_hit;
    const ymrt_render_settings &rs = prm.rs;
    const uint32_t cap = prm.cap;
    uint32_t *const ctrs[2] = {cnt + kCtrShadow, cnt_next + kCtrActive};
    uint32_t *const qs[2] = {ps.q_shadow, ps.queue[(pass + 1) & 1]};
    constexpr uint32_t kLobes = kDiffuse ? 1u << kSlotDiffuse
                                : kMetal ? (1u << kSlotMetal) | (1u << kSlotDiffuse)
                                         : 0u;
    run_items<2>(lds.stage, share, cnt + (kVolume     ? kCtrWorkShadeVol
                        : kDiffuse ? kCtrWorkShadeDiffuse
                        : kMetal   ? kCtrWorkShadeMetal
                                   : kCtrWorkShade),
                 n, ctrs, qs,
                 [&](uint32_t i, uint32_t &p, bool(&out)[2]) {
        {
            p = q[i];
            const float4 bi = *ps.beta(p);
            uint32_t info = __float_as_uint(bi.w);
            int depth = info_depth(info);
            bool never_scatter = (info & kInfoNeverScatter) != 0;
            const uint32_t vertex = info_vertex(info) + 1;
            const uint4 ha = *ps.hit_a(p);
            const float4 hb = *ps.hit_b(p);
            const f3 ray_d = xyz(*ps.ray_d(p));
            f3 beta = xyz(bi);
            Sampler smp = load_sampler(ps, p);
            ShadowEmit so{ps, p, (uint32_t)depth << kShDepthShift | sh_vertex_bits(vertex)};
            bool alive = false;       // a next extension ray
            f3 emitted = s3(0.0f);    // radiance of a light the path ends on
            const f3 sh_beta = beta;
            float sel_pdf = 0.0f;
            f3 next_o = s3(0.0f), next_d = s3(0.0f);
            uint32_t next_li = kEmpty, next_lt = kEmpty;
            bool pending = false;
            if constexpr (kVolume) {
                const Transfer t = load_transfer(ps, p, cap);
                int vi[kMaxBoundaryRecord];
                float gs[kMaxBoundaryRecord], vw[kMaxBoundaryRecord];
                const int nv = t.volumes(vi, sc.volume_count);
#pragma unroll
                for (int k = 0; k < kMaxBoundaryRecord; ++k) {
                    gs[k] = k < nv ? sc.volumes[vi[k]].g : 0.0f;
                    vw[k] = k < nv ? 1.0f / (float)nv : 0.0f;
                }
                const f3 vpos = xyz(hb);
                so.flags |= kShVolume;
                if (rs.enable_distant_light && sc.distant_count > 0 && nv > 0) {
                    const DevDistant &dl = sc.distant[pick_distant(sc.distant_count, sampler_next(sc, smp))];
                    {
                        f3 ldir = s3(0.0f), Li = s3(0.0f);
                        float lpdf = 0.0f;
                        const float u0 = sampler_next(sc, smp);
                        const float u1 = sampler_next(sc, smp);
                        distant_sample_li(dl, u0, u1, ldir, Li, lpdf);
                        float wpdf = 0.0f;
                        const float ph = mixed_phase_eval(vw, gs, nv, -ray_d, ldir, wpdf);
                        if (ph > kMinColorEpsilon)
                            so.emit(2, vpos, ldir, kTMax, false, s3(gmin(ph, kMaxColorClamp)),
                                    min3(Li, s3(kMaxColorClamp)), power_heuristic(lpdf, wpdf));
                    }
                    {
                        f3 pwi = s3(0.0f);
                        float ppdf = 0.0f, pw = 0.0f;
                        const float u0 = sampler_next(sc, smp);
                        const float u1 = sampler_next(sc, smp);
                        if (mixed_phase_sample(vw, gs, nv, u0, u1, -ray_d, pw, pwi, ppdf)) {
                            float lpdf = 0.0f;
                            const f3 Li = distant_eval_li(dl, pwi, lpdf);
                            if (maxcomp(Li) > kMinColorEpsilon)
                                so.emit(3, vpos, pwi, kTMax, false, s3(gmin(pw, kMaxColorClamp)),
                                        min3(Li, s3(kMaxColorClamp)), power_heuristic(ppdf, lpdf));
                        }
                    }
                }
                if (rs.enable_shape_light && sc.light_count > 0 && nv > 0) {
                    const int li = sample_light_power(sc, sampler_next(sc, smp), sel_pdf);
                    const DevLightRec &light = sc.light_recs[li];
                    {
                        f3 ldir = s3(0.0f), lpos = s3(0.0f), lerr = s3(0.0f), lng = s3(0.0f), Li = s3(0.0f);
                        float lpdf = 0.0f;
                        const float u0 = sampler_next(sc, smp);
                        const float u1 = sampler_next(sc, smp);
                        const bool valid = light_sample_li(light, vpos, u0, u1, ldir, lpos, lerr, lng, Li, lpdf);
                        float wpdf = 0.0f;
                        const float ph = mixed_phase_eval(vw, gs, nv, -ray_d, ldir, wpdf);
                        if (ph > kMinColorEpsilon && valid)
                            so.emit(0, vpos, ldir, shadow_tmax(vpos, ldir, lpos, lerr, lng), false,
                                    s3(gmin(ph, kMaxColorClamp)), min3(Li, s3(kMaxColorClamp)),
                                    power_heuristic(lpdf, wpdf));
                    }
                    {
                        f3 pwi = s3(0.0f);
                        float ppdf = 0.0f, pw = 0.0f;
                        const float u0 = sampler_next(sc, smp);
                        const float u1 = sampler_next(sc, smp);
                        if (mixed_phase_sample(vw, gs, nv, u0, u1, -ray_d, pw, pwi, ppdf)) {
                            f3 lpos = s3(0.0f), lerr = s3(0.0f), lng = s3(0.0f);
                            float lpdf = 0.0f;
                            const f3 Li = light_eval_li(light, vpos, pwi, lpos, lerr, lng, lpdf);
                            if (maxcomp(Li) > kMinColorEpsilon)
                                so.emit(1, vpos, pwi, shadow_tmax(vpos, pwi, lpos, lerr, lng), false,
                                        s3(gmin(pw, kMaxColorClamp)), min3(Li, s3(kMaxColorClamp)),
                                        power_heuristic(ppdf, lpdf));
                        }
                    }
                }
                f3 wi = s3(0.0f);
                float pdf = 0.0f, pw = 0.0f;
                const float u0 = sampler_next(sc, smp);
                const float u1 = sampler_next(sc, smp);
                if (mixed_phase_sample(vw, gs, nv, u0, u1, -ray_d, pw, wi, pdf)) {
                    beta = beta * pw;
                    const float rr = gmin(gmax(beta.x, gmax(beta.y, beta.z)), 1.0f);
                    bool cont = true;
                    if (depth + 1 > rs.ray_depth) {
                        if (rs.enable_russian_roulette && sampler_next(sc, smp) < rr) beta = beta / gmax(rr, kMinColorEpsilon);
                        else cont = false;
                    }
                    if (cont && depth + 1 <= kMaxRayDepth) {
                        alive = true;
                        next_o = vpos;
                        next_d = normalize(wi);
                        never_scatter = false;
                        depth += 1;
                    }
                }
            } else {
                const uint32_t inst = ha.y, tri = ha.z;
                const int back = (ha.w & kHitBack) ? 1 : 0;
                const DevInstance &in = sc.instances[inst];
                const uint32_t iflags = in.flags;
                const bool is_sphere = (iflags & kInstSphere) != 0;
                const ShadeTri &st = sc.shade[in.shade_base + (is_sphere ? 0u : tri)];
                const f3 b{hb.x, hb.y, hb.z};
                f3 p0 = s3(0.0f), p1 = s3(0.0f), p2 = s3(0.0f);
                f3 pos, perr, ng;
                const float radius = gmax(in.radius, kFloatEpsilon);
                if (is_sphere) {
                    // FetchSphereShadingData (src/ShadingUtilities.cuh:636-711)
                    pos = b;
                    perr = error_gamma(5) * abs3(b);
                    ng = b / radius;
                } else {
                    p0 = f3{st.p[0], st.p[1], st.p[2]};
                    p1 = f3{st.p[3], st.p[4], st.p[5]};
                    p2 = f3{st.p[6], st.p[7], st.p[8]};
                    const float xs = fabsf(p0.x * b.x) + fabsf(p1.x * b.y) + fabsf(p2.x * b.z);
                    const float ys = fabsf(p0.y * b.x) + fabsf(p1.y * b.y) + fabsf(p2.y * b.z);
                    const float zs = fabsf(p0.z * b.x) + fabsf(p1.z * b.y) + fabsf(p2.z * b.z);
                    pos = interp3(p0, p1, p2, b);
                    perr = error_gamma(7) * f3{xs, ys, zs};
                    ng = cross(p1 - p0, p2 - p0);
                }
                const DevMaterial &m = sc.materials[in.material];
                const uint32_t mtype = m.type;
                uint32_t prio;
                fetch_ior(m, &prio);
                // the medium records give the pass-through test and the two
                // IORs; nothing later needs the records themselves
                float ray_ior, ex_ior;
                bool pass_through;
                {
                    const Transfer t = load_transfer(ps, p, cap);
                    pass_through = (t.count != 0 && prio < t.get(t.max_idx).priority) || (iflags & kInstBoundary);
                    ray_ior = t.ray_ior();
                    ex_ior = t.ex_ior(inst);
                }
                if (pass_through || mtype == YMRT_MATERIAL_LIGHT) {
                    pos = xf_position(in.o2w, pos, &perr);
                    ng = normalize(xf_transpose_vector(in.w2o, ng));
                }
                if (pass_through) {
                    // pass through without consuming depth; the medium records
                    // change at the start of the next extend
                    pending = true;
                    alive = true;
                    next_o = offset_ray_origin(pos, perr, ray_d, ng);
                    next_d = normalize(ray_d);
                    next_li = inst;
                    next_lt = tri;
                } else if (mtype == YMRT_MATERIAL_LIGHT) {
                    if (never_scatter)
                        emitted = light_clamp(rs, beta * f3{m.light_color[0], m.light_color[1], m.light_color[2]} *
                                                      m.intensity,
                                              depth);
                } else {
                    f3 sn, dpdu, dpdv;
                    f2 uv;
                    if (is_sphere) {
                        sn = ng;
                        const float theta = ym_acosf(ng.y);
                        float phi = ym_atan2f(ng.z, ng.x);
                        if (phi < 0.0f) phi += kTwoPi;
                        uv = f2{0.5f * phi * kInvPi, theta * kInvPi};
                        float sin_theta = 0.0f;
                        if (1.0f - ng.y * ng.y > 0.0f) sin_theta = sqrtf(1.0f - ng.y * ng.y);
                        float cos_phi = 1.0f, sin_phi = 0.0f;
                        if (sin_theta > 0.0f) {
                            cos_phi = ng.x / sin_theta;
                            sin_phi = ng.z / sin_theta;
                        }
                        dpdu = f3{-b.z, 0.0f, b.x} * kTwoPi;
                        dpdv = f3{b.y * cos_phi, -radius * sin_theta, sin_phi * b.y} * kPi;
                    } else {
                        sn = (iflags & kInstNoNormals)
                                 ? ng
                                 : interp3(f3{st.n[0], st.n[1], st.n[2]}, f3{st.n[3], st.n[4], st.n[5]},
                                           f3{st.n[6], st.n[7], st.n[8]}, b);
                        const f2 uv0{st.uv[0], st.uv[1]}, uv1{st.uv[2], st.uv[3]}, uv2{st.uv[4], st.uv[5]};
                        uv = f2{uv0.x * b.x + uv1.x * b.y + uv2.x * b.z, uv0.y * b.x + uv1.y * b.y + uv2.y * b.z};
                        float du01 = uv1.x - uv0.x, dv01 = uv1.y - uv0.y, du02 = uv2.x - uv0.x, dv02 = uv2.y - uv0.y;
                        float det = du01 * dv02 - dv01 * du02;
                        if (fabsf(det) < 1E-8f) {
                            du01 = 1.0f;
                            dv01 = 0.0f;
                            du02 = 0.0f;
                            dv02 = 1.0f;
                            det = 1.0f;
                        }
                        const float idet = 1.0f / det;
                        const f3 dp01 = p1 - p0, dp02 = p2 - p0;
                        dpdu = (dv02 * dp01 - dv01 * dp02) * idet;
                        dpdv = (-du02 * dp01 + du01 * dp02) * idet;
                    }
                    const f3 pos_obj = pos;
                    pos = xf_position(in.o2w, pos, &perr);
                    sn = normalize(xf_transpose_vector(in.w2o, sn));
                    ng = normalize(xf_transpose_vector(in.w2o, ng));
                    dpdu = xf_vector(in.o2w, dpdu);
                    dpdv = xf_vector(in.o2w, dpdv);
                    const bool is_default = mtype == YMRT_MATERIAL_DEFAULT;
                    const uint32_t normal_tex = kGraph && is_default ? m.normal_mapping_tex : kEmpty;
                    const uint32_t bump_tex = kGraph && is_default && normal_tex == kEmpty ? m.bump_mapping_tex : kEmpty;
                    TexEval<kGraph> tx{sc, TexCoord{uv, pos, pos_obj}, lds.tex, (int)lane_id()};
                    float4 duv = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                    if (bump_tex != kEmpty)
                        duv = camera_uv_differentials(sc.camera, pos, sn, ng, dpdu, dpdv, rs.width, rs.height, 0.25f,
                                                      0.25f);
                    Bsdf bs;
                    init_shading_space(bs, tx, normal_tex, bump_tex, back, ray_d, ng, sn, dpdu, dpdv, in.w2o, duv);
                    bs.mask = 0;
                    if (is_default) init_default_bsdf<kClass>(tx, bs, m, ray_d, back, ray_ior, ex_ior);
                    // adjoint replay: an albedo or texel factor of this vertex
                    // scales every later deposit of the path (next-event ones
                    // included); a target roughness scales each next-event ray
                    // by its own BSDF value and the continuation by its own
                    int32_t rough_entry = -1;
                    float rough_r = 0.0f, adj_gc = 0.0f;
                    f3 adj_dl = s3(0.0f);
                    if constexpr (kAdj) {
                        const AdjParams &A = prm.adj;
                        const int32_t as = A.alb_slot[in.material];
                        const bool tex_on = A.tex != kEmpty && m.diffuse_albedo_tex == A.tex;
                        rough_entry = A.rough_slot[in.material];
                        if (as >= 0 || tex_on || rough_entry >= 0)
                            adj_dl = adj_pixel(prm, p) * (xyz(ps.out[p]) - xyz(*ps.L(p)));
                        if (as >= 0) {
#pragma unroll
                            for (int c = 0; c < 3; ++c) {
                                const float al = m.diffuse_albedo[c];
                                if (al > 0.0f) sums.albedo((uint32_t)as, c, comp(adj_dl, c) / al);
                            }
                        }
                        if (tex_on) adj_texels(sc, A, uv, adj_dl);
                        if (rough_entry >= 0) rough_r = m.roughness_x;
                    }
                    const f3 wo = bs.to_local(-ray_d);
                    if (rs.enable_distant_light && sc.distant_count > 0) {
                        const DevDistant &dl = sc.distant[pick_distant(sc.distant_count, sampler_next(sc, smp))];
                        {
                            f3 ldir = s3(0.0f), Li = s3(0.0f);
                            float lpdf = 0.0f;
                            const float u0 = sampler_next(sc, smp);
                            const float u1 = sampler_next(sc, smp);
                            distant_sample_li(dl, u0, u1, ldir, Li, lpdf);
                            const f3 lwi = bs.to_local(ldir);
                            float wpdf = 0.0f;
                            const f3 f = bsdf_eval<kLobes>(bs, wo, lwi, wpdf);
                            if (maxcomp(f) > kMinColorEpsilon) {
                                const bool transmit = dot(-ray_d, ng) * dot(ldir, ng) < 0.0f;
                                const bool invalid = (!same_hemi(wo, lwi) && !transmit) || (same_hemi(wo, lwi) && transmit);
                                if (!invalid)
                                    so.emit(2, offset_ray_origin(pos, perr, ldir, ng), ldir, kTMax, transmit,
                                            min3(f, s3(kMaxColorClamp)), min3(Li, s3(kMaxColorClamp)),
                                            power_heuristic(lpdf, wpdf),
                                            rough_entry >= 0 ? ggx_rough_dlog(rough_r, wo, lwi) : 0.0f);
                            }
                        }
                        {
                            f3 bw = s3(0.0f), bwi = s3(0.0f);
                            float bpdf = 0.0f;
                            const float u0 = sampler_next(sc, smp);
                            const float u1 = sampler_next(sc, smp);
                            const float u2 = sampler_next(sc, smp);
                            if (bsdf_sample<kLobes>(bs, wo, bw, bwi, bpdf, u0, u1, u2)) {
                                const f3 ldir = bs.to_world(bwi);
                                float lpdf = 0.0f;
                                const f3 Li = distant_eval_li(dl, ldir, lpdf);
                                if (maxcomp(Li) > kMinColorEpsilon) {
                                    const bool transmit = dot(-ray_d, ng) * dot(ldir, ng) < 0.0f;
                                    const bool invalid =
                                        (!same_hemi(wo, bwi) && !transmit) || (same_hemi(wo, bwi) && transmit);
                                    if (!invalid)
                                        so.emit(3, offset_ray_origin(pos, perr, ldir, ng), ldir, kTMax, transmit,
                                                min3(bw, s3(kMaxColorClamp)), min3(Li, s3(kMaxColorClamp)),
                                                power_heuristic(bpdf, lpdf),
                                                rough_entry >= 0 ? ggx_rough_dlog(rough_r, wo, bwi) : 0.0f);
                                }
                            }
                        }
                    }
                    if (rs.enable_shape_light && sc.light_count > 0) {
                        const int li = sample_light_power(sc, sampler_next(sc, smp), sel_pdf);
                        const DevLightRec &light = sc.light_recs[li];
                        {
                            f3 ldir = s3(0.0f), lpos = s3(0.0f), lerr = s3(0.0f), lng = s3(0.0f), Li = s3(0.0f);
                            float lpdf = 0.0f;
                            const float u0 = sampler_next(sc, smp);
                            const float u1 = sampler_next(sc, smp);
                            const bool valid = light_sample_li(light, pos, u0, u1, ldir, lpos, lerr, lng, Li, lpdf);
                            const f3 lwi = bs.to_local(ldir);
                            float wpdf = 0.0f;
                            const f3 f = bsdf_eval<kLobes>(bs, wo, lwi, wpdf);
                            if (maxcomp(f) > kMinColorEpsilon && valid) {
                                const bool transmit = dot(-ray_d, ng) * dot(ldir, ng) < 0.0f;
                                const bool invalid = (!same_hemi(wo, lwi) && !transmit) || (same_hemi(wo, lwi) && transmit);
                                if (!invalid)
                                    so.emit(0, offset_ray_origin(pos, perr, ldir, ng), ldir,
                                            shadow_tmax(pos, ldir, lpos, lerr, lng), transmit,
                                            min3(f, s3(kMaxColorClamp)), min3(Li, s3(kMaxColorClamp)),
                                            power_heuristic(lpdf, wpdf),
                                            rough_entry >= 0 ? ggx_rough_dlog(rough_r, wo, lwi) : 0.0f);
                            }
                        }
                        {
                            f3 bw = s3(0.0f), bwi = s3(0.0f);
                            float bpdf = 0.0f;
                            const float u0 = sampler_next(sc, smp);
                            const float u1 = sampler_next(sc, smp);
                            const float u2 = sampler_next(sc, smp);
                            if (bsdf_sample<kLobes>(bs, wo, bw, bwi, bpdf, u0, u1, u2)) {
                                const f3 ldir = bs.to_world(bwi);
                                f3 lpos = s3(0.0f), lerr = s3(0.0f), lng = s3(0.0f);
                                float lpdf = 0.0f;
                                const f3 Li = light_eval_li(light, pos, ldir, lpos, lerr, lng, lpdf);
                                if (maxcomp(Li) > kMinColorEpsilon) {
                                    const bool transmit = dot(-ray_d, ng) * dot(ldir, ng) < 0.0f;
                                    const bool invalid =
                                        (!same_hemi(wo, bwi) && !transmit) || (same_hemi(wo, bwi) && transmit);
                                    if (!invalid)
                                        so.emit(1, offset_ray_origin(pos, perr, ldir, ng), ldir,
                                                shadow_tmax(pos, ldir, lpos, lerr, lng), transmit,
                                                min3(bw, s3(kMaxColorClamp)), min3(Li, s3(kMaxColorClamp)),
                                                power_heuristic(bpdf, lpdf),
                                                rough_entry >= 0 ? ggx_rough_dlog(rough_r, wo, bwi) : 0.0f);
                                }
                            }
                        }
                    }
                    f3 wi = s3(0.0f), bw = s3(0.0f);
                    float pdf = 0.0f;
                    const float u0 = sampler_next(sc, smp);
                    const float u1 = sampler_next(sc, smp);
                    const float u2 = sampler_next(sc, smp);
                    if (bsdf_sample<kLobes>(bs, wo, bw, wi, pdf, u0, u1, u2)) {
                        if constexpr (kAdj) {
                            if (rough_entry >= 0) {
                                adj_gc = ggx_rough_dlog(rough_r, wo, wi);
                                sums.roughness((uint32_t)rough_entry, (adj_dl.x + adj_dl.y + adj_dl.z) * adj_gc);
                            }
                        }
                        beta = beta * bw;
                        const float rr = gmin(gmax(beta.x, gmax(beta.y, beta.z)), 1.0f);
                        bool cont = true;
                        if (depth + 1 > rs.ray_depth) {
                            if (rs.enable_russian_roulette && sampler_next(sc, smp) < rr) beta = beta / gmax(rr, kMinColorEpsilon);
                            else cont = false;
                        }
                        if (cont) {
                            const f3 nd = bs.to_world(wi);
                            const bool transmit = dot(-ray_d, ng) * dot(nd, ng) < 0.0f;
                            const bool invalid = (!same_hemi(wo, wi) && !transmit) || (same_hemi(wo, wi) && transmit);
                            if (!invalid && depth + 1 <= kMaxRayDepth) {
                                pending = transmit;
                                alive = true;
                                next_o = offset_ray_origin(pos, perr, nd, ng);
                                next_d = normalize(nd);
                                next_li = inst;
                                next_lt = tri;
                                never_scatter = false;
                                depth += 1;
                            }
                        }
                    }
                    // the shadow stage subtracts the continuation's factor from
                    // each next-event ray's own
                    if constexpr (kAdj)
                        ps.adj_g[p] = make_uint2(rough_entry >= 0 ? (uint32_t)rough_entry : kEmpty,
                                                 __float_as_uint(adj_gc));
                }
            }
            // ---------------------------------------------- write back
            const bool nee = (so.flags & kShActiveMask) != 0;
            store_sampler(ps, p, smp);
            if (nee) {
                out[0] = true;
                if (!alive) so.flags |= kShTerminate;
                ps.sh_flags[p] = so.flags;
                *ps.sh_c(p) = f4(sh_beta, sel_pdf);
            } else if (!alive) {
                // the path's radiance changes here only where it ends on a
                // light; elsewhere it stays in HBM (adding 0 to -0 gives the
                // same output as the reference's sum: a path's radiance
                // starts at +0)
                ps.out[p] = f4(xyz(*ps.L(p)) + emitted, 0.0f);
            }
            info = (uint32_t)depth | (never_scatter ? kInfoNeverScatter : 0u) | (pending ? kInfoPendingBunch : 0u) |
                   (vertex << 16);
            if (alive) {
                out[1] = true;
                *ps.ray_o(p) = f4(next_o, __uint_as_float(next_li));
                *ps.ray_d(p) = f4(next_d, __uint_as_float(next_lt));
                *ps.beta(p) = f4(beta, __uint_as_float(info));
            }
        }
    });
    sums.end();
}


template <bool kVolume, bool kGraph, uint32_t kClass, bool kAdj>
__device__ __forceinline__ uint32_t shade_class(const ShadeLds &lds, const FrameSlot *__restrict__ fs, uint32_t nfs,
                                                uint32_t pass, uint32_t rot)
{
    constexpr uint32_t kQueue = kVolume ? kCtrHitVol : kClass == kMatDiffuse ? kCtrHitDiffuse
                                : kClass == kMatMetal ? kCtrHitMetal : kCtrHit;
    constexpr uint32_t kWork = kVolume ? kCtrWorkShadeVol : kClass == kMatDiffuse ? kCtrWorkShadeDiffuse
                               : kClass == kMatMetal ? kCtrWorkShadeMetal : kCtrWorkShade;
    const uint32_t used = for_slots<kBlock, kBlock * kSub>(
        fs, nfs, [&](const FrameSlot &f) { return pass_counter(f, pass, kQueue); },
        [&](const FrameSlot &f) { return pass_work(f, pass, kWork); },
        [&](const FrameSlot &f, const Share &share) {
            shade_body<kVolume, kGraph, kClass, kAdj>(lds, f.sc, f.prm, f.ps, pass, share);
        },
        rot);
    return (rot + used) % gridDim.x;
}

// One shading class per launch.
template <bool kVolume, bool kGraph, uint32_t kClass = kMatGeneral, bool kAdj = false>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(kGraph ? 2 : 3))) void k_shade_m(const FrameSlot *__restrict__ fs, uint32_t nfs, uint32_t pass)
{
    __shared__ uint32_t stage[2 * kSub * kBlock];
    __shared__ float tex_stk[kGraph && !kVolume ? kTexStack * 3 * kBlock : 1];
    __shared__ float adj_lds[kAdj ? kAdjLds : 1];
    shade_class<kVolume, kGraph, kClass, kAdj>(ShadeLds{stage, tex_stk, adj_lds}, fs, nfs, pass, 0);
}

// All shading classes of a pass in one launch, and with kMedia the volume
// vertices: for short queues and for frames with texture graphs
// (launch_multi_shade).  Launched one after another, each class is a chain of
// dependent loads of 25-35 us, on a short queue with most of the GPU idle; here
// a class' waves are others than those the classes before it took.
template <bool kMedia, bool kGraph = false>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(kGraph ? 2 : 3))) void k_shade_all_m(const FrameSlot *__restrict__ fs, uint32_t nfs, uint32_t pass)
{
    __shared__ uint32_t stage[2 * kSub * kBlock];
    __shared__ float tex_stk[kGraph ? kTexStack * 3 * kBlock : 1];
    const ShadeLds lds{stage, tex_stk, nullptr};
    uint32_t rot = shade_class<false, kGraph, kMatGeneral, false>(lds, fs, nfs, pass, 0);
    rot = shade_class<false, kGraph, kMatMetal, false>(lds, fs, nfs, pass, rot);
    rot = shade_class<false, kGraph, kMatDiffuse, false>(lds, fs, nfs, pass, rot);
    if constexpr (kMedia) shade_class<true, false, kMatGeneral, false>(lds, fs, nfs, pass, rot);
}



// ------------------------------------------------------------ shadow
// NEE contribution of a path's shadow rays: per light kind, the sum of
// mis * tr * f * Li over the rays that reached the light (ShadowSum::add, in
// slot order within a kind), divided by the light-selection pdf, clamped and
// deposited (shadow_deposit), distant light first (EvalDistantLight,
// src/Shading.cu:83-198, then EvalShapeLight 294-417, as the shading stage
// adds them at 2217-2240).  kAdj (the adjoint's replay): at a surface vertex
// with a target roughness, each ray's deposit D adds adj . D * (g_ray -
// g_continuation) to that roughness's gradient (the continuation's event
// counted D with the continuation's factor).
template <bool kAdj>
struct ShadowSum {
    f3 shape = s3(0.0f), dist = s3(0.0f);
    f3 rc[kAdj ? kShadowSlots : 1];
    float rg[kAdj ? kShadowSlots : 1];
    __device__ __forceinline__ ShadowSum()
    {
        if constexpr (kAdj)
            static_for<0, kShadowSlots>([&](auto K) {
                rc[K()] = s3(0.0f);
                rg[K()] = 0.0f;
            });
    }
    // shadow ray k of path p reached its light with transmittance tr; returns
    // its term
    __device__ __forceinline__ f3 add(const PathState &ps, uint32_t p, int k, f3 tr)
    {
        const float4 f4v = ps.shadow(k, p)[2];
        const float4 li4 = ps.shadow(k, p)[3];
        const f3 c = ((f4v.w * tr) * xyz(f4v)) * xyz(li4);
        if (k < 2) shape = shape + c;
        else dist = dist + c;
        if constexpr (kAdj)
            static_for<0, kShadowSlots>([&](auto K) {
                if (K() == k) {
                    rc[K()] = c;
                    rg[K()] = li4.w;
                }
            });
        return c;
    }
};

template <bool kAdj>
__device__ __forceinline__ void shadow_deposit(const PtParams &prm, const PathState &ps, uint32_t p, uint32_t fl,
                                               uint32_t distant_count, const ShadowSum<kAdj> &sum,
                                               AdjSums<kAdj> *sums)
{
    const float4 c4 = *ps.sh_c(p);
    const f3 beta = xyz(c4);
    if constexpr (kAdj) {
        if (!(fl & kShVolume)) {
            const uint2 ag = ps.adj_g[p];
            if (ag.x != kEmpty) {
                const float gc = __uint_as_float(ag.y);
                const f3 a = adj_pixel(prm, p);
                float acc = 0.0f;
                static_for<0, kShadowSlots>([&](auto K) {
                    const float scale = K() < 2 ? safe_rcp(c4.w) : (float)distant_count;
                    const f3 d = beta * (sum.rc[K()] * scale);
                    acc += dot(a, d) * (sum.rg[K()] - gc);
                });
                sums->roughness(ag.x, acc);
            }
        }
    }
    const int depth = (int)((fl >> kShDepthShift) & 0xFFu);
    f3 L = xyz(*ps.L(p));
    if (distant_count > 0) L = L + light_clamp(prm.rs, beta * (sum.dist / (1.0f / (float)distant_count)), depth);
    // EvalShapeLight returns direct * SafeRcp(select pdf); the volume variant
    // divides when the pdf is positive.
    const f3 sel = (fl & kShVolume) ? (c4.w > 0.0f ? sum.shape / c4.w : s3(0.0f)) : sum.shape * safe_rcp(c4.w);
    L = L + light_clamp(prm.rs, beta * sel, depth);
    if (fl & kShTerminate) ps.out[p] = f4(L, 0.0f);
    else *ps.L(p) = f4(L, 0.0f);
}

// Any-hit for each shadow ray against non-boundary instances
// (BVHTraverseShadow, src/ShadingUtilities.cuh:563-635).  In scenes with media,
// paths with an unoccluded ray go on to k_transmit for the transmittance along
// it; the others are finished here.
template <bool kMedia, bool kSphere, int kStack, bool kAdj = false>
__device__ __forceinline__ void shadow_body(const DevScene &sc, const PtParams &prm, const PathState &ps, uint32_t pass,
                                            const Share &share)
{
    __shared__ uint32_t stack[kStackWindow * kBlock];
    __shared__ float pre_park[kPreSlots * kBlock];
    __shared__ float adj_lds[kAdj ? kAdjLds : 1];
    AdjSums<kAdj> sums{adj_lds, &prm.adj};
    sums.begin();
    uint32_t *cnt = prm.counters + pass * kCtrStride;
    LaneScratch<kBlock, kStackWindow, true> ls{stack, nullptr, nullptr, nullptr, (int)lane_id(), ps.spill,
                                               ps.spill_threads, blockIdx.x * kBlock + threadIdx.x, pre_park};
    uint32_t nsh = 0;
    TraceCounters tc{0, 0};
    RefillRange<16> rr(share, cnt + kCtrWorkShadow, cnt[kCtrShadow]);

    // one lane walks its path's recorded rays (slots k) in order
    const TravScene ts(sc);
    Traversal<kModeSkipBoundary, true, false, true, kSphere, kStack> tv;
    uint32_t p = 0, fl = 0;
    int k = 0;
    int r = kLaneIdle;
    auto start_ray = [&]() {
        const float4 o4 = gload(ps.shadow(k, p));
        const float4 d4 = gload(ps.shadow(k, p) + 1);
        Query q;
        q.o = xyz(o4);
        q.d = xyz(d4);
        q.tmin = kTMin;
        q.tmax = o4.w;
        q.last_inst = kEmpty;
        q.last_tri = kEmpty;
        r = tv.init(sc, q);
    };
    for (;;) {
        uint32_t item = 0;
        if (rr.more && rr.refill(r == kLaneIdle, item)) {
            p = gload(ps.q_shadow + item);
            fl = gload(ps.sh_flags + p);
            k = __builtin_ctz(fl & kShActiveMask);  // a queued path records at least one ray
            start_ray();
        }
        const uint32_t want = rr.want();
        for (;;) {
            const uint64_t busy = __ballot(r == kTravContinue);
            if (busy == 0 || (uint32_t)(kBlock - __popcll(busy)) >= want) break;
            wave_step<24, false>(tv, r, ts, ls, tc);
        }
        // finished rays: note the result, start the path's next ray or
        // finish the path (a ray can end in init, hence the loop)
        while (r != kTravContinue && r != kLaneIdle) {
            ++nsh;
            if (r == kTravOverflow) atomicOr(prm.error, 1u);
            if (r == kTravMiss) fl |= kShClear0 << k;
            const uint32_t rest = fl & kShActiveMask & ~((2u << k) - 1u);
            if (rest) {
                k = __builtin_ctz(rest);
                start_ray();
            } else {
                r = kLaneIdle;
                const bool walk = kMedia && prm.media && (fl & kShClearMask);
                if (walk) {
                    ps.sh_flags[p] = fl;
                    ps.flag[p] = (pass << kFlagBits) | kFlagTransmit;
                } else {
                    ShadowSum<kAdj> sum;
                    static_for<0, kShadowSlots>([&](auto K) {
                        if ((fl & (1u << K())) && (fl & (kShClear0 << K()))) sum.add(ps, p, K(), s3(1.0f));
                    });
                    shadow_deposit<kAdj>(prm, ps, p, fl, sc.distant_count, sum, &sums);
                }
            }
        }
        if (!rr.more && __ballot(r != kLaneIdle) == 0) break;
    }
    sums.end();
    wave_add64(prm.stats + kStatShadow, nsh);
    wave_add64(prm.stats + kStatShadowNodes, tc.nodes);
    wave_add64(prm.stats + kStatShadowTris, tc.tris);
}


template <bool kMedia, bool kSphere, int kStack, bool kAdj = false>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(kAdj ? 4 : 5))) void k_shadow_m(const FrameSlot *__restrict__ fs, uint32_t nfs, uint32_t pass)
{
    for_slots<kBlock, kBlock * kSub>(
        fs, nfs, [&](const FrameSlot &f) { return pass_counter(f, pass, kCtrShadow); },
        [&](const FrameSlot &f) { return pass_work(f, pass, kCtrWorkShadow); },
        [&](const FrameSlot &f, const Share &share) {
            shadow_body<kMedia, kSphere, kStack, kAdj>(f.sc, f.prm, f.ps, pass, share);
        });
}



// Transmittance of the unoccluded shadow rays of paths in media: TraceTr
// (src/VolumeEval.cuh:420-468) walks the boundary instances along the ray,
// updating the medium records at each crossing and multiplying the segment
// transmittances (EvalTr, 253-418).
// kHet as k_medium's.  kAdj (the adjoint's replay): the shadow_finish
// roughness terms, and with a target grid volume each ray's ratio-tracking
// events, found by walking the ray a second time with the same random
// numbers once its deposit is known.
template <bool kSphere, int kStack, int kHet, bool kAdj = false>
__device__ __forceinline__ void transmit_body(const DevScene &sc, const PtParams &prm, const PathState &ps, uint32_t pass,
                                              const Share &share)
{
    __shared__ float tex_stk[kHet == 2 ? kTexStack * 3 * kBlock : 1];
    __shared__ uint32_t stack[kStackWindow * kBlock];
    __shared__ uint32_t nbp[kNearbyCap * kBlock];
    __shared__ float nbt[kNearbyCap * kBlock];
    __shared__ int nbb[kNearbyCap * kBlock];
    uint32_t *cnt = prm.counters + pass * kCtrStride;
    const uint32_t n = cnt[kCtrTransmit];
    const uint32_t cap = prm.cap;
    LaneScratch<kBlock, kStackWindow> ls{stack, nbp, nbt, nbb, (int)lane_id(), ps.spill, ps.spill_threads,
                                         blockIdx.x * kBlock + threadIdx.x};
    uint32_t ntr = 0;
    TraceCounters tc{0, 0};
    __shared__ float adj_lds[kAdj ? kAdjLds : 1];
    AdjSums<kAdj> sums{adj_lds, &prm.adj};
    sums.begin();
    run_items<0>(nullptr, share, cnt + kCtrWorkTransmit, n, nullptr, nullptr, [&](uint32_t i, uint32_t &slot, bool(&)[1]) {
        {
            const uint32_t p = ps.q_transmit[i];
            slot = p;
            const uint32_t fl = ps.sh_flags[p];
            HashRng rng;
            {
                // 64-bit like k_raygen: a frame may hold more than 2^32 path slots
                const uint64_t gp = prm.chunk_base + p;
                const uint32_t spp = (uint32_t)prm.rs.spp;
                const uint64_t vpix = gp / spp;
                const uint32_t s = (uint32_t)(gp - vpix * spp);
                const uint32_t tile = (uint32_t)(vpix >> 8), within = (uint32_t)(vpix & 255u);
                const uint32_t ty = tile / prm.tiles_x, tx = tile - ty * prm.tiles_x;
                const uint32_t px = tx * 16u + (within & 15u), py = ty * 16u + (within >> 4);
                rng.key[0] = py * prm.rs.width + px;
                rng.key[1] = sh_vertex(fl);
                rng.key[2] = s;
                rng.key[3] = (uint32_t)prm.frame;
                rng.ctr = 0;
            }
            ShadowSum<kAdj> sum;
            // distant-light rays first, as the shading stage evaluates them
#pragma unroll 1
            for (int j = 0; j < kShadowSlots; ++j) {
                const int k = (j + 2) & 3;
                if (!(fl & (1u << k)) || !(fl & (kShClear0 << k))) continue;
                auto walk = [&](auto &&ev) -> f3 {
                    const float4 o4 = ps.shadow(k, p)[0];
                    const float4 d4 = ps.shadow(k, p)[1];
                    f3 tr = s3(1.0f);
                    // the vertex's records and nearby list are reloaded per ray
                    // rather than held across the loop (fewer live registers)
                    Transfer t = load_transfer(ps, p, cap);
                    if (fl & (kShTransmit0 << k)) boundary_bunch(sc, t, load_nearby(ps, p, cap, *ps.hit_a(p)));
                    Query tq;
                    tq.o = xyz(o4);
                    tq.d = xyz(d4);
                    tq.tmin = kTMin;
                    tq.tmax = o4.w;
                    // a vertex with shadow rays lies on no boundary (those
                    // are passed through), so there is no triangle to skip
                    tq.last_inst = kEmpty;
                    tq.last_tri = kEmpty;
                    const float maxd = o4.w;
                    float traced = kTMin;
                    int guard = 0;
                    while (traced < maxd) {
                        Hit bh;
                        bh.back = 0;
                        int bnc = 0;
                        int br = 0;
                        ++ntr;
                        if (sc.has_boundaries)
                            br = traverse<kModeBoundaryOnly, false, true, true, kSphere, kStack>(sc, tq, bh, bnc, ls, tc);
                        if (br < 0) {
                            atomicOr(prm.error, 1u);
                            break;
                        }
                        if (br == 0) {
                            tr = tr * eval_tr<kHet>(sc, tq.o, tq.d, t, gmax(maxd - traced, 0.0f), rng, tex_stk, ev);
                            break;
                        }
                        tr = tr * eval_tr<kHet>(sc, tq.o, tq.d, t, bh.t, rng, tex_stk, ev);
                        traced += bh.t;
                        f3 bp, bperr, bng;
                        hit_geometry(sc, bh.inst, bh.tri, bh.b0, bh.b1, bh.b2, bp, bperr, bng);
                        NearbyList bnb;
                        bnb.n = bnc;
                        static_for<0, kNearbyMax>([&](auto J) {
                            bnb.prim[J()] = nbp[J() * kBlock + lane_id()];
                            bnb.t[J()] = nbt[J() * kBlock + lane_id()];
                            bnb.back[J()] = nbb[J() * kBlock + lane_id()];
                        });
                        boundary_bunch(sc, t, bnb);
                        // the next segment is a new Ray, direction renormalised
                        tq.o = offset_ray_origin(bp, bperr, tq.d, bng);
                        tq.d = normalize(tq.d);
                        tq.tmax = kTMax;
                        tq.last_inst = bh.inst;
                        tq.last_tri = bh.tri;
                        if (++guard > 64) break;
                    }
                    return tr;
                };
                const uint32_t ctr0 = rng.ctr;
                const f3 tr = walk(NoTrackEvents{});
                const f3 c = sum.add(ps, p, k, tr);
                if constexpr (kAdj && kHet > 0) {
                    if (prm.adj.vol != kEmpty) {
                        // this ray's deposit, as shadow_deposit sums it
                        const float4 c4 = *ps.sh_c(p);
                        const float scale = k >= 2 ? (float)sc.distant_count
                                            : (fl & kShVolume) ? (c4.w > 0.0f ? 1.0f / c4.w : 0.0f)
                                                               : safe_rcp(c4.w);
                        const float d = dot(adj_pixel(prm, p), xyz(c4) * (c * scale));
                        if (d != 0.0f) {
                            const uint32_t ctr1 = rng.ctr;
                            rng.ctr = ctr0;
                            AdjTrackEvents ev = adj_track(sc, prm.adj, d, kAdjRayEvents);
                            (void)walk(ev);
                            rng.ctr = ctr1;
                        }
                    }
                }
            }
            shadow_deposit<kAdj>(prm, ps, p, fl, sc.distant_count, sum, &sums);
        }
    });
    sums.end();
    wave_add64(prm.stats + kStatTransmittance, ntr);
    wave_add64(prm.stats + kStatTransmitNodes, tc.nodes);
    wave_add64(prm.stats + kStatTransmitTris, tc.tris);
}


template <bool kSphere, int kStack, int kHet, bool kAdj = false>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(kHet == 0 ? 3 : kHet == 1 ? 2 : 1))) void k_transmit_m(const FrameSlot *__restrict__ fs, uint32_t nfs, uint32_t pass)
{
    for_slots<kBlock, kBlock * kSub>(
        fs, nfs, [&](const FrameSlot &f) { return pass_counter(f, pass, kCtrTransmit); },
        [&](const FrameSlot &f) { return pass_work(f, pass, kCtrWorkTransmit); },
        [&](const FrameSlot &f, const Share &share) {
            transmit_body<kSphere, kStack, kHet, kAdj>(f.sc, f.prm, f.ps, pass, share);
        });
}



// ------------------------------------------------------------ flush
// Paths still queued after the last pass end with the radiance they carry.
__device__ __forceinline__ void flush_body(const PtParams &prm, const PathState &ps, uint32_t pass)
{
    uint32_t *cnt = prm.counters + pass * kCtrStride;
    const uint32_t n = cnt[kCtrActive];
    const uint32_t *q = ps.queue[pass & 1];
    for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
        const uint32_t p = q[i];
        ps.out[p] = *ps.L(p);
    }
}


// one row of the grid (blockIdx.y) per slot
__global__ __launch_bounds__(kBlock) void k_flush_m(const FrameSlot *__restrict__ fs, uint32_t nfs, uint32_t pass)
{
    const FrameSlot &f = fs[blockIdx.y];
    flush_body(f.prm, f.ps, pass);
}



// ------------------------------------------------------------ resolve
__device__ __forceinline__ void resolve_body(const PtParams &prm, const PathState &ps, float4 *noise)
{
    const uint32_t spp = (uint32_t)prm.rs.spp;
    const uint32_t pix_in_chunk = prm.chunk_paths / spp;
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= pix_in_chunk) return;
    const uint64_t vpix = prm.chunk_base / spp + k;
    const uint32_t tile = (uint32_t)(vpix >> 8), within = (uint32_t)(vpix & 255u);
    const uint32_t ty = tile / prm.tiles_x, tx = tile - ty * prm.tiles_x;
    const uint32_t px = tx * 16u + (within & 15u), py = ty * 16u + (within >> 4);
    if (px >= prm.rs.width || py >= prm.rs.height) return;
    const float inv = 1.0f / (float)(prm.rs.spp > 1 ? prm.rs.spp : 1);
    float a0 = 0.0f, a1 = 0.0f, a2 = 0.0f, a3 = 0.0f;
    const float4 *o = ps.out + (size_t)k * spp;
    for (uint32_t s = 0; s < spp; ++s) {
        const float4 v = o[s];
        a0 += v.x * inv;
        a1 += v.y * inv;
        a2 += v.z * inv;
        a3 += inv;
    }
    noise[(size_t)py * prm.rs.width + px] = make_float4(a0, a1, a2, a3);
    // the id image holds sample 0's camera-ray instance (RayTraceEditorView,
    // src/Shading.cu:1545-1547, keeps whichever sample wrote last)
    if (prm.aov) prm.aov[(size_t)py * prm.rs.width + px] = ps.first_hit[(size_t)k * spp];
}


// one row of the grid (blockIdx.y) per slot, each into its frame's image
__global__ void k_resolve_m(const FrameSlot *__restrict__ fs)
{
    const FrameSlot &f = fs[blockIdx.y];
    resolve_body(f.prm, f.ps, f.prm.noise);
}



// ------------------------------------------------------------ post
__global__ void k_accumulate(const float4 *noise, float4 *accum, uint32_t n, int frame)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float4 v = noise[i];
    if (frame == 1) {
        accum[i] = v;
        return;
    }
    const float4 a = accum[i];
    const float fm1 = (float)(frame - 1), fr = (float)frame;
    accum[i] = make_float4((a.x * fm1 + v.x) / fr, (a.y * fm1 + v.y) / fr, (a.z * fm1 + v.z) / fr,
                           (a.w * fm1 + v.w) / fr);
}

__global__ void k_tonemap(float4 *img, uint32_t n, float gamma, float exposure)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float4 v = img[i];
    float c[3] = {v.x, v.y, v.z};
    for (int k = 0; k < 3; ++k) {
        const float x = c[k] * exposure;
        const float y = (x * (2.51f * x + 0.03f)) / (x * (2.43f * x + 0.59f) + 0.14f);
        c[k] = ym_powf(y, 1.0f / gamma);
    }
    img[i] = make_float4(c[0], c[1], c[2], 1.0f);
}

// ------------------------------------------------------------ launchers
// Persistent pass kernels: the caller's persistent_waves, or by default one
// wave per 64 paths of the launch (all slots), at most
// kMaxPersistentWaves (the traversal spill area holds kSpillThreads threads);
// launch_persistent then holds each kernel to the waves the GPU has room for.
// Waves a queue has no share for leave at once (for_slots).  Every pass kernel
// deals its queue over the grid it gets, so the count changes timing only.
uint32_t persistent_waves(uint64_t paths, uint32_t requested, uint32_t spill_threads)
{
    static_assert(kMaxPersistentWaves * kBlock == kSpillThreads, "one spill row per lane");
    const uint32_t most = spill_threads / kBlock;  // one spill row per lane
    const uint64_t waves = (paths + kBlock - 1) / kBlock;
    const uint64_t cap = std::min<uint64_t>(requested ? requested : most, most);
    return (uint32_t)std::max<uint64_t>(std::min(waves, cap), 1);
}

// ------------------------------------------------------------ multi-frame launchers
// One launch per stage for every slot of a round (ymrt_render_batch).  The
// variant is the union of the slots' scene features (each feature's code is
// inert where a scene lacks it); waves: the persistent grid shared by all
// slots; blocks: the most compaction / resolve blocks any slot needs.
__global__ __launch_bounds__(kBlock) void k_active_m(const FrameSlot *__restrict__ fs, uint32_t nfs, uint32_t pass,
                                                     uint32_t *out)
{
    uint32_t v = 0;
    for (uint32_t s = threadIdx.x; s < nfs; s += kBlock) v += fs[s].prm.counters[pass * kCtrStride + kCtrActive];
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    if (threadIdx.x == 0) *out = v;
}

// A persistent pass kernel gets at most as many one-wave blocks as the GPU
// holds at once (its occupancy times the CU count, queried once per
// kernel): further waves could only start once the stage's work has run
// out, and each would still take one fetch atomic on its counter.
template <typename... Params, typename... Args>
static void launch_persistent(void (*kernel)(Params...), uint32_t waves, hipStream_t s, Args... args)
{
    static std::mutex mu;
    static std::unordered_map<const void *, uint32_t> resident;
    uint32_t cap = 0;
    {
        std::lock_guard<std::mutex> lock(mu);
        auto it = resident.find((const void *)kernel);
        if (it == resident.end()) {
            int blocks = 0, dev = 0, cus = 0;
            if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, kernel, kBlock, 0) == hipSuccess &&
                hipGetDevice(&dev) == hipSuccess &&
                hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess)
                cap = (uint32_t)(blocks * cus);
            resident.emplace((const void *)kernel, cap);
        } else {
            cap = it->second;
        }
    }
    const uint32_t grid = cap > 0 && cap < waves ? cap : waves;
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(kBlock), 0, s, args...);
}

int launch_multi_active(const FrameSlot *fs, uint32_t nfs, uint32_t pass, uint32_t *out, hipStream_t s)
{
    hipLaunchKernelGGL(k_active_m, dim3(1), dim3(kBlock), 0, s, fs, nfs, pass, out);
    YM_HIP(hipGetLastError());
    return YMRT_OK;
}

int launch_multi_raygen(const FrameSlot *fs, uint32_t nfs, uint32_t waves, hipStream_t s)
{
    launch_persistent(k_raygen_m, waves, s, fs, nfs);
    YM_HIP(hipGetLastError());
    return YMRT_OK;
}

template <bool kNearby, bool kMedia, bool kSphere>
static void extend_m(const FrameSlot *fs, uint32_t nfs, uint32_t waves, uint32_t pass, hipStream_t s)
{
    launch_persistent((k_extend_m<kNearby, kMedia, kSphere, kMaxStackDepth>), waves, s, fs, nfs, pass);
}

int launch_multi_extend(const FrameSlot *fs, uint32_t nfs, const MultiVariant &v, uint32_t waves, uint32_t pass,
                        hipStream_t s)
{
    const int k = (v.nearby ? 4 : 0) | (v.media ? 2 : 0) | (v.sphere ? 1 : 0);
    switch (k) {
    case 0: extend_m<false, false, false>(fs, nfs, waves, pass, s); break;
    case 1: extend_m<false, false, true>(fs, nfs, waves, pass, s); break;
    case 2: extend_m<false, true, false>(fs, nfs, waves, pass, s); break;
    case 3: extend_m<false, true, true>(fs, nfs, waves, pass, s); break;
    case 4: extend_m<true, false, false>(fs, nfs, waves, pass, s); break;
    case 5: extend_m<true, false, true>(fs, nfs, waves, pass, s); break;
    case 6: extend_m<true, true, false>(fs, nfs, waves, pass, s); break;
    default: extend_m<true, true, true>(fs, nfs, waves, pass, s); break;
    }
    YM_HIP(hipGetLastError());
    return YMRT_OK;
}

int launch_multi_medium(const FrameSlot *fs, uint32_t nfs, const MultiVariant &v, uint32_t waves, uint32_t pass,
                        hipStream_t s)
{
    if (v.adj && v.het == 2) launch_persistent((k_medium_m<2, true>), waves, s, fs, nfs, pass);
    else if (v.adj && v.het == 1) launch_persistent((k_medium_m<1, true>), waves, s, fs, nfs, pass);
    else if (v.het == 2) launch_persistent(k_medium_m<2>, waves, s, fs, nfs, pass);
    else if (v.het == 1) launch_persistent(k_medium_m<1>, waves, s, fs, nfs, pass);
    else launch_persistent(k_medium_m<0>, waves, s, fs, nfs, pass);
    YM_HIP(hipGetLastError());
    return YMRT_OK;
}

// launched: counts the kernels it launches (so does launch_multi_shade).
int launch_multi_compact(const FrameSlot *fs, uint32_t nfs, uint32_t blocks, uint32_t pass, int mode, hipStream_t s,
                         uint32_t *launched)
{
    const dim3 g(blocks ? blocks : 1, nfs), b(kCompactThreads), g1(4, nfs), b1(kScanThreads);
    // the longest chunk of the launch has at most this many slots
    const uint64_t longest = (uint64_t)blocks * kCompactSpan;
    if (longest <= kCompactSmall && nfs * longest * longest <= kCompactReads) {
        const dim3 gs(std::max(blocks, 1u) * (kCompactSpan / kScanThreads), nfs);
        if (mode == kCompactShade) hipLaunchKernelGGL(k_compact_small_m<kCompactShade>, gs, b1, 0, s, fs, pass);
        else if (mode == kCompactMedium) hipLaunchKernelGGL(k_compact_small_m<kCompactMedium>, gs, b1, 0, s, fs, pass);
        else hipLaunchKernelGGL(k_compact_small_m<kCompactTransmit>, gs, b1, 0, s, fs, pass);
        YM_HIP(hipGetLastError());
        *launched += 1;
        return YMRT_OK;
    }
    if (mode == kCompactShade) {
        hipLaunchKernelGGL(k_compact_count_m<kCompactShade>, g, b, 0, s, fs, pass);
        hipLaunchKernelGGL(k_compact_scan_m<kCompactShade>, g1, b1, 0, s, fs);
        hipLaunchKernelGGL(k_compact_scatter_m<kCompactShade>, g, b, 0, s, fs, pass);
    } else if (mode == kCompactMedium) {
        hipLaunchKernelGGL(k_compact_count_m<kCompactMedium>, g, b, 0, s, fs, pass);
        hipLaunchKernelGGL(k_compact_scan_m<kCompactMedium>, g1, b1, 0, s, fs);
        hipLaunchKernelGGL(k_compact_scatter_m<kCompactMedium>, g, b, 0, s, fs, pass);
    } else {
        hipLaunchKernelGGL(k_compact_count_m<kCompactTransmit>, g, b, 0, s, fs, pass);
        hipLaunchKernelGGL(k_compact_scan_m<kCompactTransmit>, g1, b1, 0, s, fs);
        hipLaunchKernelGGL(k_compact_scatter_m<kCompactTransmit>, g, b, 0, s, fs, pass);
    }
    YM_HIP(hipGetLastError());
    *launched += 3;
    return YMRT_OK;
}

template <bool kGraph, bool kAdj>
static void shade_m(const FrameSlot *fs, uint32_t nfs, uint32_t waves, uint32_t pass, hipStream_t s)
{
    launch_persistent((k_shade_m<false, kGraph, kMatGeneral, kAdj>), waves, s, fs, nfs, pass);
    launch_persistent((k_shade_m<false, kGraph, kMatDiffuse, kAdj>), waves, s, fs, nfs, pass);
    launch_persistent((k_shade_m<false, kGraph, kMatMetal, kAdj>), waves, s, fs, nfs, pass);
}

// With up to this many paths the shading classes share one launch (not in
// frames with texture graphs and media, nor in the adjoint's replay, for which
// no such kernel is built).  One launch against one per class, ms per frame at
// 2^16, 2^18, 2^19 and 2^21 paths: Cornell 1.64 and 2.01, 2.94 and 3.34, 4.56
// and 4.89, 8.92 and 8.97; outdoor with fog 3.13 and 4.21, 4.97 and 5.98, 6.59
// and 7.39, 12.9 and 12.8; smoke 5.48 and 6.67, 8.21 and 9.26, 11.4 and 11.9,
// 28.9 and 27.4; interior 3.89 and 4.22, 6.24 and 6.47, 10.6 and 10.0, 21.1 and
// 20.6.  Long queues lose: their waves run different classes at once, which
// share an instruction cache.
// Frames with texture graphs and no media share one launch at any length: all
// their classes run at 2 waves per SIMD, and one class' waves fill what another
// leaves at its end.  At 2^16, 2^18, 0.8 M, 2.1 M and 4.2 M paths: Cornell with a
// checkerboard 1.66 and 2.08, 3.06 and 3.46, 5.17 and 5.54, 7.48 and 7.85, 13.8
// and 14.3; the interior with one graph-textured object 3.18 and 3.43, 5.23 and
// 5.56, 9.10 and 9.67, 15.6 and 17.2, 25.8 and 27.2; a batch of six such rooms
// without and one small frame with a graph 39.8 and 42.2.  A box whose every
// wall runs a graph is the exception, between 2^18 and 2^21 paths: 1.84 and
// 2.18, 3.57 and 3.51, 6.99 and 6.52, 10.8 and 10.7, 20.9 and 21.8.
constexpr uint64_t kShadeAllPaths = 1u << 18;

// paths: no fewer than the launch's queues hold together.
int launch_multi_shade(const FrameSlot *fs, uint32_t nfs, const MultiVariant &v, uint64_t paths, uint32_t waves,
                       uint32_t pass, hipStream_t s, uint32_t *launched)
{
    if (v.graph && !v.media && !v.adj) {
        launch_persistent((k_shade_all_m<false, true>), waves, s, fs, nfs, pass);
        YM_HIP(hipGetLastError());
        *launched += 1;
        return YMRT_OK;
    }
    if (paths <= kShadeAllPaths && !v.graph && !v.adj) {
        if (v.media) launch_persistent(k_shade_all_m<true>, waves, s, fs, nfs, pass);
        else launch_persistent(k_shade_all_m<false>, waves, s, fs, nfs, pass);
        YM_HIP(hipGetLastError());
        *launched += 1;
        return YMRT_OK;
    }
    if (v.graph) v.adj ? shade_m<true, true>(fs, nfs, waves, pass, s) : shade_m<true, false>(fs, nfs, waves, pass, s);
    else v.adj ? shade_m<false, true>(fs, nfs, waves, pass, s) : shade_m<false, false>(fs, nfs, waves, pass, s);
    // volume vertices carry no adjoint events of their own
    if (v.media) launch_persistent((k_shade_m<true, false>), waves, s, fs, nfs, pass);
    YM_HIP(hipGetLastError());
    *launched += v.media ? 4 : 3;
    return YMRT_OK;
}

int launch_multi_shadow(const FrameSlot *fs, uint32_t nfs, const MultiVariant &v, uint32_t waves, uint32_t pass,
                        hipStream_t s)
{
    if (v.adj) {
        if (v.sphere) {
            if (v.media) launch_persistent((k_shadow_m<true, true, kMaxStackDepth, true>), waves, s, fs, nfs, pass);
            else launch_persistent((k_shadow_m<false, true, kMaxStackDepth, true>), waves, s, fs, nfs, pass);
        } else {
            if (v.media) launch_persistent((k_shadow_m<true, false, kMaxStackDepth, true>), waves, s, fs, nfs, pass);
            else launch_persistent((k_shadow_m<false, false, kMaxStackDepth, true>), waves, s, fs, nfs, pass);
        }
    } else if (v.sphere) {
        if (v.media) launch_persistent((k_shadow_m<true, true, kMaxStackDepth>), waves, s, fs, nfs, pass);
        else launch_persistent((k_shadow_m<false, true, kMaxStackDepth>), waves, s, fs, nfs, pass);
    } else {
        if (v.media) launch_persistent((k_shadow_m<true, false, kMaxStackDepth>), waves, s, fs, nfs, pass);
        else launch_persistent((k_shadow_m<false, false, kMaxStackDepth>), waves, s, fs, nfs, pass);
    }
    YM_HIP(hipGetLastError());
    return YMRT_OK;
}

int launch_multi_transmit(const FrameSlot *fs, uint32_t nfs, const MultiVariant &v, uint32_t waves, uint32_t pass,
                          hipStream_t s)
{
    if (v.adj) {
        if (v.sphere) {
            if (v.het == 2) launch_persistent((k_transmit_m<true, kMaxStackDepth, 2, true>), waves, s, fs, nfs, pass);
            else if (v.het == 1) launch_persistent((k_transmit_m<true, kMaxStackDepth, 1, true>), waves, s, fs, nfs, pass);
            else launch_persistent((k_transmit_m<true, kMaxStackDepth, 0, true>), waves, s, fs, nfs, pass);
        } else {
            if (v.het == 2) launch_persistent((k_transmit_m<false, kMaxStackDepth, 2, true>), waves, s, fs, nfs, pass);
            else if (v.het == 1) launch_persistent((k_transmit_m<false, kMaxStackDepth, 1, true>), waves, s, fs, nfs, pass);
            else launch_persistent((k_transmit_m<false, kMaxStackDepth, 0, true>), waves, s, fs, nfs, pass);
        }
    } else if (v.sphere) {
        if (v.het == 2) launch_persistent((k_transmit_m<true, kMaxStackDepth, 2>), waves, s, fs, nfs, pass);
        else if (v.het == 1) launch_persistent((k_transmit_m<true, kMaxStackDepth, 1>), waves, s, fs, nfs, pass);
        else launch_persistent((k_transmit_m<true, kMaxStackDepth, 0>), waves, s, fs, nfs, pass);
    } else {
        if (v.het == 2) launch_persistent((k_transmit_m<false, kMaxStackDepth, 2>), waves, s, fs, nfs, pass);
        else if (v.het == 1) launch_persistent((k_transmit_m<false, kMaxStackDepth, 1>), waves, s, fs, nfs, pass);
        else launch_persistent((k_transmit_m<false, kMaxStackDepth, 0>), waves, s, fs, nfs, pass);
    }
    YM_HIP(hipGetLastError());
    return YMRT_OK;
}

int launch_multi_flush(const FrameSlot *fs, uint32_t nfs, uint32_t pass, hipStream_t s)
{
    hipLaunchKernelGGL(k_flush_m, dim3(64, nfs), dim3(kBlock), 0, s, fs, nfs, pass);
    YM_HIP(hipGetLastError());
    return YMRT_OK;
}

int launch_multi_resolve(const FrameSlot *fs, uint32_t nfs, uint32_t pixel_blocks, hipStream_t s)
{
    hipLaunchKernelGGL(k_resolve_m, dim3(pixel_blocks ? pixel_blocks : 1, nfs), dim3(256), 0, s, fs);
    YM_HIP(hipGetLastError());
    return YMRT_OK;
}


// Texture graph at n given coordinates: coords[i*8 + 0..7] = (s, t,
// p_world.xyz, p_object.xyz), out[i*3 + 0..2] = the texture's rgb.
__global__ __launch_bounds__(kBlock) void k_texture_eval(DevScene sc, uint32_t tex, const float *coords, uint32_t n,
                                                         float *out)
{
    __shared__ float tex_stk[kTexStack * 3 * kBlock];
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const float *c = coords + (size_t)i * 8;
    TexEval<true> tx{sc, TexCoord{f2{c[0], c[1]}, f3{c[2], c[3], c[4]}, f3{c[5], c[6], c[7]}}, tex_stk,
                     (int)threadIdx.x};
    const f3 v = tx.eval(tex);
    out[(size_t)i * 3 + 0] = v.x;
    out[(size_t)i * 3 + 1] = v.y;
    out[(size_t)i * 3 + 2] = v.z;
}

int launch_texture_eval(const DevScene &sc, uint32_t tex, const float *coords, uint32_t n, float *out, hipStream_t s)
{
    YM_REQUIRE(tex < sc.texture_count, "texture index out of range");
    if (n == 0) return YMRT_OK;
    hipLaunchKernelGGL(k_texture_eval, dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, s, sc, tex, coords, n, out);
    YM_HIP(hipGetLastError());
    return YMRT_OK;
}

int accumulate(const float *noise, float *accum, uint32_t w, uint32_t h, int frame, hipStream_t s)
{
    const uint32_t n = w * h;
    if (n == 0) return YMRT_OK;
    hipLaunchKernelGGL(k_accumulate, dim3((n + 255) / 256), dim3(256), 0, s, reinterpret_cast<const float4 *>(noise),
                       reinterpret_cast<float4 *>(accum), n, frame);
    YM_HIP(hipGetLastError());
    return YMRT_OK;
}

int tonemap(float *rgba, uint32_t w, uint32_t h, float gamma, float exposure, hipStream_t s)
{
    const uint32_t n = w * h;
    if (n == 0) return YMRT_OK;
    hipLaunchKernelGGL(k_tonemap, dim3((n + 255) / 256), dim3(256), 0, s, reinterpret_cast<float4 *>(rgba), n, gamma,
                       exposure);
    YM_HIP(hipGetLastError());
    return YMRT_OK;
}

}  // namespace ym
