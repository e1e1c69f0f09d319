// Extend (closest hit) and connect (any hit) kernels.
//
// Persistent threads: the grid fills the GPU once; each wave64 lane runs a
// traversal state machine and, whenever its ray finishes, the lanes that went
// idle fetch new ray indices with one wave-aggregated atomic (dynamic ray
// fetching, Aila & Laine 2009) — so lanes do not wait for the longest ray of a
// batch and no blocks are launched for rays that do not exist.
//
// Stack traversal of the 128-byte 4-wide nodes (the binary LBVH collapsed two
// levels per node, halving the chain of dependent node fetches per ray; one node
// is one 128-byte cache line). The stack is a per-thread column of LDS
// ([depth][thread], bank-conflict free), deeper entries go to a per-thread slot
// in global memory. Hit leaves (one triangle each) wait in a small queue per lane,
// in the order of their entry distance (order_key); internal children go on the
// stack, the nearest on top. A wave intersects queued leaves when three eighths of
// its busy lanes have some: a ray has one leaf hit per ten node steps, so testing at once
// ran the triangle test for a few lanes of 64 in nearly every step. The triangles
// are tested in the order in which a sequential traversal meets them, and a leaf
// whose entry lies behind the closest hit by then is dropped, as that traversal
// would have: an entry distance never decreases from a node to its children, so
// what the late hit lets through meanwhile is dropped too. Every FP operation
// matches the sequential restatement in the oracle, and hits agree bit for bit.
//
// Bounded by the return of divergent node loads and the vector pipe together (64 % and
// 53 % busy on 10^6 incoherent rays), and by the longest rays at the end of a
// launch. Against one triangle test per leaf in the step, a sorting network with
// selects, refills below 16 lanes and one fetch counter (both builds in turn in one run,
// passes in a row, which is how every time in this file is taken): 1920x1080 frame of the
// 3.1M-triangle scene 3.11 -> 2.83 ms, the reference estimator's frame on 2058
// triangles 4.69 -> 3.44 ms, 512x512 turntable 2.44 -> 2.34 ms. The reference frame varies
// between runs, 3.4 to 3.7 ms with what the process measured before it.
//
// The ray/box and ray/triangle tests and the child order key are in ohpt_trace.h.
#pragma clang fp contract(off)

#include "ohpt_trace.h"

namespace ohpt {
namespace {

using namespace trace;

// Lanes keep stepping without refilling while at least this many are busy (10^6 rays:
// 531 us a call at 16, 517 at 24, 506 at 32, 500 at 40; turntable 2.36, 2.35, 2.32, 2.33 ms).
#ifndef OHPT_REFILL_THRESHOLD
#define OHPT_REFILL_THRESHOLD 32
#endif
constexpr int kRefillThreshold = OHPT_REFILL_THRESHOLD;

// Queued leaves are intersected once kDrainAt eighths of the busy lanes have some, until
// fewer than kDrainTo eighths do (3 / 2, 4 / 3 and 3 / 1 within 1 %, 2 / 1 slower by 1 %).
constexpr uint32_t kDrainAt = 3, kDrainTo = 2;
constexpr uint32_t kPend = 8;   // entries per lane, a power of two of at least 4
static_assert(kPend >= 4 && (kPend & (kPend - 1)) == 0, "a node step can queue four leaves");

// Ray sources/sinks of the four kernels.
struct ExtendIO {
    static constexpr bool kPosTmin = true;
    const uint32_t* queue;
    const float4* ray_o;
    const float4* ray_d;
    float4* hits;
    __device__ __forceinline__ void load(uint32_t j, float3& o, float3& d, float& tmin, float& tmax) const {
        const uint32_t pid = queue[j];
        const float4 a = ray_o[pid], b = ray_d[pid];
        o = make_float3(a.x, a.y, a.z);
        d = make_float3(b.x, b.y, b.z);
        tmin = 0.0f;
        tmax = INFINITY;
    }
    __device__ __forceinline__ void store(const DevScene&, uint32_t j, float4 h) const { hits[j] = h; }
};

struct ConnectIO {
    static constexpr bool kPosTmin = true;
    const float4* sh_o;
    const float4* sh_d;
    const float4* sh_c;
    float4* ln0;
    float4* ln1;
    uint32_t* vis;        // optional: per-path visibility bits for path replay
    uint32_t bounce;
    __device__ __forceinline__ void load(uint32_t j, float3& o, float3& d, float& tmin, float& tmax) const {
        const float4 a = sh_o[j], b = sh_d[j];
        o = make_float3(a.x, a.y, a.z);
        d = make_float3(b.x, b.y, b.z);
        tmin = 0.0f;
        tmax = a.w;
    }
    __device__ __forceinline__ void store(const DevScene&, uint32_t j, float4 h) const {
        if (__float_as_uint(h.y) != kMiss) return;
        const uint32_t tag = __float_as_uint(sh_d[j].w);
        const uint32_t pid = tag >> 1;
        float4* dst = (tag & 1u) ? ln1 : ln0;
        const float4 c = sh_c[j];
        float4 v = dst[pid];
        v.x += c.x; v.y += c.y; v.z += c.z;
        dst[pid] = v;
        if (vis) atomicOr(&vis[pid], 1u << (2u * bounce + (tag & 1u)));
    }
};

struct RaysIO {
    static constexpr bool kPosTmin = false;
    const float4* rays;
    float4* hits;
    uint32_t* occl;
    __device__ __forceinline__ void load(uint32_t j, float3& o, float3& d, float& tmin, float& tmax) const {
        const float4 a = rays[(size_t)j * 2], b = rays[(size_t)j * 2 + 1];
        o = make_float3(a.x, a.y, a.z);
        d = make_float3(b.x, b.y, b.z);
        tmin = a.w;
        tmax = b.w;
    }
    __device__ __forceinline__ void store(const DevScene& S, uint32_t j, float4 h) const {
        const uint32_t s = __float_as_uint(h.y);
        if (occl) {
            occl[j] = s != kMiss ? 1u : 0u;
        } else {
            if (s != kMiss) h.y = S.tris[(size_t)s * 3].w;   // slot -> caller's triangle id
            hits[j] = h;
        }
    }
};

// The reference estimator's rays (its traceRayEXT calls: t from 0.001): closest-hit
// rays of the queue up to o.w (10000, or 0 for a path that only waits for its
// shadow rays), shadow rays up to sh_o.w, whose visibility marks the pending
// contribution (w = 2) for the next shading step to add.
struct RefExtendIO {
    const uint32_t* queue;
    const float4* ray_o;
    const float4* ray_d;
    float4* hits;
    __device__ __forceinline__ void load(uint32_t j, float3& o, float3& d, float& tmin, float& tmax) const {
        const uint32_t pid = queue[j];
        const float4 a = ray_o[pid], b = ray_d[pid];
        o = make_float3(a.x, a.y, a.z);
        d = make_float3(b.x, b.y, b.z);
        tmin = 0.001f;
        tmax = a.w;
    }
    __device__ __forceinline__ void store(const DevScene&, uint32_t j, float4 h) const { hits[j] = h; }
};

struct RefConnectIO {
    const float4* sh_o;
    const float4* sh_d;
    float4* ln0;
    float4* ln1;
    __device__ __forceinline__ void load(uint32_t j, float3& o, float3& d, float& tmin, float& tmax) const {
        const float4 a = sh_o[j], b = sh_d[j];
        o = make_float3(a.x, a.y, a.z);
        d = make_float3(b.x, b.y, b.z);
        tmin = 0.001f;
        tmax = a.w;
    }
    __device__ __forceinline__ void store(const DevScene&, uint32_t j, float4 h) const {
        if (__float_as_uint(h.y) != kMiss) return;
        const uint32_t tag = __float_as_uint(sh_d[j].w);
        float4* dst = (tag & 1u) ? ln1 : ln0;
        dst[tag >> 1].w = 2.0f;
    }
};

struct RefFusedIO {
    static constexpr bool kPosTmin = true;
    RefExtendIO ext;
    RefConnectIO con;
    uint32_t n_ext;
    __device__ __forceinline__ bool any_hit(uint32_t j) const { return j >= n_ext; }
    __device__ __forceinline__ void load(uint32_t j, float3& o, float3& d, float& tmin, float& tmax) const {
        if (j < n_ext) ext.load(j, o, d, tmin, tmax);
        else con.load(j - n_ext, o, d, tmin, tmax);
    }
    __device__ __forceinline__ void store(const DevScene& S, uint32_t j, float4 h) const {
        if (j < n_ext) ext.store(S, j, h);
        else con.store(S, j - n_ext, h);
    }
};

// kMode: 0 closest hit, 1 any hit, 2 per ray (IO::any_hit(j)).
// Extension rays of one bounce and shadow rays of the previous one, traced by
// one launch: indices [0, n_ext) are closest-hit rays, the rest any-hit.
struct FusedIO {
    static constexpr bool kPosTmin = true;
    ExtendIO ext;
    ConnectIO con;
    uint32_t n_ext;
    __device__ __forceinline__ bool any_hit(uint32_t j) const { return j >= n_ext; }
    __device__ __forceinline__ void load(uint32_t j, float3& o, float3& d, float& tmin, float& tmax) const {
        if (j < n_ext) ext.load(j, o, d, tmin, tmax);
        else con.load(j - n_ext, o, d, tmin, tmax);
    }
    __device__ __forceinline__ void store(const DevScene& S, uint32_t j, float4 h) const {
        if (j < n_ext) ext.store(S, j, h);
        else con.store(S, j - n_ext, h);
    }
};

// kStats: count node visits and triangle tests into stats[0..1] (profiling
// launches only; the counters cost registers).
template <int kMode, bool kStats, class IO>
__device__ __forceinline__ void persistent_trace(const DevScene& S, const IO& io, uint32_t count,
                                                 uint32_t* fetch, uint32_t* lds_col, uint2* pend,
                                                 uint32_t* ovf, unsigned long long* stats) {
    const uint32_t lane = lane_id();
    RayPre r;
    uint32_t cur = 0, j = 0, sp = 0;
    // closest hit so far: distance tclose (tmax while none), slot hprim, barycentrics hu, hv
    float tmin = 0.0f, tclose = 0.0f, hu = 0.0f, hv = 0.0f;
    uint32_t hprim = kMiss;
    float tgroup = 0.0f;           // tclose when the first leaf of the tested one's node came up
    bool active = false, anyhit = kMode == 1;
    bool fin = false;              // nothing left to visit; the queued leaves remain
    uint32_t qh = 0, qn = 0;       // queued leaves: first entry, count
    uint32_t nv = 0, nt = 0;
    // The first ray of every thread is its global index (no atomics: launches with
    // fewer rays than resident threads never touch the counters). The rays beyond
    // are dealt in runs of 64 to `groups` groups of blocks, each with a counter of its
    // own in its own cache line: with one counter every wave's additions queued at one
    // address (one counter / 64 with all else alike: the reference estimator's 1080p frame
    // 5.09 / 3.39 ms, the 3.1M-triangle frame 2.98 / 2.84 ms, its 10^6 rays 615 / 505 us,
    // turntable 2.44 / 2.33 ms).
    const uint32_t nthreads = gridDim.x * blockDim.x;
    bool drained = nthreads >= count;
    const uint32_t groups = min(kFetchGroups, gridDim.x), group = blockIdx.x % groups;
    fetch += group * kFetchStride;
    auto start = [&](uint32_t idx) {
        float3 o, d;
        float tmax;
        j = idx;
        if constexpr (kMode == 2) anyhit = io.any_hit(j);
        io.load(j, o, d, tmin, tmax);
        r = ray_setup(o, d);
        tclose = tmax;
        hprim = kMiss;
        hu = hv = 0.0f;
        cur = 0;
        sp = 0;
        fin = false;
        qn = 0;
        active = S.n_tris > 0;
        if (!active) io.store(S, j, make_float4(tclose, __uint_as_float(hprim), hu, hv));
    };
    {
        const uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
        if (g < count) start(g);
    }
    for (;;) {
        // ---- refill idle lanes with new rays (one atomic per wave)
        if (!drained) {
            const uint64_t want = __ballot(!active);
            if (want != 0) {
                const int leader = __ffsll((unsigned long long)want) - 1;
                uint32_t base = 0;
                if ((int)lane == leader) base = atomicAdd(fetch, (uint32_t)__popcll(want));
                base = __shfl(base, leader);
                const uint32_t k = base + __builtin_amdgcn_mbcnt_hi((uint32_t)(want >> 32),
                                                                    __builtin_amdgcn_mbcnt_lo((uint32_t)want, 0u));
                const uint32_t last = base + (uint32_t)__popcll(want);
                drained = nthreads + ((last >> 6) * groups + group) * 64u + (last & 63u) >= count;
                if (!active) {
                    const uint32_t idx = nthreads + ((k >> 6) * groups + group) * 64u + (k & 63u);
                    if (idx < count) start(idx);
                }
            }
        }
        if (__ballot(active) == 0) {
            if (drained) break;
            continue;
        }
        // ---- traverse until too many lanes have finished (or to the end once drained)
        do {
            if (active && !fin && qn <= kPend - 4) {
                if constexpr (kStats) ++nv;
                const float4* np = S.nodes4 + (size_t)cur * 8;
                const float4 lx = np[0], ly = np[1], lz = np[2], hx = np[3], hy = np[4], hz = np[5];
                const uint4 rf = reinterpret_cast<const uint4*>(np)[6];
                const float e[4] = {box_hit(r, lx.x, ly.x, lz.x, hx.x, hy.x, hz.x, tmin, tclose),
                                    box_hit(r, lx.y, ly.y, lz.y, hx.y, hy.y, hz.y, tmin, tclose),
                                    box_hit(r, lx.z, ly.z, lz.z, hx.z, hy.z, hz.z, tmin, tclose),
                                    box_hit(r, lx.w, ly.w, lz.w, hx.w, hy.w, hz.w, tmin, tclose)};
                const uint32_t c[4] = {rf.x, rf.y, rf.z, rf.w};
                // each hit child's rank by sort key among the hit children of its kind (leaf or
                // internal): 6 compares, and the lane masks are combined in scalar registers
                bool leaf[4], inner[4], lt[4][4];
                uint32_t key[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const bool hit = e[i] != INFINITY && c[i] != kMiss;
                    leaf[i] = hit && (c[i] & kLeafBit);
                    inner[i] = hit && !(c[i] & kLeafBit);
                    key[i] = IO::kPosTmin ? order_key_pos(e[i], i) : order_key(e[i], i);
                }
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int k = i + 1; k < 4; ++k) {
                        const bool less = key[i] < key[k];
                        const bool same = (leaf[i] && leaf[k]) || (inner[i] && inner[k]);
                        lt[i][k] = same && less;
                        lt[k][i] = same && !less;
                    }
                uint32_t rank[4], nleaf = 0, ninner = 0;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    rank[i] = 0;
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        if (k != i) rank[i] += lt[k][i] ? 1u : 0u;
                    nleaf += leaf[i] ? 1u : 0u;
                    ninner += inner[i] ? 1u : 0u;
                }
                // leaves join the queue nearest first; a node's first one keeps the leaf bit
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (leaf[i])
                        pend[((qh + qn + rank[i]) & (kPend - 1)) * kTraceBlock] =
                            make_uint2(rank[i] == 0 ? c[i] : c[i] & ~kLeafBit, __float_as_uint(e[i]));
                qn += nleaf;
                // internal children go on the stack, the nearest on top, and the top is next
                sp += ninner;
                if (sp <= kStackLds) {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (inner[i]) lds_col[(sp - 1 - rank[i]) * kTraceBlock] = c[i];
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const uint32_t at = sp - 1 - rank[i];
                        if (inner[i]) {
                            if (at < kStackLds) lds_col[at * kTraceBlock] = c[i];
                            else ovf[at - kStackLds] = c[i];
                        }
                    }
                }
                if (sp == 0) {
                    fin = true;
                } else {
                    --sp;
                    cur = sp < kStackLds ? lds_col[sp * kTraceBlock] : ovf[sp - kStackLds];
                }
                if (fin && qn == 0) {
                    io.store(S, j, make_float4(tclose, __uint_as_float(hprim), hu, hv));
                    active = false;
                }
            }
            // ---- intersect queued leaves once enough lanes have some, or no lane can step
            uint32_t busy = (uint32_t)__popcll(__ballot(active));
            uint32_t waiting = (uint32_t)__popcll(__ballot(active && qn > 0));
            const bool stuck = __ballot(active && !fin && qn <= kPend - 4) == 0;
            if (waiting > 0 && (stuck || waiting * 8 >= busy * kDrainAt)) {
                do {
                    if (active && qn > 0) {
                        const uint2 w = pend[qh * kTraceBlock];
                        qh = (qh + 1) & (kPend - 1);
                        --qn;
                        if (w.x & kLeafBit) tgroup = tclose;
                        bool done = fin && qn == 0;
                        if (__uint_as_float(w.y) <= tgroup) {
                            const uint32_t s = w.x & ~kLeafBit;
                            const float4* tp = S.tris + (size_t)s * 3;
                            const float4 ta = tp[0], tb = tp[1], tc = tp[2];
                            float tt, uu, vv;
                            if constexpr (kStats) ++nt;
                            if (tri_hit(r, ta, tb, tc, tmin, tclose, tt, uu, vv)) {
                                tclose = tt;
                                hprim = s;
                                hu = uu;
                                hv = vv;
                                if (anyhit) done = true;
                            }
                        }
                        if (done) {
                            io.store(S, j, make_float4(tclose, __uint_as_float(hprim), hu, hv));
                            active = false;
                            qn = 0;
                        }
                    }
                    busy = (uint32_t)__popcll(__ballot(active));
                    waiting = (uint32_t)__popcll(__ballot(active && qn > 0));
                } while (waiting > 0 && waiting * 8 >= busy * kDrainTo);
            }
        } while (__popcll(__ballot(active)) >= (drained ? 1 : kRefillThreshold));
    }
    if constexpr (kStats) {
        for (int off = 32; off > 0; off >>= 1) {
            nv += __shfl_xor(nv, off);
            nt += __shfl_xor(nt, off);
        }
        if (lane == 0) {
            atomicAdd(&stats[0], (unsigned long long)nv);
            atomicAdd(&stats[1], (unsigned long long)nt);
        }
    }
}

template <bool kStats>
__global__ __launch_bounds__(kTraceBlock) void k_extend(DevScene S, ExtendIO io, const uint32_t* __restrict__ count,
                                                        uint32_t* __restrict__ fetch, uint32_t* __restrict__ ovf,
                                                        unsigned long long* __restrict__ stats) {
    __shared__ uint32_t lds[kStackLds * kTraceBlock];
    __shared__ uint2 pend[kPend * kTraceBlock];
    const uint32_t g = blockIdx.x * kTraceBlock + threadIdx.x;
    persistent_trace<0, kStats>(S, io, *count, fetch, lds + threadIdx.x, pend + threadIdx.x, ovf + (size_t)g * kStackOvf, stats);
}

template <bool kStats>
__global__ __launch_bounds__(kTraceBlock) void k_extend_connect(DevScene S, FusedIO io,
                                                                const uint32_t* __restrict__ count_ext,
                                                                const uint32_t* __restrict__ count_sh,
                                                                uint32_t* __restrict__ fetch,
                                                                uint32_t* __restrict__ ovf,
                                                                unsigned long long* __restrict__ stats) {
    __shared__ uint32_t lds[kStackLds * kTraceBlock];
    __shared__ uint2 pend[kPend * kTraceBlock];
    const uint32_t g = blockIdx.x * kTraceBlock + threadIdx.x;
    io.n_ext = *count_ext;
    persistent_trace<2, kStats>(S, io, io.n_ext + *count_sh, fetch, lds + threadIdx.x, pend + threadIdx.x, ovf + (size_t)g * kStackOvf,
                                stats);
}

__global__ __launch_bounds__(kTraceBlock) void k_ref_trace(DevScene S, RefFusedIO io,
                                                           const uint32_t* __restrict__ count_ext,
                                                           const uint32_t* __restrict__ count_sh,
                                                           uint32_t* __restrict__ fetch, uint32_t* __restrict__ ovf) {
    __shared__ uint32_t lds[kStackLds * kTraceBlock];
    __shared__ uint2 pend[kPend * kTraceBlock];
    const uint32_t g = blockIdx.x * kTraceBlock + threadIdx.x;
    io.n_ext = *count_ext;
    persistent_trace<2, false>(S, io, io.n_ext + *count_sh, fetch, lds + threadIdx.x, pend + threadIdx.x, ovf + (size_t)g * kStackOvf,
                               nullptr);
}

template <bool kAnyHit>
__global__ __launch_bounds__(kTraceBlock) void k_rays(DevScene S, RaysIO io, uint32_t n, uint32_t* __restrict__ fetch,
                                                      uint32_t* __restrict__ ovf) {
    __shared__ uint32_t lds[kStackLds * kTraceBlock];
    __shared__ uint2 pend[kPend * kTraceBlock];
    const uint32_t g = blockIdx.x * kTraceBlock + threadIdx.x;
    persistent_trace<kAnyHit ? 1 : 0, false>(S, io, n, fetch, lds + threadIdx.x, pend + threadIdx.x, ovf + (size_t)g * kStackOvf, nullptr);
}

__device__ __forceinline__ void sort2(uint32_t& a, uint32_t& b) {
    const uint32_t lo = min(a, b), hi = max(a, b);
    a = lo;
    b = hi;
}

// A ray per thread, for batches that are resident at once: without refills a launch lasts
// as long as its slowest wave, and a leaf that is intersected in its node's step, next nodes
// kept in registers and no queue make a step shorter. Same order, same hits. Persistent /
// this kernel, closest hits on the 3.1M-triangle scene: 64 random rays 119 / 104 us, 5,000
// 192 / 159, 100,003 252 / 200, 327,680 378 / 298 (pinhole 433 / 324); any hit 112 / 104,
// 189 / 166, 235 / 203, 342 / 298; 200,000 triangles 205 / 168 and Cornell box 64 / 53 at
// 327,680. (A loop per lane instead of the ballot is as fast for any hits, but takes 174 us for
// 64 closest hits: lanes that push then run ahead of lanes that pop.)
template <bool kAnyHit>
__global__ __launch_bounds__(kTraceBlock) void k_rays_direct(DevScene S, RaysIO io, uint32_t n,
                                                             uint32_t* __restrict__ ovf) {
    __shared__ uint32_t lds[kStackLds * kTraceBlock];
    const uint32_t j = blockIdx.x * kTraceBlock + threadIdx.x;
    if (j >= n) return;
    uint32_t* const lds_col = lds + threadIdx.x;
    ovf += (size_t)j * kStackOvf;
    float3 o, d;
    float tmin, tclose, hu = 0.0f, hv = 0.0f;
    io.load(j, o, d, tmin, tclose);
    const RayPre r = ray_setup(o, d);
    uint32_t hprim = kMiss, cur = 0, sp = 0;
    bool more = S.n_tris > 0;
    // the wave's lanes step together until the last one is done
    while (__ballot(more) != 0) {
        if (!more) continue;
        const float4* np = S.nodes4 + (size_t)cur * 8;
        const float4 lx = np[0], ly = np[1], lz = np[2], hx = np[3], hy = np[4], hz = np[5];
        const uint4 rf = reinterpret_cast<const uint4*>(np)[6];
        const float e[4] = {box_hit(r, lx.x, ly.x, lz.x, hx.x, hy.x, hz.x, tmin, tclose),
                            box_hit(r, lx.y, ly.y, lz.y, hx.y, hy.y, hz.y, tmin, tclose),
                            box_hit(r, lx.z, ly.z, lz.z, hx.z, hy.z, hz.z, tmin, tclose),
                            box_hit(r, lx.w, ly.w, lz.w, hx.w, hy.w, hz.w, tmin, tclose)};
        const uint32_t c[4] = {rf.x, rf.y, rf.z, rf.w};
        // the hit children in key order, a missed one (+inf, or an empty slot) last
        uint32_t key[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) key[i] = order_key(c[i] == kMiss ? INFINITY : e[i], i);
        sort2(key[0], key[1]);
        sort2(key[2], key[3]);
        sort2(key[0], key[2]);
        sort2(key[1], key[3]);
        sort2(key[1], key[2]);
        uint32_t child[4];
        float entry[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const uint32_t sl = key[k] & 3u;
            child[k] = sl == 0 ? c[0] : (sl == 1 ? c[1] : (sl == 2 ? c[2] : c[3]));
            entry[k] = key[k] >= order_key(INFINITY, 0) ? INFINITY
                                                        : (sl == 0 ? e[0] : (sl == 1 ? e[1] : (sl == 2 ? e[2] : e[3])));
        }
        bool done = false;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (entry[k] != INFINITY && (child[k] & kLeafBit) && !done) {
                const uint32_t s = child[k] & ~kLeafBit;
                const float4* tp = S.tris + (size_t)s * 3;
                const float4 ta = tp[0], tb = tp[1], tc = tp[2];
                float tt, uu, vv;
                if (tri_hit(r, ta, tb, tc, tmin, tclose, tt, uu, vv)) {
                    tclose = tt;
                    hprim = s;
                    hu = uu;
                    hv = vv;
                    done = kAnyHit;
                }
            }
        }
        // internal children still within the closest hit: the nearest next, the rest on the
        // stack, the nearer ones on top
        bool next = false;
        uint32_t first = 0;
#pragma unroll
        for (int k = 3; k >= 0; --k) {
            if (entry[k] != INFINITY && !(child[k] & kLeafBit) && entry[k] <= tclose && !done) {
                if (next) {
                    if (sp < kStackLds) lds_col[sp * kTraceBlock] = first;
                    else ovf[sp - kStackLds] = first;
                    ++sp;
                }
                first = child[k];
                next = true;
            }
        }
        if (next) {
            cur = first;
        } else if (sp > 0 && !done) {
            --sp;
            cur = sp < kStackLds ? lds_col[sp * kTraceBlock] : ovf[sp - kStackLds];
        } else {
            more = false;
        }
    }
    io.store(S, j, make_float4(tclose, __uint_as_float(hprim), hu, hv));
}

__global__ __launch_bounds__(256) void k_zero_fetch(uint32_t* p) { p[blockIdx.x * 256 + threadIdx.x] = 0u; }

uint32_t g_grid = 0;

}  // namespace

uint32_t trace_grid_blocks() {
    if (g_grid == 0) {
        int dev = 0, cus = 0, per_cu = 0;
        (void)hipGetDevice(&dev);
        (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
        (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_extend_connect<false>, kTraceBlock, 0);
        if (cus <= 0) cus = 256;
        if (per_cu <= 0) per_cu = 8;
        g_grid = (uint32_t)(cus * per_cu);
    }
    return g_grid;
}

size_t trace_overflow_bytes() { return (size_t)trace_grid_blocks() * kTraceBlock * kStackOvf * 4; }

void launch_extend(const DevScene& S, const uint32_t* queue, const uint32_t* count, uint32_t max_count,
                   const float4* ray_o, const float4* ray_d, float4* hits, uint32_t* fetch, uint32_t* ovf,
                   unsigned long long* stats, hipStream_t s, uint32_t max_blocks) {
    if (max_count == 0) return;
    ExtendIO io{queue, ray_o, ray_d, hits};
    uint32_t grid = std::min(trace_grid_blocks(), (max_count + kTraceBlock - 1) / kTraceBlock);
    if (max_blocks) grid = std::min(grid, max_blocks);
    if (stats) k_extend<true><<<grid, kTraceBlock, 0, s>>>(S, io, count, fetch, ovf, stats);
    else k_extend<false><<<grid, kTraceBlock, 0, s>>>(S, io, count, fetch, ovf, nullptr);
}

void launch_extend_connect(const DevScene& S, const uint32_t* queue, const uint32_t* count_ext, uint32_t max_ext,
                           const float4* ray_o, const float4* ray_d, float4* hits, const uint32_t* count_sh,
                           uint32_t max_sh, const float4* sh_o, const float4* sh_d, const float4* sh_c, float4* ln0,
                           float4* ln1, uint32_t* fetch, uint32_t* ovf, uint32_t* vis, uint32_t bounce,
                           unsigned long long* stats, hipStream_t s, uint32_t max_blocks) {
    if (max_ext + max_sh == 0) return;
    FusedIO io{ExtendIO{queue, ray_o, ray_d, hits}, ConnectIO{sh_o, sh_d, sh_c, ln0, ln1, vis, bounce}, 0u};
    uint32_t grid = std::min(trace_grid_blocks(), (max_ext + max_sh + kTraceBlock - 1) / kTraceBlock);
    if (max_blocks) grid = std::min(grid, max_blocks);
    if (stats) k_extend_connect<true><<<grid, kTraceBlock, 0, s>>>(S, io, count_ext, count_sh, fetch, ovf, stats);
    else k_extend_connect<false><<<grid, kTraceBlock, 0, s>>>(S, io, count_ext, count_sh, fetch, ovf, nullptr);
}

void launch_ref_trace(const DevScene& S, const uint32_t* queue, const uint32_t* count_ext, uint32_t max_ext,
                      const float4* ray_o, const float4* ray_d, float4* hits, const uint32_t* count_sh,
                      uint32_t max_sh, const float4* sh_o, const float4* sh_d, float4* ln0, float4* ln1,
                      uint32_t* fetch, uint32_t* ovf, hipStream_t s, uint32_t max_blocks) {
    if (max_ext + max_sh == 0) return;
    RefFusedIO io{RefExtendIO{queue, ray_o, ray_d, hits}, RefConnectIO{sh_o, sh_d, ln0, ln1}, 0u};
    uint32_t grid = std::min(trace_grid_blocks(), (max_ext + max_sh + kTraceBlock - 1) / kTraceBlock);
    if (max_blocks) grid = std::min(grid, max_blocks);
    k_ref_trace<<<grid, kTraceBlock, 0, s>>>(S, io, count_ext, count_sh, fetch, ovf);
}

void launch_trace_rays(const DevScene& S, const float4* rays, float4* hits, uint32_t n, uint32_t* fetch,
                       uint32_t* ovf, hipStream_t s, uint32_t max_blocks) {
    if (n == 0) return;
    RaysIO io{rays, hits, nullptr};
    uint32_t grid = std::min(trace_grid_blocks(), (n + kTraceBlock - 1) / kTraceBlock);
    if (max_blocks) grid = std::min(grid, max_blocks);
    if (n <= grid * kTraceBlock) {
        k_rays_direct<false><<<grid, kTraceBlock, 0, s>>>(S, io, n, ovf);
        return;
    }
    k_zero_fetch<<<kFetchWords / 256, 256, 0, s>>>(fetch);
    k_rays<false><<<grid, kTraceBlock, 0, s>>>(S, io, n, fetch, ovf);
}

void launch_occluded_rays(const DevScene& S, const float4* rays, uint32_t* out, uint32_t n, uint32_t* fetch,
                          uint32_t* ovf, hipStream_t s) {
    if (n == 0) return;
    RaysIO io{rays, nullptr, out};
    const uint32_t grid = std::min(trace_grid_blocks(), (n + kTraceBlock - 1) / kTraceBlock);
    if (n <= grid * kTraceBlock) {
        k_rays_direct<true><<<grid, kTraceBlock, 0, s>>>(S, io, n, ovf);
        return;
    }
    k_zero_fetch<<<kFetchWords / 256, 256, 0, s>>>(fetch);
    k_rays<true><<<grid, kTraceBlock, 0, s>>>(S, io, n, fetch, ovf);
}

}  // namespace ohpt
