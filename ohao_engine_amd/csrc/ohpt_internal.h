// Host-side declarations shared by the translation units of libohpt.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "ohpt_device.h"

namespace ohpt {

// ---- LBVH build (lbvh.hip) --------------------------------------------------
struct LbvhBuffers {
    // inputs (device): tri_pos n*9 floats (global order), nrm n*9 (or null), uv n*6 (or null), mat n
    const float* tri_pos;
    const float* tri_nrm;
    const float* tri_uv;
    const uint32_t* tri_mat;
    uint32_t n;
    // outputs (device, preallocated): nodes (max(n-1,1))*64 B, tris n*48 B, attrs n*64 B, prim n
    float4* nodes;
    float4* tris;
    float4* attrs;
    uint32_t* prim;        // slot -> original triangle id
    uint32_t* slot_of;     // original triangle id -> slot
    // scratch (device): see lbvh_scratch_bytes
    void* scratch;
};
size_t lbvh_scratch_bytes(uint32_t n);
// Returns 0 or a HIP error; writes max leaf depth to *depth_out and the number
// of 4-wide nodes to *n4_out (host) when not null.
hipError_t lbvh_build(const LbvhBuffers& b, hipStream_t s, uint32_t* depth_out, uint32_t* n4_out);
// Refit of a committed tree: b.prim (slot -> triangle) and b.nodes (topology,
// parent in field 14) are kept; the triangles are re-gathered from b.tri_pos /
// tri_nrm / tri_uv / tri_mat and every box recomputed bottom-up, then the
// 4-wide numbering is rebuilt in scratch for bvh4_collapse.
hipError_t lbvh_refit(const LbvhBuffers& b, hipStream_t s);
// Column-major 4x4 world matrix and row-major 3x3 normal matrix (inverse
// transpose of its upper 3x3) of one mesh, in double.
struct MeshTransform {
    double m[16];
    double n[9];
    int has_world;
};
// World-space triangle corners of one mesh (nt triangles, idx into object-space
// vertices vpos / vnrm) into tpos / tnrm (nt*9 floats each, at the mesh's
// first triangle). tnrm null: no normals; vnrm null with tnrm: geometric normals.
void launch_transform_mesh(const float* vpos, const float* vnrm, const uint32_t* idx, uint32_t nt,
                           const MeshTransform& x, float* tpos, float* tnrm, hipStream_t s);
// Corner uvs of one mesh (nt*6 floats into tuv); vuv null: zeros.
void launch_gather_uv(const float* vuv, const uint32_t* idx, uint32_t nt, float* tuv, hipStream_t s);
// After lbvh_build or lbvh_refit with the same buffers (scratch still holding
// depths and the 4-wide numbering): writes the n4 x 128 B 4-wide nodes.
hipError_t bvh4_collapse(const LbvhBuffers& b, float4* nodes4, hipStream_t s);

// Standalone stable radix sort of 32-bit keys with 32-bit values (exposed for tests).
size_t radix_sort_scratch_bytes(uint32_t n);
// Exclusive scan of n u32 in place (one block; n up to a few 100k), total to *total (device).
hipError_t exclusive_scan_u32(uint32_t* data, uint32_t n, uint32_t* total, hipStream_t s);
hipError_t radix_sort_pairs(uint32_t* keys, uint32_t* vals, uint32_t n, uint32_t key_bits, void* scratch,
                            hipStream_t s);

// ---- traversal (traverse.hip) ---------------------------------------------
// Launch shape of the traversal kernels (compile-time; -D overrides for tuning sweeps).
#ifndef OHPT_TRACE_BLOCK
#define OHPT_TRACE_BLOCK 128
#endif
#ifndef OHPT_STACK_LDS
#define OHPT_STACK_LDS 16   // with the leaf queue 16 KB per block: the VGPR-bound 5 waves per SIMD (10 blocks) fill a CU's 160 KB
#endif
constexpr uint32_t kTraceBlock = OHPT_TRACE_BLOCK;
constexpr uint32_t kStackLds = OHPT_STACK_LDS;   // per-thread LDS stack entries
constexpr uint32_t kStackOvf = 72;               // per-thread global overflow entries
constexpr uint32_t kMaxTreeDepth = 60;   // commit rejects deeper trees (binary leaf depth, root = 1)
// a binary tree of leaf depth D has at most D/2 levels of 4-wide nodes; each but the
// last (its children are leaves) leaves at most three entries behind, and the four of the
// deepest one are on the stack before the nearest is taken off
static_assert(kStackLds + kStackOvf >= 3 * (kMaxTreeDepth / 2 - 1) + 1, "traversal stack shallower than the deepest tree");
static_assert(kTraceBlock % 64 == 0 && kTraceBlock <= 1024, "trace block must be whole waves");

// Dynamic ray fetching: one counter per group of blocks, each in a cache line of its own.
constexpr uint32_t kFetchGroups = 64;
constexpr uint32_t kFetchStride = 32;                          // words from one counter to the next
constexpr uint32_t kFetchWords = kFetchGroups * kFetchStride;  // counters of one launch
static_assert(kFetchWords % 256 == 0, "cleared in blocks of 256 words");

// Persistent-thread grid of the traversal kernels and the size of their
// global stack-overflow buffer (one kStackOvf slot per resident thread).
uint32_t trace_grid_blocks();
size_t trace_overflow_bytes();

// Closest hit for queued paths: ray of path queue[j] -> hits[j] = (t, slot|miss, u, v).
// `fetch` are kFetchWords zeroed words for dynamic ray fetching. max_blocks != 0 caps
// the persistent grid (launches of concurrent lanes share the GPU).
void launch_extend(const DevScene& S, const uint32_t* queue, const uint32_t* count, uint32_t max_count,
                   const float4* ray_o, const float4* ray_d, float4* hits, uint32_t* fetch, uint32_t* ovf,
                   unsigned long long* stats, hipStream_t s, uint32_t max_blocks = 0);
// One launch for the extension rays of bounce b+1 (closest hit, into `hits`) and the
// shadow rays of bounce b (any hit): sh_o[j] = (o, tmax), sh_d[j] = (d, pid*2+k bits),
// sh_c[j] = contribution; unoccluded ones add sh_c into ln[k][pid] and, when `vis` is
// given, set bit 2*bounce+k of vis[pid] (for path replay).
void launch_extend_connect(const DevScene& S, const uint32_t* queue, const uint32_t* count_ext, uint32_t max_ext,
                           const float4* ray_o, const float4* ray_d, float4* hits, const uint32_t* count_sh,
                           uint32_t max_sh, const float4* sh_o, const float4* sh_d, const float4* sh_c, float4* ln0,
                           float4* ln1, uint32_t* fetch, uint32_t* ovf, uint32_t* vis, uint32_t bounce,
                           unsigned long long* stats, hipStream_t s, uint32_t max_blocks = 0);
// Caller rays (ox,oy,oz,tmin,dx,dy,dz,tmax) -> (t, prim|miss, u, v) / occluded flags.
// max_blocks != 0 caps the persistent grid (ovf then needs max_blocks * kTraceBlock
// * kStackOvf words instead of trace_overflow_bytes()).
void launch_trace_rays(const DevScene& S, const float4* rays, float4* hits, uint32_t n, uint32_t* fetch,
                       uint32_t* ovf, hipStream_t s, uint32_t max_blocks = 0);
void launch_occluded_rays(const DevScene& S, const float4* rays, uint32_t* out, uint32_t n, uint32_t* fetch,
                          uint32_t* ovf, hipStream_t s);

// ---- integrator (integrator.hip) ------------------------------------------
struct FrameParams {
    ohpt_camera cam;
    uint32_t width, height;
    uint32_t n_paths;          // paths of this launch (a lane: a contiguous range of the batch)
    uint32_t sample_base;      // sample index of the first sample of this batch
    uint32_t pid_base;         // first path id of the launch; pid = k*W*H + slot over the whole batch
    uint32_t max_bounces, rr_start, sampler, flags;
    float firefly_clamp, ray_eps;
    uint32_t row_groups;       // slot -> pixel: pixel_of_slot with this many row groups (0, 1: identity)
};

struct PathState {
    float4* o;        // ray origin
    float4* d;        // ray dir, w = previous BSDF pdf
    float4* T;        // throughput
    float4* L;        // radiance from emission / env hits
    float4* ln0;      // light NEE radiance
    float4* ln1;      // env NEE radiance
    float4* aov0;     // first-hit albedo.xyz, depth
    float4* aov1;     // first-hit normal.xyz, hit flag
    uint32_t* q[2];   // extend queues (ping-pong)
    float4* hits;
    float4* sh_o;
    float4* sh_d;
    float4* sh_c;
    uint32_t* counters;   // kCounterWords: extend counts, shadow counts
    uint32_t* fetch;      // kFetchWords per traversal launch: dynamic-fetch counters
    uint32_t capacity;
    // Adjoint only (null otherwise): closest hit of every path vertex, written by the
    // forward pass at [bounce * capacity + pid] and read back by the replay, which
    // then traces nothing.
    float4* hit_log;
};
// Queue lengths in pairs of words, one pair per traversal step b: word 2b the
// closest-hit rays of step b, word 2b + 1 the shadow rays that step b - 1
// queued (traced in the same launch; word 1 stays 0). A shading step queues
// both with one 64-bit addition (block_append).
constexpr uint32_t ext_counter(uint32_t b) { return 2u * b; }
constexpr uint32_t sh_counter(uint32_t b) { return 2u * b + 1u; }
constexpr uint32_t kCounterWords = 128;
constexpr uint32_t kMaxTraceLaunches = 64;        // traversal launches of one batch
// depth 60 steps to pair 61, the reference estimator's 2 + 2 * 30 steps to pair 62
static_assert(sh_counter(62) < kCounterWords && kCounterWords % 2 == 0, "counter pairs stay 8-byte aligned and inside their words");

// The dynamic-fetch counters of traversal launch b of a batch.
inline uint32_t* fetch_counters(const PathState& ps, uint32_t b) { return ps.fetch + (size_t)b * kFetchWords; }
// Zeroes the queue lengths and the fetch counters of the batch's first `launches` traversals.
void launch_clear_counters(const PathState& ps, uint32_t launches, hipStream_t s);
// Zeroes n float4 of each of five buffers.
void launch_clear_frame(float4* a, float4* b, float4* c, float4* d, float4* e, uint32_t n, hipStream_t s);
void launch_fill_u32(uint32_t* p, uint32_t v, uint32_t n, hipStream_t s);
void launch_generate(const FrameParams& f, const PathState& ps, hipStream_t s);
void launch_shade(const DevScene& S, const FrameParams& f, const PathState& ps, uint32_t bounce, hipStream_t s);
// The reference's own estimator in wavefront form (compat.hip). A batch of
// paths (pid = k * W * H + slot, as FrameParams) steps through the camera ray,
// the specular chain and the diffuse chain; step s traces every live path's
// closest-hit ray together with the shadow rays that step s - 1 emitted, then
// shades. Per-path arrays: o (origin, tmax), d (direction, pdf of the last
// direction), T (throughput, state bits), L (radiance, sample dimension; the
// sample's value once it ends), ln0 / ln1 (pending light / environment
// contribution, w 1 pending, 2 unoccluded), aov0.w (PCG state), aov1 (the
// camera ray's hit, from which the diffuse chain starts).
struct RefFrame {
    ohpt_camera cam;
    uint32_t width, height;
    uint32_t n_paths, sample_base, pid_base;
    uint32_t max_bounces, sampler, flags, revision;
    float firefly_clamp;
    uint32_t row_groups;
};
constexpr uint32_t kRefMaxBounces = 30;   // 2 + 2 * 30 steps fit the 64 counter slots
inline uint32_t ref_steps(uint32_t max_bounces) { return 2u + 2u * max_bounces; }
void launch_ref_generate(const RefFrame& f, const PathState& ps, hipStream_t s);
void launch_ref_shade(const DevScene& S, const RefFrame& f, const PathState& ps, uint32_t step, hipStream_t s);
void launch_ref_accumulate(const RefFrame& f, const PathState& ps, float4* accum, float4* moments, hipStream_t s);
// Closest-hit rays of the queue (t in [0.001, o.w]) and shadow rays (t in
// [0.001, sh_o.w]; unoccluded: ln0 / ln1[pid].w = 2), one persistent launch.
void launch_ref_trace(const DevScene& S, const uint32_t* queue, const uint32_t* count_ext, uint32_t max_ext,
                      const float4* ray_o, const float4* ray_d, float4* hits, const uint32_t* count_sh,
                      uint32_t max_sh, const float4* sh_o, const float4* sh_d, float4* ln0, float4* ln1,
                      uint32_t* fetch, uint32_t* ovf, hipStream_t s, uint32_t max_blocks = 0);
// Path-replay adjoint of one shading step (same random numbers, recorded visibility).
void launch_shade_adjoint(const DevScene& S, const FrameParams& f, const PathState& ps, uint32_t bounce,
                          const uint32_t* vis, float4* lrem, const float4* dl_dimage, float inv_spp,
                          uint32_t* rec_key, uint32_t* rec_val, uint32_t* rec_count, uint32_t* rec_overflow,
                          hipStream_t s);
// Deterministic mode: sums runs of equal keys (sorted records) into arena[key].
void launch_segment_reduce(const uint32_t* keys, const uint32_t* vals, uint32_t n, float* arena, hipStream_t s);
// Deterministic mode: compacts the records of nv path vertices (count[v] of them in
// vertex v's fixed slots) into okey/oval in vertex order; *total_out (host) = records.
// tiles: record_tiles(nv) + 1 words. Synchronous.
uint32_t record_tiles(uint32_t nv);
hipError_t compact_records(const uint32_t* count, uint32_t nv, const uint32_t* key, const uint32_t* val,
                           uint32_t* tiles, uint32_t* okey, uint32_t* oval, uint32_t* total_out, hipStream_t s);
// lrem[pid] = total radiance of path pid from the forward pass
// lrem[pid] = L + light-NEE + env-NEE radiance for pid in [pid_base, pid_base + n)
void launch_adjoint_init(const PathState& ps, uint32_t pid_base, uint32_t n, float4* lrem, hipStream_t s);
void launch_accumulate(const FrameParams& f, const PathState& ps, float4* accum, float4* moments,
                       float4* aov_albedo, float4* aov_normal, float4* disp, hipStream_t s);
void launch_resolve(const float4* accum, float4* out, uint32_t n, hipStream_t s);
void launch_tonemap(const float4* accum, uint8_t* out, uint32_t n, hipStream_t s);
void launch_resolve_aovs(const float4* accum, const float4* aov_albedo, const float4* aov_normal,
                         float* albedo, float* normal, float* depth, uint32_t n, hipStream_t s);

// ---- texel layout (texture.hip) ---------------------------------------------
// n texels of `channels` floats -> the packed copy (float4 per texel, missing
// channels 0 and a three-channel alpha 1; one float for one channel), and the mean
// of each of the first three channels as three doubles at the start of scratch.
size_t texel_mean_scratch_bytes();
void launch_texel_pack(const float* src, size_t n, uint32_t channels, float* packed, void* scratch, hipStream_t s);
// n packed float4 texels -> 2 or 3 floats each (1 and 4 channels are stored dense).
void launch_texel_unpack(const float* packed, size_t n, uint32_t channels, float* dst, hipStream_t s);

// ---- environment (env.hip) -------------------------------------------------
// Per-row luminance*sin(theta) prefix sums, normalised, plus marginal (env_cdf.cpp:13-61).
// Also fills the guide tables: marg_guide 2^env_guide_log2(H)+1 entries,
// cond_guide H rows of 2^env_guide_log2(W)+1 entries.
uint32_t env_guide_log2(uint32_t n);
hipError_t env_cdf_build(const float4* env, uint32_t W, uint32_t H, float* marg, float* cond,
                         float* row_sum, float* integral_dev, uint32_t* marg_guide, uint32_t* cond_guide,
                         hipStream_t s);
// Environment importance samples for inspection: u (n x 2) -> out (n x 4: dir.xyz, pdf; pdf 0 = no sample).
void launch_env_sample(const DevScene& S, const float* u, float4* out, uint32_t n, hipStream_t s);

// ---- variance-guided a-trous comparator (atrous.hip) ----------------------------
// The reference's SVGF spatial pass on the accumulated frame (mean display
// colour, display-luminance variance, first-hit AOVs): out = W*H RGBA32F
// display values in [0,1].
constexpr int kSvgfIterations = 5;           // steps 1, 2, 4, 8, 16 (atrous_denoise.cpp:29)
constexpr float kSvgfSigmaL = 0.4f;          // atrous_denoise.cpp:38-40
constexpr float kSvgfSigmaN = 0.30f;
constexpr float kSvgfSigmaD = 2.0f;
size_t svgf_scratch_bytes(uint32_t W, uint32_t H);
hipError_t svgf_atrous(const float4* accum, const float4* disp, const float4* aov_albedo,
                       const float4* aov_normal, uint32_t W, uint32_t H, float4* out, void* scratch,
                       hipStream_t s);

// ---- denoiser (denoiser.hip) ---------------------------------------------------
// Inference on device-resident guides (RGBA32F radiance/albedo/normal, F32
// depth; albedo/normal/depth may be null) into device RGBA32F `out`; returns
// an OHPT_* status. Synchronous.
int denoiser_infer_device(ohpt_denoiser* d, const float* rad, const float* alb, const float* nrm, const float* dep,
                          float* out, uint32_t width, uint32_t height);

// ---- host helpers shared by the C-ABI translation units --------------------
// Thread-local last-error message behind ohpt_last_error(); returns `code`.
int set_error(int code, const char* msg);
int set_hip_error(const char* what, hipError_t e);

// Owning device allocation that only grows.
struct DevBuf {
    void* p = nullptr;
    size_t bytes = 0;
    DevBuf() = default;
    DevBuf(const DevBuf&) = delete;
    DevBuf& operator=(const DevBuf&) = delete;
    DevBuf(DevBuf&& o) noexcept : p(o.p), bytes(o.bytes) { o.p = nullptr; o.bytes = 0; }
    DevBuf& operator=(DevBuf&& o) noexcept {
        if (this != &o) { release(); p = o.p; bytes = o.bytes; o.p = nullptr; o.bytes = 0; }
        return *this;
    }
    ~DevBuf() { release(); }
    void release() {
        if (p) (void)hipFree(p);
        p = nullptr;
        bytes = 0;
    }
    hipError_t ensure(size_t n) {
        if (n <= bytes && p) return hipSuccess;
        release();
        if (n == 0) return hipSuccess;
        hipError_t e = hipMalloc(&p, n);
        if (e == hipSuccess) bytes = n;
        else p = nullptr;
        return e;
    }
    template <class T> T* as() const { return reinterpret_cast<T*>(p); }
};

}  // namespace ohpt
