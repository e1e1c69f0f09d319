// C-ABI of the path-tracing core (include/ohpt.h). Host orchestration only:
// device memory, scene upload + LBVH commit, the wavefront frame loop on one
// HIP stream, readbacks and timing.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <deque>
#include <mutex>
#include <string>
#include <vector>

#include "ohpt_internal.h"

using namespace ohpt;

namespace {

thread_local std::string g_err;

int fail(int code, const std::string& msg) {
    g_err = msg;
    return code;
}
int fail_hip(const char* what, hipError_t e) {
    g_err = std::string(what) + ": " + hipGetErrorString(e);
    return OHPT_ERR_HIP;
}

}  // namespace

namespace ohpt {
int set_error(int code, const char* msg) { return fail(code, msg); }
int set_hip_error(const char* what, hipError_t e) { return fail_hip(what, e); }
}  // namespace ohpt

namespace {

#define HIPCHK(x)                                   \
    do {                                            \
        hipError_t e_ = (x);                        \
        if (e_ != hipSuccess) return fail_hip(#x, e_); \
    } while (0)

// Waits for the stream where a call returns early, so that no copy enqueued so far still
// reads or writes host memory that the call or its caller owns.
struct WaitOnError {
    hipStream_t stream;
    bool armed = true;
    ~WaitOnError() {
        if (armed) (void)hipStreamSynchronize(stream);
    }
};

struct TexStore {
    DevBuf data;
    uint32_t w = 0, h = 0, c = 0;
    double mean[3] = {0, 0, 0};   // mean texel per channel as sampled (one channel reads as grey)
    size_t packed_floats() const { return (size_t)w * h * (c >= 2 ? 4u : 1u); }
};

}  // namespace

struct ohpt_context {
    int device = 0;
    hipStream_t stream = nullptr;
    uint32_t W = 0, H = 0;

    // scene staging (host, caller's global triangle order)
    bool in_scene = false;
    // one record per added mesh: its object-space data and triangle range, so a
    // new world matrix can be applied later (ohpt_scene_set_mesh_transform)
    struct MeshRec {
        uint32_t base = 0, nt = 0;
        std::vector<float> pos, nrm, uv;   // object space, per vertex
        std::vector<uint32_t> idx;
        bool flat = false;              // idx is 0, 1, 2, ..: the vertices are the triangles' corners
        double world[16];               // the transform of the committed geometry
        bool has_world = false;
        // transform set by ohpt_scene_set_mesh_transform, applied by the next
        // refit: until then the emitter table stays that of the committed tree
        double next_world[16];
        bool next_has_world = false;
        bool pending = false;
        // device copies of pos / nrm / idx, uploaded at the mesh's first refit
        DevBuf d_vpos, d_vnrm, d_idx;
    };
    std::vector<MeshRec> meshes;
    bool refit_pending = false;   // a mesh transform changed since the last commit/refit
    std::vector<uint32_t> h_mat;
    bool any_nrm = false, any_uv = false;
    uint32_t n_tris = 0;
    bool committed = false;
    uint32_t tree_depth = 0;

    DevBuf d_nodes, d_nodes4, d_tris, d_attrs, d_prim, d_slot_of;
    uint32_t n_nodes4 = 0;
    // the committed scene's world-space triangles in add order (n*9 positions,
    // normals, n*6 uvs, n materials) and the LBVH scratch, kept for refits: filled from
    // the mesh records at the commit (the emitter table is computed from them too).
    DevBuf d_tpos, d_tnrm, d_tuv, d_tmat, d_lbvh_scratch;

    std::vector<ohpt_material> h_materials;
    DevBuf d_mats;
    std::vector<TexStore> textures;
    DevBuf d_texdesc;
    std::vector<ohpt_light> h_lights;
    DevBuf d_lights;
    DevBuf d_emit, d_emit_cdf;
    uint32_t n_emit = 0;
    float emit_total = 0.0f;

    DevBuf d_env, d_marg, d_cond, d_rowsum, d_integral, d_marg_guide, d_cond_guide;
    uint32_t env_w = 0, env_h = 0;
    float env_intensity = 1.0f;

    ohpt_camera cam{};
    ohpt_settings st{};
    uint32_t seed = 0;
    uint32_t sample_index = 0;
    // the accumulation holds samples of the reference estimator, which records
    // no first-hit guides or display sums (cleared with the accumulation)
    bool reference_samples = false;

    DevBuf d_accum, d_moments, d_aov_albedo, d_aov_normal, d_disp;

    // path state
    uint32_t capacity = 0;
    DevBuf ps_o, ps_d, ps_T, ps_L, ps_ln0, ps_ln1, ps_aov0, ps_aov1, ps_q0, ps_q1, ps_hits, sh_o, sh_d, sh_c,
        counters, ovf, tmp, tstats;   // ovf: fetch counters, then stack slots
    uint32_t ovf_rays = 0;
    DevBuf adj_vis, adj_lrem, adj_dldi, adj_hits;   // path-replay adjoint state
    DevBuf rec_key2, rec_val2, rec_count, rec_tiles; // deterministic mode: compacted records
    size_t grad_total = 0;                           // floats in the gradient arena (record keys are below it)
    DevBuf grad_arena;                      // dL/d(texel) of all textures, packed like the textures
    std::vector<size_t> grad_off;           // per-texture offset in the arena (floats)
    DevBuf rec_key, rec_val, rec_scratch;   // deterministic-mode gradient records
    DevBuf rec_flag;                        // set by a vertex with more records than its fixed slots
    DevBuf dn_guides, dn_out;               // resolved guides + output staging of ohpt_denoise

    hipEvent_t ev_start = nullptr, ev_stop = nullptr;
    std::vector<hipEvent_t> ev_pool;
    // A frame's paths split into kLanes independent wavefronts on their own
    // streams, so the tail of one lane's traversal overlaps the others' work.
    // Three lanes and the context stream use the four hardware queues a process
    // gets by default (GPU_MAX_HW_QUEUES): measured 3.00 ms per pipelined 1080p
    // frame against 3.07 ms with two lanes and 4.5 ms with four (queues shared).
#ifndef OHPT_LANES
#define OHPT_LANES 3
#endif
    static constexpr int kLanes = OHPT_LANES;
    // Concurrent lanes each run their persistent traversal grid at this share
    // (percent) of the full-occupancy grid, so one lane's launch does not hold
    // every slot of the GPU while the others' kernels wait for it to drain
    // (pipelined 1080p frame: 2.80 ms at 75 %, 2.83-2.96 at 85 %, 2.89 at 65 %,
    // 2.93 at 55 %, 3.03 with full grids).
#ifndef OHPT_LANE_GRID_PCT
#define OHPT_LANE_GRID_PCT 75
#endif
    static constexpr uint32_t kLaneGridPct = OHPT_LANE_GRID_PCT;
    hipStream_t lane_stream[kLanes] = {};
    hipEvent_t ev_fork = nullptr, ev_lane[kLanes] = {};
    // Frame pipelining: consecutive batches alternate between two copies of the
    // arrays the accumulation reads (radiance sums and first-hit guides), so a lane
    // starts its next batch while the other lane, or the accumulation of the last
    // batch, is still running. ev_acc[s] follows the last accumulation that read
    // copy s. stream_dirty: the context stream took other work since the lanes last
    // forked from it (an upload, a read, an adjoint), so the next lanes wait for it.
    int render_set = 0;
    hipEvent_t ev_acc[2] = {};
    bool acc_pending[2] = {false, false};
    bool stream_dirty = true;
    ohpt_stats stats{};
};

namespace {

// Prologue of every entry point but ohpt_render: the device, and the mark that
// the context stream is about to take work the next render's lanes must wait for.
hipError_t enter(ohpt_context* c) {
    c->stream_dirty = true;
    return hipSetDevice(c->device);
}

// Persistent traversal grid of one lane: the full grid for a lone wavefront,
// kLaneGridPct of it for each of several concurrent lanes.
uint32_t lane_trace_blocks(int nl) {
    if (nl <= 1) return 0u;
    return std::max<uint32_t>(1u, trace_grid_blocks() * ohpt_context::kLaneGridPct / 100u);
}

DevScene scene_view(ohpt_context* c) {
    DevScene S{};
    S.nodes4 = c->d_nodes4.as<float4>();
    S.tris = c->d_tris.as<float4>();
    S.attrs = c->d_attrs.as<float4>();
    S.n_tris = c->committed ? c->n_tris : 0u;
    S.n_materials = (uint32_t)std::max<size_t>(c->h_materials.size(), 1);
    S.mats = c->d_mats.as<float4>();
    S.tex = c->d_texdesc.as<TexDesc>();
    S.n_tex = (uint32_t)c->textures.size();
    S.n_lights = (uint32_t)c->h_lights.size();
    S.lights = c->d_lights.as<float4>();
    S.emit = c->d_emit.as<float4>();
    S.emit_cdf = c->d_emit_cdf.as<float>();
    S.n_emit = c->n_emit;
    S.emit_total = c->emit_total;
    S.env = c->d_env.as<float4>();
    S.env_marg = c->d_marg.as<float>();
    S.env_cond = c->d_cond.as<float>();
    S.env_marg_guide = c->d_marg_guide.as<uint32_t>();
    S.env_cond_guide = c->d_cond_guide.as<uint32_t>();
    S.env_marg_log2 = env_guide_log2(c->env_h);
    S.env_cond_log2 = env_guide_log2(c->env_w);
    S.env_w = c->env_w;
    S.env_h = c->env_h;
    S.env_intensity = c->env_intensity;
    return S;
}

int alloc_frame(ohpt_context* c) {
    const size_t npix = (size_t)c->W * c->H;
    HIPCHK(c->d_accum.ensure(npix * 16));
    HIPCHK(c->d_moments.ensure(npix * 16));
    HIPCHK(c->d_aov_albedo.ensure(npix * 16));
    HIPCHK(c->d_aov_normal.ensure(npix * 16));
    HIPCHK(c->d_disp.ensure(npix * 16));
    return OHPT_OK;
}

int clear_frame(ohpt_context* c) {
    const size_t npix = (size_t)c->W * c->H;
    launch_clear_frame(c->d_accum.as<float4>(), c->d_moments.as<float4>(), c->d_aov_albedo.as<float4>(),
                       c->d_aov_normal.as<float4>(), c->d_disp.as<float4>(), (uint32_t)npix, c->stream);
    HIPCHK(hipGetLastError());
    c->reference_samples = false;
    return OHPT_OK;
}

// Guide buffers (first-hit albedo / normal / depth, display sums) exist only for
// samples of the physically based integrator.
int need_guides(const ohpt_context* c, const char* what) {
    if (c->reference_samples)
        return fail(OHPT_ERR_STATE, std::string(what) +
                                        ": the accumulation holds reference-estimator samples, which record no "
                                        "first-hit guides (reset and render with the physically based integrator)");
    return OHPT_OK;
}

// Fetch counters of the traversals (every lane's), then the stack overflow slots of the
// first `lanes` lanes, in one allocation that only grows: from the one lane of a ray query,
// which waits for its traversal, to every lane of a render or an adjoint, in ensure_paths,
// which waits for all streams first. So it is never replaced under a launch in flight.
constexpr size_t kTraceFetchWords = (size_t)kFetchWords * kMaxTraceLaunches * ohpt_context::kLanes;
hipError_t ensure_trace_scratch(ohpt_context* c, int lanes) {
    return c->ovf.ensure(kTraceFetchWords * 4 + trace_overflow_bytes() * (size_t)lanes);
}
uint32_t* trace_fetch(ohpt_context* c) { return c->ovf.as<uint32_t>(); }

int ensure_paths(ohpt_context* c, uint32_t n) {
    if (n <= c->capacity) return OHPT_OK;
    // the buffers are replaced: nothing in flight may still use them
    HIPCHK(hipStreamSynchronize(c->stream));
    for (int l = 0; l < ohpt_context::kLanes; ++l) HIPCHK(hipStreamSynchronize(c->lane_stream[l]));
    c->acc_pending[0] = c->acc_pending[1] = false;
    c->stream_dirty = true;
    c->capacity = 0;   // until every buffer has its new size
    const size_t N = n;
    HIPCHK(c->ps_o.ensure(N * 16));
    HIPCHK(c->ps_d.ensure(N * 16));
    HIPCHK(c->ps_T.ensure(N * 16));
    HIPCHK(c->ps_L.ensure(2 * N * 16));     // two copies (render_set)
    HIPCHK(c->ps_ln0.ensure(2 * N * 16));
    HIPCHK(c->ps_ln1.ensure(2 * N * 16));
    HIPCHK(c->ps_aov0.ensure(2 * N * 16));
    HIPCHK(c->ps_aov1.ensure(2 * N * 16));
    HIPCHK(c->ps_q0.ensure(N * 4));
    HIPCHK(c->ps_q1.ensure(N * 4));
    HIPCHK(c->ps_hits.ensure(N * 16));
    HIPCHK(c->sh_o.ensure(2 * N * 16));
    HIPCHK(c->sh_d.ensure(2 * N * 16));
    HIPCHK(c->sh_c.ensure(2 * N * 16));
    HIPCHK(c->counters.ensure((size_t)kCounterWords * 4 * ohpt_context::kLanes));
    HIPCHK(ensure_trace_scratch(c, ohpt_context::kLanes));
    c->ovf_rays = 2 * n;
    c->capacity = n;
    return OHPT_OK;
}

// Lane `lane` of a batch: paths [pid_base, pid_base + n) share the per-path
// arrays; its queues, hits and shadow rays use the matching ranges of the
// batch-sized buffers, its counters and stack overflow slots are its own.
PathState lane_view(const PathState& ps, uint32_t pid_base, int lane) {
    PathState p = ps;
    p.q[0] = ps.q[0] + pid_base;
    p.q[1] = ps.q[1] + pid_base;
    p.hits = ps.hits + pid_base;
    p.sh_o = ps.sh_o + 2 * (size_t)pid_base;
    p.sh_d = ps.sh_d + 2 * (size_t)pid_base;
    p.sh_c = ps.sh_c + 2 * (size_t)pid_base;
    p.counters = ps.counters + (size_t)lane * kCounterWords;
    p.fetch = ps.fetch + (size_t)lane * kMaxTraceLaunches * kFetchWords;
    return p;
}

uint32_t* lane_ovf(ohpt_context* c, int lane) {
    return c->ovf.as<uint32_t>() + kTraceFetchWords + (size_t)lane * (trace_overflow_bytes() / 4);
}

// set: which copy of the arrays the accumulation reads (0 or 1)
PathState path_state(ohpt_context* c, int set = 0) {
    PathState p{};
    const size_t off = (size_t)set * c->capacity;
    p.o = c->ps_o.as<float4>();
    p.d = c->ps_d.as<float4>();
    p.T = c->ps_T.as<float4>();
    p.L = c->ps_L.as<float4>() + off;
    p.ln0 = c->ps_ln0.as<float4>() + off;
    p.ln1 = c->ps_ln1.as<float4>() + off;
    p.aov0 = c->ps_aov0.as<float4>() + off;
    p.aov1 = c->ps_aov1.as<float4>() + off;
    p.q[0] = c->ps_q0.as<uint32_t>();
    p.q[1] = c->ps_q1.as<uint32_t>();
    p.hits = c->ps_hits.as<float4>();
    p.sh_o = c->sh_o.as<float4>();
    p.sh_d = c->sh_d.as<float4>();
    p.sh_c = c->sh_c.as<float4>();
    p.counters = c->counters.as<uint32_t>();
    p.fetch = trace_fetch(c);
    p.capacity = c->capacity;
    return p;
}

float id_bits(int32_t id) {
    float f;
    std::memcpy(&f, &id, 4);
    return f;
}

// Mean luminance of a material's emitted radiance (emissive x the emissive
// texture's channel means): the weight of its triangles in the emitter table.
double emit_weight(const ohpt_context* c, const ohpt_material& m) {
    double e[3] = {m.emissive[0], m.emissive[1], m.emissive[2]};
    if (m.emissive_tex >= 0 && (size_t)m.emissive_tex < c->textures.size())
        for (int k = 0; k < 3; ++k) e[k] *= c->textures[(size_t)m.emissive_tex].mean[k];
    return 0.2126 * e[0] + 0.7152 * e[1] + 0.0722 * e[2];
}

int upload_materials_dev(ohpt_context* c) {
    const size_t n = std::max<size_t>(c->h_materials.size(), 1);
    HIPCHK(c->d_mats.ensure(n * 64));
    std::vector<float4> packed(n * 4, make_float4(0, 0, 0, 0));
    for (size_t i = 0; i < c->h_materials.size(); ++i) {
        const ohpt_material& m = c->h_materials[i];
        packed[i * 4 + 0] = make_float4(m.base_color[0], m.base_color[1], m.base_color[2], m.roughness);
        packed[i * 4 + 1] = make_float4(m.metallic, m.specular_f0, m.emissive[0], m.emissive[1]);
        packed[i * 4 + 2] = make_float4(m.emissive[2], id_bits(m.albedo_tex), id_bits(m.roughness_tex),
                                        id_bits(m.metallic_tex));
        packed[i * 4 + 3] = make_float4(id_bits(m.normal_tex), id_bits(m.orm_tex), id_bits(m.emissive_tex),
                                        (float)emit_weight(c, m));
    }
    if (c->h_materials.empty()) {
        const float none = id_bits(-1);
        packed[0] = make_float4(0.8f, 0.8f, 0.8f, 0.5f);
        packed[1] = make_float4(0.0f, 0.04f, 0.0f, 0.0f);
        packed[2] = make_float4(0.0f, none, none, none);
        packed[3] = make_float4(none, none, none, 0.0f);
    }
    HIPCHK(hipMemcpyAsync(c->d_mats.p, packed.data(), packed.size() * 16, hipMemcpyHostToDevice, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    return OHPT_OK;
}

// World matrix and normal matrix (inverse transpose of the upper 3x3,
// pt_closesthit.rchit:66) of a mesh record.
MeshTransform mesh_transform(const ohpt_context::MeshRec& m) {
    MeshTransform x{};
    const double* M = m.world;
    for (int k = 0; k < 16; ++k) x.m[k] = M[k];
    x.has_world = m.has_world ? 1 : 0;
    const double a = M[0], b = M[4], cc = M[8], d = M[1], e = M[5], f = M[9], g = M[2], h = M[6], i = M[10];
    const double det = a * (e * i - f * h) - b * (d * i - f * g) + cc * (d * h - e * g);
    double* N = x.n;   // row-major, applied as n' = N n
    N[0] = 1; N[1] = 0; N[2] = 0; N[3] = 0; N[4] = 1; N[5] = 0; N[6] = 0; N[7] = 0; N[8] = 1;
    if (std::fabs(det) > 0) {
        N[0] = (e * i - f * h) / det; N[1] = -(d * i - f * g) / det; N[2] = (d * h - e * g) / det;
        N[3] = -(b * i - cc * h) / det; N[4] = (a * i - cc * g) / det; N[5] = -(a * h - b * g) / det;
        N[6] = (b * f - cc * e) / det; N[7] = -(a * f - cc * d) / det; N[8] = (a * e - b * d) / det;
    }
    return x;
}

// World-space corners P (9 floats) of triangle t of mesh m and, when
// `normals`, its corner normals Nn (the transformed vertex normals, or the
// geometric normal for a mesh without them). The arithmetic of
// k_transform_mesh, which does the same on the device for refits.
void world_triangle(const ohpt_context::MeshRec& m, const MeshTransform& x, uint32_t t, bool normals, float P[9],
                    float Nn[9]) {
    const double* M = x.m;
    const double* N = x.n;
    const bool has_n = !m.nrm.empty();
    for (int k = 0; k < 3; ++k) {
        const uint32_t vi = m.idx[(size_t)t * 3 + k];
        const double px = m.pos[(size_t)vi * 3], py = m.pos[(size_t)vi * 3 + 1], pz = m.pos[(size_t)vi * 3 + 2];
        if (x.has_world) {
            P[k * 3 + 0] = (float)(M[0] * px + M[4] * py + M[8] * pz + M[12]);
            P[k * 3 + 1] = (float)(M[1] * px + M[5] * py + M[9] * pz + M[13]);
            P[k * 3 + 2] = (float)(M[2] * px + M[6] * py + M[10] * pz + M[14]);
        } else {
            P[k * 3 + 0] = (float)px; P[k * 3 + 1] = (float)py; P[k * 3 + 2] = (float)pz;
        }
        if (normals && has_n) {
            const double nx = m.nrm[(size_t)vi * 3], ny = m.nrm[(size_t)vi * 3 + 1], nz = m.nrm[(size_t)vi * 3 + 2];
            double o0 = nx, o1 = ny, o2 = nz;
            if (x.has_world) {
                o0 = N[0] * nx + N[1] * ny + N[2] * nz;
                o1 = N[3] * nx + N[4] * ny + N[5] * nz;
                o2 = N[6] * nx + N[7] * ny + N[8] * nz;
            }
            Nn[k * 3 + 0] = (float)o0; Nn[k * 3 + 1] = (float)o1; Nn[k * 3 + 2] = (float)o2;
        }
    }
    if (normals && !has_n) {
        const float e1[3] = {P[3] - P[0], P[4] - P[1], P[5] - P[2]}, e2[3] = {P[6] - P[0], P[7] - P[1], P[8] - P[2]};
        const float n[3] = {e1[1] * e2[2] - e1[2] * e2[1], e1[2] * e2[0] - e1[0] * e2[2], e1[0] * e2[1] - e1[1] * e2[0]};
        for (int k = 0; k < 3; ++k) for (int q = 0; q < 3; ++q) Nn[k * 3 + q] = n[q];
    }
}

// Emitter table: triangles whose material emits, weighted by area x the
// material's emitter weight; each record carries the vertices and uvs. The
// emitting triangles' world positions come from their mesh records with the
// meshes' current transforms (a refit moves geometry on the device only).
int build_emitters(ohpt_context* c) {
    c->n_emit = 0;
    c->emit_total = 0.0f;
    if (!c->committed || c->h_materials.empty()) return OHPT_OK;
    std::vector<double> mw(c->h_materials.size());
    bool any = false;
    for (size_t k = 0; k < mw.size(); ++k) {
        mw[k] = emit_weight(c, c->h_materials[k]);
        any |= mw[k] > 0;
    }
    if (!any) return OHPT_OK;
    std::vector<float4> rec;
    std::vector<double> w;
    double total = 0.0;
    for (const ohpt_context::MeshRec& m : c->meshes) {
      const MeshTransform x = mesh_transform(m);
      for (uint32_t tri = 0; tri < m.nt; ++tri) {
        const uint32_t i = m.base + tri;
        const uint32_t mi = c->h_mat.empty() ? 0u : c->h_mat[i];
        if (mi >= c->h_materials.size()) continue;
        const double l = mw[mi];
        if (!(l > 0)) continue;
        float t[9], q[9];
        world_triangle(m, x, tri, c->any_nrm, t, q);
        const double e1[3] = {(double)t[3] - t[0], (double)t[4] - t[1], (double)t[5] - t[2]};
        const double e2[3] = {(double)t[6] - t[0], (double)t[7] - t[1], (double)t[8] - t[2]};
        const double cx = e1[1] * e2[2] - e1[2] * e2[1], cy = e1[2] * e2[0] - e1[0] * e2[2],
                     cz = e1[0] * e2[1] - e1[1] * e2[0];
        const double area = 0.5 * std::sqrt(cx * cx + cy * cy + cz * cz);
        if (!(area > 0)) continue;
        // vertex normals define the emitting side: store the triangle with
        // vertices 1 and 2 swapped when the normals oppose the winding
        bool sw = false;
        if (c->any_nrm) {
            const double nx = (double)q[0] + q[3] + q[6], ny = (double)q[1] + q[4] + q[7],
                         nz = (double)q[2] + q[5] + q[8];
            sw = nx * nx + ny * ny + nz * nz > 1e-24 && cx * nx + cy * ny + cz * nz < 0;
        }
        const float* v1 = t + (sw ? 6 : 3);
        const float* v2 = t + (sw ? 3 : 6);
        float mb;
        std::memcpy(&mb, &mi, 4);
        rec.push_back(make_float4(t[0], t[1], t[2], (float)area));
        rec.push_back(make_float4(v1[0], v1[1], v1[2], mb));
        rec.push_back(make_float4(v2[0], v2[1], v2[2], 0.0f));
        float uv[6] = {0, 0, 0, 0, 0, 0};
        if (!m.uv.empty())
            for (int k = 0; k < 3; ++k)
                std::memcpy(uv + 2 * k, &m.uv[(size_t)m.idx[(size_t)tri * 3 + k] * 2], 8);
        const float* u1 = uv + (sw ? 4 : 2);
        const float* u2 = uv + (sw ? 2 : 4);
        rec.push_back(make_float4(uv[0], uv[1], u1[0], u1[1]));
        rec.push_back(make_float4(u2[0], u2[1], 0.0f, 0.0f));
        w.push_back(area * l);
        total += area * l;
      }
    }
    if (rec.empty()) return OHPT_OK;
    std::vector<float> cdf(w.size());
    double acc = 0;
    for (size_t i = 0; i < w.size(); ++i) { acc += w[i]; cdf[i] = (float)(acc / total); }
    cdf.back() = 1.0f;
    HIPCHK(c->d_emit.ensure(rec.size() * 16));
    HIPCHK(c->d_emit_cdf.ensure(cdf.size() * 4));
    HIPCHK(hipMemcpyAsync(c->d_emit.p, rec.data(), rec.size() * 16, hipMemcpyHostToDevice, c->stream));
    HIPCHK(hipMemcpyAsync(c->d_emit_cdf.p, cdf.data(), cdf.size() * 4, hipMemcpyHostToDevice, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    c->n_emit = (uint32_t)w.size();
    c->emit_total = (float)total;
    return OHPT_OK;
}

int upload_texdesc(ohpt_context* c) {
    std::vector<TexDesc> td(std::max<size_t>(c->textures.size(), 1));
    for (size_t i = 0; i < c->textures.size(); ++i) {
        td[i].data = c->textures[i].data.as<float>();
        const bool has_grad = c->grad_arena.p && i < c->grad_off.size();
        td[i].grad = has_grad ? c->grad_arena.as<float>() + c->grad_off[i] : nullptr;
        td[i].grad_base = has_grad ? (uint32_t)c->grad_off[i] : 0u;
        td[i].w = c->textures[i].w;
        td[i].h = c->textures[i].h;
        td[i].c = c->textures[i].c;
    }
    HIPCHK(c->d_texdesc.ensure(td.size() * sizeof(TexDesc)));
    HIPCHK(hipMemcpyAsync(c->d_texdesc.p, td.data(), td.size() * sizeof(TexDesc), hipMemcpyHostToDevice,
                          c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    return OHPT_OK;
}

// ---- scratch of the no-allocation ray query (ohpt_trace_rays_noalloc) ------
// One array per device, in the code object: the traversal's dynamic-fetch
// counters (first 8 KiB) and the per-thread stack-overflow slots of a
// persistent grid of kNoAllocBlocks blocks (36 MiB + 8 KiB). Host code never
// uses the array's name as an address: ohpt_create resolves each device's
// copy with hipGetSymbolAddress once, and the kernels receive that pointer.
constexpr uint32_t kNoAllocBlocks = 1024;
constexpr size_t kNoAllocOvfBytes = (size_t)kNoAllocBlocks * kTraceBlock * kStackOvf * 4;
constexpr size_t kNoAllocScratchBytes = kFetchWords * 4 + kNoAllocOvfBytes;
constexpr uint32_t kNoAllocMaxRays = 1u << 31;   // keeps the 32-bit fetch counter from wrapping
constexpr int kMaxDevices = 64;
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];
void* g_scratch_dev[kMaxDevices] = {};
std::mutex g_scratch_mu;

// With `device` current: resolves and keeps that device's address of `scratch`.
int noalloc_scratch_setup(int device) {
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (device < 0 || device >= kMaxDevices) return fail(OHPT_ERR_UNSUPPORTED, "ohpt_create: device index above 63");
    if (g_scratch_dev[device]) return OHPT_OK;
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return fail_hip("hipGetSymbolAddress(scratch)", e);
    g_scratch_dev[device] = p;
    return OHPT_OK;
}

void* noalloc_scratch(int device) {
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    return (device >= 0 && device < kMaxDevices) ? g_scratch_dev[device] : nullptr;
}

double elapsed(hipEvent_t a, hipEvent_t b) {
    float ms = 0.0f;
    if (hipEventElapsedTime(&ms, a, b) != hipSuccess) return 0.0;
    return ms;
}

// Calls that read the committed tree: OHPT_ERR_STATE while a scene is being
// staged (ohpt_scene_begin dropped the old tree), OHPT_ERR_NO_SCENE before the
// first commit.
int need_tree(const ohpt_context* c, const char* what) {
    if (c->in_scene)
        return fail(OHPT_ERR_STATE, std::string(what) + ": a scene is being staged (call ohpt_scene_commit)");
    if (!c->committed) return fail(OHPT_ERR_NO_SCENE, std::string(what) + ": no committed scene");
    return OHPT_OK;
}

}  // namespace

extern "C" {

const char* ohpt_last_error(void) { return g_err.c_str(); }
int ohpt_abi_version(void) { return OHPT_ABI_VERSION; }

int ohpt_create(ohpt_context** out, int device, uint32_t width, uint32_t height) {
    if (!out || width == 0 || height == 0) return fail(OHPT_ERR_INVALID_ARG, "ohpt_create: bad arguments");
    *out = nullptr;
    int ndev = 0;
    HIPCHK(hipGetDeviceCount(&ndev));
    if (device < 0 || device >= ndev) return fail(OHPT_ERR_INVALID_ARG, "ohpt_create: no such device");
    HIPCHK(hipSetDevice(device));
    if (int r0 = noalloc_scratch_setup(device)) return r0;
    auto* c = new ohpt_context();
    c->device = device;
    c->W = width;
    c->H = height;
    bool ok = hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) == hipSuccess &&
              hipEventCreate(&c->ev_start) == hipSuccess && hipEventCreate(&c->ev_stop) == hipSuccess &&
              hipEventCreateWithFlags(&c->ev_fork, hipEventDisableTiming) == hipSuccess &&
              hipEventCreateWithFlags(&c->ev_acc[0], hipEventDisableTiming) == hipSuccess &&
              hipEventCreateWithFlags(&c->ev_acc[1], hipEventDisableTiming) == hipSuccess;
    for (int l = 0; ok && l < ohpt_context::kLanes; ++l)
        ok = hipStreamCreateWithFlags(&c->lane_stream[l], hipStreamNonBlocking) == hipSuccess &&
             hipEventCreateWithFlags(&c->ev_lane[l], hipEventDisableTiming) == hipSuccess;
    if (!ok) {
        ohpt_destroy(c);
        return fail(OHPT_ERR_HIP, "ohpt_create: stream/event creation failed");
    }
    // reference offline defaults: maxBounces 4, Sobol sampler, RR after bounce 1 (rt_settings.hpp:50-61)
    c->st.max_bounces = 4;
    c->st.rr_start = 2;
    c->st.sampler = OHPT_SAMPLER_SOBOL_OWEN;
    c->st.flags = OHPT_FLAG_AOVS;
    // reference Camera defaults: position (0,0,2.5), yaw -90, pitch 0, fov 45 (camera.cpp:16-22)
    c->cam = ohpt_camera{{0.0f, 0.0f, 2.5f}, {0.0f, 0.0f, -1.0f}, {1.0f, 0.0f, 0.0f}, {0.0f, 1.0f, 0.0f},
                         (float)std::tan(45.0 * M_PI / 360.0)};
    int r = alloc_frame(c);
    if (r == OHPT_OK) r = clear_frame(c);
    if (r == OHPT_OK) r = upload_materials_dev(c);
    if (r == OHPT_OK) r = upload_texdesc(c);
    if (r != OHPT_OK) { ohpt_destroy(c); return r; }
    *out = c;
    return OHPT_OK;
}

int ohpt_destroy(ohpt_context* c) {
    if (!c) return fail(OHPT_ERR_INVALID_ARG, "ohpt_destroy: null context");
    (void)hipSetDevice(c->device);
    if (c->stream) (void)hipStreamSynchronize(c->stream);
    for (int l = 0; l < ohpt_context::kLanes; ++l)
        if (c->lane_stream[l]) (void)hipStreamSynchronize(c->lane_stream[l]);
    for (auto e : c->ev_pool) (void)hipEventDestroy(e);
    if (c->ev_start) (void)hipEventDestroy(c->ev_start);
    if (c->ev_stop) (void)hipEventDestroy(c->ev_stop);
    if (c->ev_fork) (void)hipEventDestroy(c->ev_fork);
    for (auto e : c->ev_acc)
        if (e) (void)hipEventDestroy(e);
    for (int l = 0; l < ohpt_context::kLanes; ++l) {
        if (c->ev_lane[l]) (void)hipEventDestroy(c->ev_lane[l]);
        if (c->lane_stream[l]) (void)hipStreamDestroy(c->lane_stream[l]);
    }
    if (c->stream) (void)hipStreamDestroy(c->stream);
    delete c;
    return OHPT_OK;
}

int ohpt_resize(ohpt_context* c, uint32_t width, uint32_t height) {
    if (!c || width == 0 || height == 0) return fail(OHPT_ERR_INVALID_ARG, "ohpt_resize: bad arguments");
    HIPCHK(enter(c));
    HIPCHK(hipStreamSynchronize(c->stream));
    c->W = width;
    c->H = height;
    int r = alloc_frame(c);
    if (r != OHPT_OK) return r;
    c->sample_index = c->seed;
    return clear_frame(c);
}

// ---------------------------------------------------------------- scene
extern "C++" {
namespace {
// Staging of this size stays with the context for the next upload; a call that needed more
// gives it back once its copies and kernels are done.
constexpr size_t kKeptStaging = 256u << 20;
void give_back(ohpt_context* c, size_t needed) {
    if (needed > kKeptStaging) c->tmp.release();
}

// Runs of meshes below kHostMeshTriangles are expanded on the host: the four
// copies of a mesh take about as long as this loop over that many triangles, so a scene
// of many small meshes is uploaded in few copies.
constexpr uint32_t kHostMeshTriangles = 2048;
struct MeshRun {
    size_t base = 0;
    std::vector<float> pos, nrm, uv;
};

// Meshes [begin, end), which follow one another in the scene, into r.
void expand_meshes(const ohpt_context* c, size_t begin, size_t end, MeshRun& r) {
    size_t n = 0;
    for (size_t i = begin; i < end; ++i) n += c->meshes[i].nt;
    r.base = c->meshes[begin].base;
    r.pos.resize(n * 9);
    if (c->any_nrm) r.nrm.resize(n * 9);
    if (c->any_uv) r.uv.resize(n * 6);
    float *P = r.pos.data(), *N = r.nrm.data(), *U = r.uv.data();
    for (size_t i = begin; i < end; ++i) {
        const ohpt_context::MeshRec& m = c->meshes[i];
        const MeshTransform x = mesh_transform(m);
        for (uint32_t t = 0; t < m.nt; ++t, P += 9) {
            world_triangle(m, x, t, c->any_nrm, P, N);
            if (c->any_nrm) N += 9;
            if (!c->any_uv) continue;
            for (int k = 0; !m.uv.empty() && k < 3; ++k)
                std::memcpy(U + 2 * k, &m.uv[(size_t)m.idx[(size_t)t * 3 + k] * 2], 8);
            U += 6;
        }
    }
}

int place_run(ohpt_context* c, const MeshRun& r) {
    auto up = [&](const DevBuf& dst, size_t per, const std::vector<float>& v) {
        return v.empty() ? hipSuccess
                         : hipMemcpyAsync(dst.as<float>() + r.base * per, v.data(), v.size() * 4, hipMemcpyHostToDevice,
                                          c->stream);
    };
    HIPCHK(up(c->d_tpos, 9, r.pos));
    HIPCHK(up(c->d_tnrm, 9, r.nrm));
    HIPCHK(up(c->d_tuv, 6, r.uv));
    return OHPT_OK;
}

// World-space corners, normals and uvs of one mesh record into the scene's device
// arrays. A mesh whose vertices are its triangles' corners in order, untransformed, is
// copied as it is; the others are gathered on the device from their vertices.
// (Loading the 200,000-triangle lantern, one flat mesh: 5.5 -> 3.9 ms; the host expanded
// every corner in double, into zeroed arrays, before the copy.)
// staged: grows to the staging bytes it used.
int place_mesh(ohpt_context* c, const ohpt_context::MeshRec& m, size_t& staged) {
    if (m.nt == 0) return OHPT_OK;
    float* const tpos = c->d_tpos.as<float>() + (size_t)m.base * 9;
    float* const tnrm = c->any_nrm ? c->d_tnrm.as<float>() + (size_t)m.base * 9 : nullptr;
    float* const tuv = c->any_uv ? c->d_tuv.as<float>() + (size_t)m.base * 6 : nullptr;
    const size_t corners = (size_t)m.nt * 3;
    auto up = [&](void* dst, const void* src, size_t bytes) {
        return hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, c->stream);
    };
    if (m.flat && !m.has_world && (!tnrm || !m.nrm.empty()) && (!tuv || !m.uv.empty())) {
        HIPCHK(up(tpos, m.pos.data(), corners * 12));
        if (tnrm) HIPCHK(up(tnrm, m.nrm.data(), corners * 12));
        if (tuv) HIPCHK(up(tuv, m.uv.data(), corners * 8));
        return OHPT_OK;
    }
    const size_t pb = m.pos.size() * 4, nb = m.nrm.size() * 4, ub = m.uv.size() * 4, ib = corners * 4;
    auto pad = [](size_t b) { return (b + 15) & ~size_t(15); };
    const size_t bytes = pad(pb) + pad(nb) + pad(ub) + ib;
    staged = std::max(staged, bytes);
    HIPCHK(c->tmp.ensure(bytes));
    char* const dp = c->tmp.as<char>();
    char* const dn = dp + pad(pb);
    char* const du = dn + pad(nb);
    char* const di = du + pad(ub);
    HIPCHK(up(dp, m.pos.data(), pb));
    if (nb) HIPCHK(up(dn, m.nrm.data(), nb));
    if (ub) HIPCHK(up(du, m.uv.data(), ub));
    HIPCHK(up(di, m.idx.data(), ib));
    const uint32_t* const idx = reinterpret_cast<const uint32_t*>(di);
    launch_transform_mesh(reinterpret_cast<const float*>(dp), nb ? reinterpret_cast<const float*>(dn) : nullptr, idx,
                          m.nt, mesh_transform(m), tpos, tnrm, c->stream);
    if (tuv) launch_gather_uv(ub ? reinterpret_cast<const float*>(du) : nullptr, idx, m.nt, tuv, c->stream);
    HIPCHK(hipGetLastError());
    return OHPT_OK;
}
}  // namespace
}  // extern "C++"

// Staging replaces the host copy of the committed scene, so the committed tree
// is dropped here: until ohpt_scene_commit, calls that read the tree
// (render, adjoint, refit, exports, ray queries) return OHPT_ERR_STATE.
int ohpt_scene_begin(ohpt_context* c) {
    if (!c) return fail(OHPT_ERR_INVALID_ARG, "ohpt_scene_begin: null context");
    HIPCHK(enter(c));
    HIPCHK(hipStreamSynchronize(c->stream));
    c->in_scene = true;
    c->committed = false;
    c->n_nodes4 = 0;
    c->tree_depth = 0;
    c->n_emit = 0;
    c->emit_total = 0.0f;
    c->refit_pending = false;
    c->meshes.clear();
    c->h_mat.clear();
    c->any_nrm = c->any_uv = false;
    c->n_tris = 0;
    return OHPT_OK;
}

int ohpt_scene_add_mesh(ohpt_context* c, const float* positions, const float* normals, const float* uvs,
                        uint32_t nv, const uint32_t* indices, uint32_t nt, const uint32_t* mat_ids,
                        uint32_t material_base, const float* world) {
    if (!c || !c->in_scene) return fail(OHPT_ERR_STATE, "ohpt_scene_add_mesh: call ohpt_scene_begin first");
    if (!positions || (nt && !indices)) return fail(OHPT_ERR_INVALID_ARG, "ohpt_scene_add_mesh: null arrays");
    if ((uint64_t)c->n_tris + nt >= 0x7FFFFFFFull) return fail(OHPT_ERR_INVALID_ARG, "ohpt_scene_add_mesh: too many triangles");
    uint32_t top = 0, off = 0;   // largest index; bits by which any index differs from its position
    for (size_t i = 0; i < (size_t)nt * 3; ++i) {
        top = std::max(top, indices[i]);
        off |= indices[i] ^ (uint32_t)i;
    }
    if (nt && top >= nv) return fail(OHPT_ERR_INVALID_ARG, "ohpt_scene_add_mesh: index out of range");
    const size_t base = c->n_tris;
    ohpt_context::MeshRec rec;
    rec.base = (uint32_t)base;
    rec.nt = nt;
    rec.flat = off == 0 && (uint64_t)nt * 3 <= 0xFFFFFFFFull;
    rec.pos.assign(positions, positions + (size_t)nv * 3);
    if (normals) rec.nrm.assign(normals, normals + (size_t)nv * 3);
    if (uvs) rec.uv.assign(uvs, uvs + (size_t)nv * 2);
    rec.idx.assign(indices, indices + (size_t)nt * 3);
    rec.has_world = world != nullptr;
    for (int k = 0; k < 16; ++k) rec.world[k] = world ? (double)world[k] : (k % 5 == 0 ? 1.0 : 0.0);
    if (normals) c->any_nrm = true;
    if (uvs) c->any_uv = true;
    c->h_mat.resize(base + nt);
    for (uint32_t t = 0; t < nt; ++t) c->h_mat[base + t] = material_base + (mat_ids ? mat_ids[t] : 0u);
    c->meshes.push_back(std::move(rec));
    c->n_tris += nt;
    return OHPT_OK;
}

int ohpt_scene_commit(ohpt_context* c) {
    if (!c || !c->in_scene) return fail(OHPT_ERR_STATE, "ohpt_scene_commit: no scene begun");
    HIPCHK(enter(c));
    const uint32_t n = c->n_tris;
    c->committed = false;
    if (n == 0) {
        c->committed = true;
        c->in_scene = false;
        c->tree_depth = 0;
        c->n_nodes4 = 0;
        return build_emitters(c);
    }
    // the copies read the runs and the staged meshes until the stream has been waited for
    std::deque<MeshRun> runs;
    size_t staged = 0;
    WaitOnError wait{c->stream};
    // the world-space triangles stay resident for refits
    DevBuf& pos = c->d_tpos;
    DevBuf& nrm = c->d_tnrm;
    DevBuf& uv = c->d_tuv;
    DevBuf& mat = c->d_tmat;
    HIPCHK(pos.ensure((size_t)n * 36));
    HIPCHK(mat.ensure((size_t)n * 4));
    HIPCHK(hipMemcpyAsync(mat.p, c->h_mat.data(), (size_t)n * 4, hipMemcpyHostToDevice, c->stream));
    if (c->any_nrm) {
        HIPCHK(nrm.ensure((size_t)n * 36));
    }
    if (c->any_uv) {
        HIPCHK(uv.ensure((size_t)n * 24));
    }
    for (size_t i = 0; i < c->meshes.size();) {
        if (c->meshes[i].nt >= kHostMeshTriangles) {
            if (int r = place_mesh(c, c->meshes[i++], staged)) return r;
            continue;
        }
        const size_t begin = i;
        while (i < c->meshes.size() && c->meshes[i].nt < kHostMeshTriangles) ++i;
        expand_meshes(c, begin, i, runs.emplace_back());
        if (int r = place_run(c, runs.back())) return r;
    }
    const uint32_t ni = n > 1 ? n - 1 : 1;
    HIPCHK(c->d_nodes.ensure((size_t)ni * 64));
    HIPCHK(c->d_tris.ensure((size_t)n * 48));
    HIPCHK(c->d_attrs.ensure((size_t)n * 64));
    HIPCHK(c->d_prim.ensure((size_t)n * 4));
    HIPCHK(c->d_slot_of.ensure((size_t)n * 4));
    HIPCHK(c->d_lbvh_scratch.ensure(lbvh_scratch_bytes(n)));
    LbvhBuffers b{};
    b.tri_pos = pos.as<float>();
    b.tri_nrm = c->any_nrm ? nrm.as<float>() : nullptr;
    b.tri_uv = c->any_uv ? uv.as<float>() : nullptr;
    b.tri_mat = mat.as<uint32_t>();
    b.n = n;
    b.nodes = c->d_nodes.as<float4>();
    b.tris = c->d_tris.as<float4>();
    b.attrs = c->d_attrs.as<float4>();
    b.prim = c->d_prim.as<uint32_t>();
    b.slot_of = c->d_slot_of.as<uint32_t>();
    b.scratch = c->d_lbvh_scratch.p;
    HIPCHK(hipEventRecord(c->ev_start, c->stream));
    uint32_t depth = 0, n4 = 0;
    hipError_t e = lbvh_build(b, c->stream, &depth, &n4);
    if (e != hipSuccess) return fail_hip("lbvh_build", e);
    c->tree_depth = depth;
    c->n_nodes4 = 0;
    if (depth > kMaxTreeDepth)
        return fail(OHPT_ERR_UNSUPPORTED, "ohpt_scene_commit: LBVH depth " + std::to_string(depth) +
                                              " exceeds the traversal stack");
    HIPCHK(c->d_nodes4.ensure((size_t)n4 * 128));
    e = bvh4_collapse(b, c->d_nodes4.as<float4>(), c->stream);
    if (e != hipSuccess) return fail_hip("bvh4_collapse", e);
    HIPCHK(hipEventRecord(c->ev_stop, c->stream));
    HIPCHK(hipEventSynchronize(c->ev_stop));
    wait.armed = false;
    give_back(c, staged);
    c->stats.ms_build = elapsed(c->ev_start, c->ev_stop);
    c->n_nodes4 = n4;
    c->committed = true;
    c->in_scene = false;
    return build_emitters(c);
}

// The new transform is staged: the host triangles, the emitter table and the
// tree keep the committed geometry until ohpt_scene_refit applies it, so NEE
// never samples points the traversal cannot hit.
int ohpt_scene_set_mesh_transform(ohpt_context* c, uint32_t mesh, const float* world) {
    if (!c) return fail(OHPT_ERR_INVALID_ARG, "ohpt_scene_set_mesh_transform: null context");
    if (c->in_scene) return fail(OHPT_ERR_STATE, "ohpt_scene_set_mesh_transform: a scene is being staged");
    if (mesh >= c->meshes.size()) return fail(OHPT_ERR_INVALID_ARG, "ohpt_scene_set_mesh_transform: no such mesh");
    ohpt_context::MeshRec& m = c->meshes[mesh];
    m.next_has_world = world != nullptr;
    for (int k = 0; k < 16; ++k) m.next_world[k] = world ? (double)world[k] : (k % 5 == 0 ? 1.0 : 0.0);
    m.pending = true;
    c->refit_pending = true;
    return OHPT_OK;
}

int ohpt_scene_refit(ohpt_context* c) {
    if (!c) return fail(OHPT_ERR_INVALID_ARG, "ohpt_scene_refit: null context");
    if (c->in_scene) return fail(OHPT_ERR_STATE, "ohpt_scene_refit: a scene is being staged (commit it first)");
    if (!c->committed) return fail(OHPT_ERR_NO_SCENE, "ohpt_scene_refit: no committed scene");
    HIPCHK(enter(c));
    const uint32_t n = c->n_tris;
    if (n == 0) {
        for (auto& m : c->meshes) m.pending = false;
        c->refit_pending = false;
        return OHPT_OK;
    }
    // moved meshes: their world-space triangles recomputed on the device from
    // object-space copies uploaded at a mesh's first refit (nothing else moves)
    for (auto& m : c->meshes) {
        if (!m.pending) continue;
        m.has_world = m.next_has_world;
        std::memcpy(m.world, m.next_world, sizeof m.world);
        m.pending = false;
        if (m.nt == 0) continue;
        if (!m.d_vpos.p) {
            HIPCHK(m.d_vpos.ensure(m.pos.size() * 4));
            HIPCHK(m.d_idx.ensure(m.idx.size() * 4));
            HIPCHK(hipMemcpyAsync(m.d_vpos.p, m.pos.data(), m.pos.size() * 4, hipMemcpyHostToDevice, c->stream));
            HIPCHK(hipMemcpyAsync(m.d_idx.p, m.idx.data(), m.idx.size() * 4, hipMemcpyHostToDevice, c->stream));
            if (!m.nrm.empty()) {
                HIPCHK(m.d_vnrm.ensure(m.nrm.size() * 4));
                HIPCHK(hipMemcpyAsync(m.d_vnrm.p, m.nrm.data(), m.nrm.size() * 4, hipMemcpyHostToDevice, c->stream));
            }
        }
        launch_transform_mesh(m.d_vpos.as<float>(), m.nrm.empty() ? nullptr : m.d_vnrm.as<float>(),
                              m.d_idx.as<uint32_t>(), m.nt, mesh_transform(m), c->d_tpos.as<float>() + (size_t)m.base * 9,
                              c->any_nrm ? c->d_tnrm.as<float>() + (size_t)m.base * 9 : nullptr, c->stream);
        HIPCHK(hipGetLastError());
    }
    c->refit_pending = false;
    LbvhBuffers b{};
    b.tri_pos = c->d_tpos.as<float>();
    b.tri_nrm = c->any_nrm ? c->d_tnrm.as<float>() : nullptr;
    b.tri_uv = c->any_uv ? c->d_tuv.as<float>() : nullptr;
    b.tri_mat = c->d_tmat.as<uint32_t>();
    b.n = n;
    b.nodes = c->d_nodes.as<float4>();
    b.tris = c->d_tris.as<float4>();
    b.attrs = c->d_attrs.as<float4>();
    b.prim = c->d_prim.as<uint32_t>();
    b.slot_of = c->d_slot_of.as<uint32_t>();
    b.scratch = c->d_lbvh_scratch.p;
    HIPCHK(hipEventRecord(c->ev_start, c->stream));
    hipError_t e = lbvh_refit(b, c->stream);
    if (e != hipSuccess) return fail_hip("lbvh_refit", e);
    e = bvh4_collapse(b, c->d_nodes4.as<float4>(), c->stream);
    if (e != hipSuccess) return fail_hip("bvh4_collapse", e);
    HIPCHK(hipEventRecord(c->ev_stop, c->stream));
    HIPCHK(hipEventSynchronize(c->ev_stop));
    c->stats.ms_build = elapsed(c->ev_start, c->ev_stop);
    return build_emitters(c);
}

int ohpt_scene_triangle_count(ohpt_context* c, uint64_t* out) {
    if (!c || !out) return fail(OHPT_ERR_INVALID_ARG, "ohpt_scene_triangle_count: null argument");
    *out = c->committed ? c->n_tris : 0;
    return OHPT_OK;
}

int ohpt_scene_export_bvh(ohpt_context* c, void* nodes_out, void* tris_out, uint32_t* leaf_prims_out) {
    if (!c) return fail(OHPT_ERR_INVALID_ARG, "ohpt_scene_export_bvh: null context");
    if (int r = need_tree(c, "ohpt_scene_export_bvh")) return r;
    HIPCHK(enter(c));
    const uint32_t n = c->n_tris;
    if (n == 0) return OHPT_OK;
    const uint32_t ni = n > 1 ? n - 1 : 1;
    if (nodes_out) HIPCHK(hipMemcpyAsync(nodes_out, c->d_nodes.p, (size_t)ni * 64, hipMemcpyDeviceToHost, c->stream));
    if (tris_out) HIPCHK(hipMemcpyAsync(tris_out, c->d_tris.p, (size_t)n * 48, hipMemcpyDeviceToHost, c->stream));
    if (leaf_prims_out) HIPCHK(hipMemcpyAsync(leaf_prims_out, c->d_prim.p, (size_t)n * 4, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    return OHPT_OK;
}

int ohpt_scene_export_bvh4(ohpt_context* c, void* nodes4_out, uint32_t capacity, uint32_t* count_out) {
    if (!c) return fail(OHPT_ERR_INVALID_ARG, "ohpt_scene_export_bvh4: null context");
    if (int r = need_tree(c, "ohpt_scene_export_bvh4")) return r;
    if (!count_out) return fail(OHPT_ERR_INVALID_ARG, "ohpt_scene_export_bvh4: null count");
    HIPCHK(enter(c));
    *count_out = c->n_nodes4;
    if (!nodes4_out || c->n_nodes4 == 0) return OHPT_OK;
    if (capacity < c->n_nodes4) return fail(OHPT_ERR_INVALID_ARG, "ohpt_scene_export_bvh4: buffer holds fewer nodes");
    HIPCHK(hipMemcpyAsync(nodes4_out, c->d_nodes4.p, (size_t)c->n_nodes4 * 128, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    return OHPT_OK;
}

// ---------------------------------------------------------------- materials, textures, lights
int ohpt_upload_materials(ohpt_context* c, const ohpt_material* m, uint32_t count) {
    if (!c || (count && !m)) return fail(OHPT_ERR_INVALID_ARG, "ohpt_upload_materials: bad arguments");
    for (uint32_t i = 0; i < count; ++i) {
        for (int32_t t : {m[i].albedo_tex, m[i].roughness_tex, m[i].metallic_tex, m[i].normal_tex, m[i].orm_tex,
                          m[i].emissive_tex})
            if (t >= (int32_t)c->textures.size() || t < -1)
                return fail(OHPT_ERR_INVALID_ARG, "ohpt_upload_materials: texture id out of range");
    }
    HIPCHK(enter(c));
    c->h_materials.assign(m, m + count);
    int r = upload_materials_dev(c);
    if (r != OHPT_OK) return r;
    return build_emitters(c);
}

extern "C++" {
namespace {
// Small textures are packed on the host and copied once: the two kernels and the means' way
// back take longer than the loop. Update in us, on the device / here: from the host 1 texel
// 32 / 16, 8192 of three channels 38 / 20, of four 39 / 34; from the device 1 texel 40 / 27,
// 4096 of three channels 39 / 25, of four 39 / 34.
constexpr size_t kHostTexels = 8192, kHostTexelsOnDevice = 4096, kHostGradientTexels = 10240;
int fill_small_texture(ohpt_context* c, TexStore& t, const float* texels, int on_device) {
    const size_t n = (size_t)t.w * t.h, stride = t.c >= 2 ? 4 : 1;
    std::vector<float> source, packed(n * stride, 0.0f);
    if (on_device) {
        source.resize(n * t.c);
        HIPCHK(hipMemcpy(source.data(), texels, n * t.c * 4, hipMemcpyDeviceToHost));
        texels = source.data();
    }
    double sum[3] = {0.0, 0.0, 0.0};
    for (size_t i = 0; i < n; ++i)
        for (uint32_t k = 0; k < t.c; ++k) {
            packed[i * stride + k] = texels[i * t.c + k];
            if (k < 3) sum[k] += texels[i * t.c + k];
        }
    if (t.c == 3)
        for (size_t i = 0; i < n; ++i) packed[i * 4 + 3] = 1.0f;
    HIPCHK(t.data.ensure(packed.size() * 4));
    WaitOnError wait{c->stream};
    HIPCHK(hipMemcpyAsync(t.data.p, packed.data(), packed.size() * 4, hipMemcpyHostToDevice, c->stream));
    wait.armed = false;
    HIPCHK(hipStreamSynchronize(c->stream));
    for (int k = 0; k < 3; ++k) t.mean[k] = sum[t.c == 1 ? 0 : k] / (double)n;
    return OHPT_OK;
}

// The packed texels and channel means of t from w*h*c floats. The source is first
// copied whole, in device memory too: the copy is what checks its range, reaches
// peers' memory and waits for the default stream's earlier work on it, while the
// kernels stay ordered behind the context's own renders.
int fill_texture(ohpt_context* c, TexStore& t, const float* texels, int on_device) {
    if ((size_t)t.w * t.h <= (on_device ? kHostTexelsOnDevice : kHostTexels)) return fill_small_texture(c, t, texels, on_device);
    const size_t n = (size_t)t.w * t.h, bytes = n * t.c * 4;
    const size_t mean_at = (bytes + 15) & ~size_t(15), staged = mean_at + texel_mean_scratch_bytes();
    HIPCHK(t.data.ensure(t.packed_floats() * 4));
    HIPCHK(c->tmp.ensure(staged));
    WaitOnError wait{c->stream};
    if (on_device) {
        HIPCHK(hipMemcpy(c->tmp.p, texels, bytes, hipMemcpyDefault));
        HIPCHK(hipStreamSynchronize(nullptr));
    } else {
        HIPCHK(hipMemcpyAsync(c->tmp.p, texels, bytes, hipMemcpyHostToDevice, c->stream));
    }
    char* mean = reinterpret_cast<char*>(c->tmp.p) + mean_at;
    launch_texel_pack(c->tmp.as<float>(), n, t.c, t.data.as<float>(), mean, c->stream);
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(t.mean, mean, sizeof t.mean, hipMemcpyDeviceToHost, c->stream));
    wait.armed = false;
    HIPCHK(hipStreamSynchronize(c->stream));
    give_back(c, staged);
    return OHPT_OK;
}
}  // namespace
}  // extern "C++"

int ohpt_upload_texture(ohpt_context* c, int32_t* out_id, const float* texels, uint32_t w, uint32_t h,
                        uint32_t channels) {
    if (!c || !out_id || !texels || w == 0 || h == 0 || channels == 0 || channels > 4)
        return fail(OHPT_ERR_INVALID_ARG, "ohpt_upload_texture: bad arguments");
    HIPCHK(enter(c));
    TexStore t;
    t.w = w; t.h = h; t.c = channels;
    if (int r = fill_texture(c, t, texels, 0)) return r;
    c->textures.push_back(std::move(t));
    *out_id = (int32_t)c->textures.size() - 1;
    return upload_texdesc(c);
}

// texels: same layout as the upload (w*h*channels floats); on_device = device pointer of that layout
int ohpt_update_texture(ohpt_context* c, int32_t id, const float* texels, int on_device) {
    if (!c || !texels || id < 0 || id >= (int32_t)c->textures.size())
        return fail(OHPT_ERR_INVALID_ARG, "ohpt_update_texture: bad arguments");
    HIPCHK(enter(c));
    TexStore& t = c->textures[(size_t)id];
    if (int r = fill_texture(c, t, texels, on_device)) return r;
    // an emissive texture's mean weighs its material's triangles in the emitter table
    for (const ohpt_material& m : c->h_materials)
        if (m.emissive_tex == id) {
            int r = upload_materials_dev(c);
            return r == OHPT_OK ? build_emitters(c) : r;
        }
    return OHPT_OK;
}

int ohpt_texture_info(ohpt_context* c, int32_t id, uint32_t* w, uint32_t* h, uint32_t* ch) {
    if (!c || id < 0 || id >= (int32_t)c->textures.size())
        return fail(OHPT_ERR_INVALID_ARG, "ohpt_texture_info: bad texture id");
    const TexStore& t = c->textures[(size_t)id];
    if (w) *w = t.w;
    if (h) *h = t.h;
    if (ch) *ch = t.c;
    return OHPT_OK;
}

int ohpt_clear_textures(ohpt_context* c) {
    if (!c) return fail(OHPT_ERR_INVALID_ARG, "ohpt_clear_textures: null context");
    HIPCHK(enter(c));
    HIPCHK(hipStreamSynchronize(c->stream));
    for (int l = 0; l < ohpt_context::kLanes; ++l) HIPCHK(hipStreamSynchronize(c->lane_stream[l]));
    // materials keep their constants; their bindings to the released textures go
    for (ohpt_material& m : c->h_materials) {
        m.albedo_tex = m.roughness_tex = m.metallic_tex = -1;
        m.normal_tex = m.orm_tex = m.emissive_tex = -1;
    }
    c->textures.clear();
    c->grad_off.clear();
    c->grad_total = 0;
    int r = upload_materials_dev(c);
    if (r == OHPT_OK) r = upload_texdesc(c);
    if (r == OHPT_OK) r = build_emitters(c);
    return r;
}

int ohpt_upload_lights(ohpt_context* c, const ohpt_light* lights, uint32_t count) {
    if (!c || (count && !lights)) return fail(OHPT_ERR_INVALID_ARG, "ohpt_upload_lights: bad arguments");
    HIPCHK(enter(c));
    c->h_lights.assign(lights, lights + count);
    if (count) {
        HIPCHK(c->d_lights.ensure((size_t)count * sizeof(ohpt_light)));
        HIPCHK(hipMemcpyAsync(c->d_lights.p, lights, (size_t)count * sizeof(ohpt_light), hipMemcpyHostToDevice,
                              c->stream));
        HIPCHK(hipStreamSynchronize(c->stream));
    }
    return OHPT_OK;
}

int ohpt_upload_env(ohpt_context* c, const float* rgba, uint32_t w, uint32_t h) {
    if (!c) return fail(OHPT_ERR_INVALID_ARG, "ohpt_upload_env: null context");
    HIPCHK(enter(c));
    if (!rgba || w == 0 || h == 0) {
        c->env_w = c->env_h = 0;
        return OHPT_OK;
    }
    const size_t n = (size_t)w * h;
    HIPCHK(c->d_env.ensure(n * 16));
    HIPCHK(c->d_cond.ensure(n * 4));
    HIPCHK(c->d_marg.ensure((size_t)h * 4));
    HIPCHK(c->d_rowsum.ensure((size_t)h * 4));
    HIPCHK(c->d_integral.ensure(4));
    HIPCHK(c->d_marg_guide.ensure(((size_t(1) << env_guide_log2(h)) + 1) * 4));
    HIPCHK(c->d_cond_guide.ensure(((size_t(1) << env_guide_log2(w)) + 1) * h * 4));
    HIPCHK(hipMemcpyAsync(c->d_env.p, rgba, n * 16, hipMemcpyHostToDevice, c->stream));
    hipError_t e = env_cdf_build(c->d_env.as<float4>(), w, h, c->d_marg.as<float>(), c->d_cond.as<float>(),
                                 c->d_rowsum.as<float>(), c->d_integral.as<float>(), c->d_marg_guide.as<uint32_t>(),
                                 c->d_cond_guide.as<uint32_t>(), c->stream);
    if (e != hipSuccess) return fail_hip("env_cdf_build", e);
    HIPCHK(hipStreamSynchronize(c->stream));
    c->env_w = w;
    c->env_h = h;
    return OHPT_OK;
}

int ohpt_set_env_intensity(ohpt_context* c, float scale) {
    if (!c || !(scale >= 0.0f)) return fail(OHPT_ERR_INVALID_ARG, "ohpt_set_env_intensity: bad arguments");
    c->env_intensity = scale;
    return OHPT_OK;
}

int ohpt_export_env_cdf(ohpt_context* c, float* marginal, float* conditional, float* integral) {
    if (!c || c->env_w == 0) return fail(OHPT_ERR_STATE, "ohpt_export_env_cdf: no environment");
    HIPCHK(enter(c));
    if (marginal) HIPCHK(hipMemcpyAsync(marginal, c->d_marg.p, (size_t)c->env_h * 4, hipMemcpyDeviceToHost, c->stream));
    if (conditional)
        HIPCHK(hipMemcpyAsync(conditional, c->d_cond.p, (size_t)c->env_w * c->env_h * 4, hipMemcpyDeviceToHost,
                              c->stream));
    if (integral) HIPCHK(hipMemcpyAsync(integral, c->d_integral.p, 4, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    return OHPT_OK;
}

int ohpt_env_sample(ohpt_context* c, const float* u, float* out, uint32_t n) {
    if (!c || (n && (!u || !out))) return fail(OHPT_ERR_INVALID_ARG, "ohpt_env_sample: null argument");
    if (c->env_w == 0) return fail(OHPT_ERR_STATE, "ohpt_env_sample: no environment");
    if (n == 0) return OHPT_OK;
    HIPCHK(enter(c));
    DevBuf du, dout;
    HIPCHK(du.ensure((size_t)n * 8));
    HIPCHK(dout.ensure((size_t)n * 16));
    HIPCHK(hipMemcpyAsync(du.p, u, (size_t)n * 8, hipMemcpyHostToDevice, c->stream));
    launch_env_sample(scene_view(c), du.as<float>(), dout.as<float4>(), n, c->stream);
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(out, dout.p, (size_t)n * 16, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    return OHPT_OK;
}

// ---------------------------------------------------------------- per-frame state
int ohpt_set_camera(ohpt_context* c, const ohpt_camera* cam) {
    if (!c || !cam || !(cam->tan_half_fov_y > 0.0f)) return fail(OHPT_ERR_INVALID_ARG, "ohpt_set_camera: bad camera");
    c->cam = *cam;
    return OHPT_OK;
}

int ohpt_set_settings(ohpt_context* c, const ohpt_settings* s) {
    if (!c || !s) return fail(OHPT_ERR_INVALID_ARG, "ohpt_set_settings: null argument");
    if (s->max_bounces > 60) return fail(OHPT_ERR_INVALID_ARG, "ohpt_set_settings: max_bounces > 60");
    if (s->sampler > OHPT_SAMPLER_SOBOL_OWEN) return fail(OHPT_ERR_INVALID_ARG, "ohpt_set_settings: unknown sampler");
    if (s->integrator > OHPT_INTEGRATOR_REFERENCE_GOLDEN)
        return fail(OHPT_ERR_INVALID_ARG, "ohpt_set_settings: unknown integrator");
    c->st = *s;
    return OHPT_OK;
}

int ohpt_get_settings(ohpt_context* c, ohpt_settings* s) {
    if (!c || !s) return fail(OHPT_ERR_INVALID_ARG, "ohpt_get_settings: null argument");
    *s = c->st;
    return OHPT_OK;
}

int ohpt_reset_accumulation(ohpt_context* c) {
    if (!c) return fail(OHPT_ERR_INVALID_ARG, "ohpt_reset_accumulation: null context");
    HIPCHK(enter(c));
    c->sample_index = c->seed;
    return clear_frame(c);
}

int ohpt_set_render_seed(ohpt_context* c, uint32_t seed) {
    if (!c) return fail(OHPT_ERR_INVALID_ARG, "ohpt_set_render_seed: null context");
    c->seed = seed;
    return OHPT_OK;
}

// ---------------------------------------------------------------- rendering
namespace {

// The reference's own estimator (compat.hip) in wavefront form: the frame's
// paths split into lanes as ohpt_render's, each lane stepping through
// 2 + 2 * max_bounces traversal + shading steps, then one accumulation.
int render_reference(ohpt_context* c, uint32_t spp, uint32_t render_flags) {
    if (c->st.max_bounces > kRefMaxBounces)
        return fail(OHPT_ERR_UNSUPPORTED, "ohpt_render: the reference estimator supports max_bounces <= 30");
    const uint64_t npix = (uint64_t)c->W * c->H;
    // batches of up to 2^25 paths (16 samples per pixel at 1920x1080, about 11 GB of
    // path state): one batch of the Cornell scene's 16 samples measured 71 ms against
    // 78 ms in batches of 2^22 paths
    const uint64_t target = std::max<uint64_t>(npix, 1ull << 25);
    const uint32_t per_batch = (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(spp, target / npix));
    int r = ensure_paths(c, (uint32_t)(npix * per_batch));
    if (r != OHPT_OK) return r;
    const DevScene S = scene_view(c);
    const uint32_t nsteps = ref_steps(c->st.max_bounces);
    HIPCHK(hipEventRecord(c->ev_start, c->stream));
    uint32_t remaining = spp;
    while (remaining > 0) {
        const uint32_t batch = std::min(remaining, per_batch);
        RefFrame f{};
        f.cam = c->cam;
        f.width = c->W;
        f.height = c->H;
        f.n_paths = (uint32_t)(npix * batch);
        f.sample_base = c->sample_index;
        f.max_bounces = c->st.max_bounces;
        f.sampler = c->st.sampler;
        f.flags = c->st.flags;
        f.revision = c->st.integrator == OHPT_INTEGRATOR_REFERENCE_GOLDEN ? 1u : 0u;
        f.firefly_clamp = c->st.firefly_clamp;
        const int nl = f.n_paths >= (1u << 18) ? ohpt_context::kLanes : 1;
        const uint32_t part = ((f.n_paths + nl - 1) / nl + 63u) & ~63u;
        f.row_groups = (uint32_t)nl;
        const int set = c->render_set;
        const PathState ps = path_state(c, set);
        bool fork = false;
        if (nl > 1 && c->stream_dirty) {
            HIPCHK(hipEventRecord(c->ev_fork, c->stream));
            fork = true;
            c->stream_dirty = false;
        }
        if (nl == 1) c->stream_dirty = true;
        struct Lane {
            hipStream_t s;
            RefFrame fl;
            PathState pl;
            uint32_t* ovf;
        };
        Lane ln[ohpt_context::kLanes];
        const uint32_t tblocks = lane_trace_blocks(nl);
        for (int l = 0; l < nl; ++l) {
            Lane& x = ln[l];
            x.s = nl == 1 ? c->stream : c->lane_stream[l];
            if (fork) HIPCHK(hipStreamWaitEvent(x.s, c->ev_fork, 0));
            else if (nl > 1 && c->acc_pending[set]) HIPCHK(hipStreamWaitEvent(x.s, c->ev_acc[set], 0));
            x.fl = f;
            x.fl.pid_base = std::min<uint32_t>(f.n_paths, (uint32_t)l * part);
            x.fl.n_paths = std::min<uint32_t>(f.n_paths - x.fl.pid_base, part);
            x.pl = lane_view(ps, x.fl.pid_base, l);
            x.ovf = lane_ovf(c, l);
            launch_clear_counters(x.pl, nsteps, x.s);
            launch_ref_generate(x.fl, x.pl, x.s);
        }
        // step s: the closest-hit rays queued by step s - 1 (the camera rays at s = 0)
        // with that step's shadow rays, then shading
        for (uint32_t st = 0; st < nsteps; ++st) {
            for (int l = 0; l < nl; ++l) {
                const Lane& x = ln[l];
                launch_ref_trace(S, x.pl.q[st & 1u], x.pl.counters + ext_counter(st), x.fl.n_paths, x.pl.o, x.pl.d, x.pl.hits,
                                 x.pl.counters + sh_counter(st), st ? 2u * x.fl.n_paths : 0u,
                                 x.pl.sh_o, x.pl.sh_d, x.pl.ln0, x.pl.ln1, fetch_counters(x.pl, st), x.ovf,
                                 x.s, tblocks);
            }
            for (int l = 0; l < nl; ++l) launch_ref_shade(S, ln[l].fl, ln[l].pl, st, ln[l].s);
        }
        if (nl > 1) {
            for (int l = 0; l < nl; ++l) {
                HIPCHK(hipEventRecord(c->ev_lane[l], ln[l].s));
                HIPCHK(hipStreamWaitEvent(c->stream, c->ev_lane[l], 0));
            }
        }
        launch_ref_accumulate(f, ps, c->d_accum.as<float4>(), c->d_moments.as<float4>(), c->stream);
        HIPCHK(hipEventRecord(c->ev_acc[set], c->stream));
        c->acc_pending[set] = true;
        c->render_set = set ^ 1;
        HIPCHK(hipGetLastError());
        c->sample_index += batch;
        remaining -= batch;
    }
    c->reference_samples = true;
    HIPCHK(hipEventRecord(c->ev_stop, c->stream));
    if (!(render_flags & OHPT_RENDER_ASYNC)) {
        HIPCHK(hipEventSynchronize(c->ev_stop));
        c->stats = ohpt_stats{};
        c->stats.ms_total = elapsed(c->ev_start, c->ev_stop);
        c->stats.paths = npix * spp;
    }
    return OHPT_OK;
}


}  // namespace

int ohpt_render(ohpt_context* c, uint32_t spp, uint32_t render_flags) {
    if (!c) return fail(OHPT_ERR_INVALID_ARG, "ohpt_render: null context");
    if (int r0 = need_tree(c, "ohpt_render")) return r0;
    if (spp == 0) return OHPT_OK;
    HIPCHK(hipSetDevice(c->device));
    const uint64_t npix = (uint64_t)c->W * c->H;
    const uint64_t target = std::max<uint64_t>(npix, 1ull << 22);
    const uint32_t per_batch = (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(spp, target / npix));
    if (npix * per_batch > 0x7FFFFFFFull) return fail(OHPT_ERR_INVALID_ARG, "ohpt_render: image too large");
    if (c->st.integrator != OHPT_INTEGRATOR_PHYSICAL) return render_reference(c, spp, render_flags);
    int r = ensure_paths(c, (uint32_t)(npix * per_batch));
    if (r != OHPT_OK) return r;
    const DevScene S = scene_view(c);
    const bool profile = (render_flags & 2u) != 0;
    std::vector<hipEvent_t> evs;
    auto mark = [&](hipEvent_t* out) -> int {
        if (!profile) return OHPT_OK;
        const size_t k = evs.size();
        if (k >= c->ev_pool.size()) {
            hipEvent_t e;
            HIPCHK(hipEventCreate(&e));
            c->ev_pool.push_back(e);
        }
        *out = c->ev_pool[k];
        evs.push_back(*out);
        HIPCHK(hipEventRecord(*out, c->stream));
        return OHPT_OK;
    };
    struct Seg { hipEvent_t a, b; int kind; };
    std::vector<Seg> segs;
    unsigned long long* tstats = nullptr;
    if (profile) {
        HIPCHK(c->tstats.ensure(16));
        tstats = c->tstats.as<unsigned long long>();
        launch_fill_u32(c->tstats.as<uint32_t>(), 0u, 4, c->stream);
    }
    uint32_t n_extend = 0;
    HIPCHK(hipEventRecord(c->ev_start, c->stream));
    uint64_t rays_ext = 0, rays_sh = 0;
    std::vector<uint32_t> host_counters(kCounterWords);
    uint32_t remaining = spp;
    while (remaining > 0) {
        const uint32_t batch = std::min(remaining, per_batch);
        FrameParams f{};
        f.cam = c->cam;
        f.width = c->W;
        f.height = c->H;
        f.n_paths = (uint32_t)(npix * batch);
        f.sample_base = c->sample_index;
        f.max_bounces = c->st.max_bounces;
        f.rr_start = c->st.rr_start;
        f.sampler = c->st.sampler;
        f.flags = c->st.flags;
        f.firefly_clamp = c->st.firefly_clamp;
        f.ray_eps = c->st.ray_eps;
        // Lanes: kLanes independent wavefronts on their own streams once the
        // batch is large enough; one lane on the context stream when profiling,
        // so the per-kernel events time each kernel alone.
        const int nl = (!profile && f.n_paths >= (1u << 18)) ? ohpt_context::kLanes : 1;
        const uint32_t part = ((f.n_paths + nl - 1) / nl + 63u) & ~63u;
        f.row_groups = (uint32_t)nl;
        const int set = c->render_set;
        const PathState ps = path_state(c, set);
        // Lanes wait for the context stream only when it took other work since they
        // last forked from it; otherwise just for the accumulation that last read this
        // batch's copy of the radiance arrays. A batch on the context stream itself is
        // ordered after everything and marks the stream for the next lanes.
        bool fork = false;
        if (nl > 1 && c->stream_dirty) {
            HIPCHK(hipEventRecord(c->ev_fork, c->stream));
            fork = true;
            c->stream_dirty = false;
        }
        if (nl == 1) c->stream_dirty = true;
        struct Lane {
            hipStream_t s;
            FrameParams fl;
            PathState pl;
            uint32_t* ovf;
        };
        Lane ln[ohpt_context::kLanes];
        const uint32_t tblocks = lane_trace_blocks(nl);
        for (int l = 0; l < nl; ++l) {
            Lane& x = ln[l];
            x.s = nl == 1 ? c->stream : c->lane_stream[l];
            if (fork) HIPCHK(hipStreamWaitEvent(x.s, c->ev_fork, 0));
            else if (nl > 1 && c->acc_pending[set]) HIPCHK(hipStreamWaitEvent(x.s, c->ev_acc[set], 0));
            x.fl = f;
            x.fl.pid_base = std::min<uint32_t>(f.n_paths, (uint32_t)l * part);
            x.fl.n_paths = std::min<uint32_t>(f.n_paths - x.fl.pid_base, part);
            x.pl = lane_view(ps, x.fl.pid_base, l);
            x.ovf = lane_ovf(c, l);
            launch_clear_counters(x.pl, f.max_bounces + 1, x.s);
            launch_generate(x.fl, x.pl, x.s);
        }
        // The lanes' kernels are submitted step by step (every lane's extend, then every
        // lane's shade of bounce 0, ...), so the second lane starts while the host is still
        // submitting the first lane's later steps. Extension rays of bounce b+1 and shadow
        // rays of bounce b share one traversal launch: both come from shade(b) and are independent.
        for (int l = 0; l < nl; ++l) {
            const Lane& x = ln[l];
            Seg sg{};
            if ((r = mark(&sg.a))) return r;
            launch_extend(S, x.pl.q[0], x.pl.counters, x.fl.n_paths, x.pl.o, x.pl.d, x.pl.hits,
                          fetch_counters(x.pl, 0), x.ovf, tstats, x.s, tblocks);
            ++n_extend;
            if ((r = mark(&sg.b))) return r;
            if (profile) { sg.kind = 0; segs.push_back(sg); }
        }
        for (uint32_t b = 0; b <= f.max_bounces; ++b) {
            for (int l = 0; l < nl; ++l) {
                const Lane& x = ln[l];
                Seg sg{};
                if ((r = mark(&sg.a))) return r;
                launch_shade(S, x.fl, x.pl, b, x.s);
                if ((r = mark(&sg.b))) return r;
                if (profile) { sg.kind = 1; segs.push_back(sg); }
            }
            if (b == f.max_bounces) break;
            for (int l = 0; l < nl; ++l) {
                const Lane& x = ln[l];
                Seg sg{};
                if ((r = mark(&sg.a))) return r;
                launch_extend_connect(S, x.pl.q[(b + 1) & 1u], x.pl.counters + ext_counter(b + 1), x.fl.n_paths, x.pl.o, x.pl.d,
                                      x.pl.hits, x.pl.counters + sh_counter(b + 1), 2u * x.fl.n_paths,
                                      x.pl.sh_o, x.pl.sh_d, x.pl.sh_c, x.pl.ln0, x.pl.ln1,
                                      fetch_counters(x.pl, b + 1), x.ovf, nullptr, b, tstats, x.s,
                                      tblocks);
                ++n_extend;
                if ((r = mark(&sg.b))) return r;
                if (profile) { sg.kind = 0; segs.push_back(sg); }
            }
        }
        if (nl > 1) {
            for (int l = 0; l < nl; ++l) {
                HIPCHK(hipEventRecord(c->ev_lane[l], ln[l].s));
                HIPCHK(hipStreamWaitEvent(c->stream, c->ev_lane[l], 0));
            }
        }
        launch_accumulate(f, ps, c->d_accum.as<float4>(), c->d_moments.as<float4>(), c->d_aov_albedo.as<float4>(),
                          c->d_aov_normal.as<float4>(), c->d_disp.as<float4>(), c->stream);
        HIPCHK(hipEventRecord(c->ev_acc[set], c->stream));
        c->acc_pending[set] = true;
        c->render_set = set ^ 1;
        HIPCHK(hipGetLastError());
        if (!(render_flags & OHPT_RENDER_ASYNC)) {
            host_counters.resize((size_t)kCounterWords * nl);
            HIPCHK(hipMemcpyAsync(host_counters.data(), ps.counters, (size_t)kCounterWords * 4 * nl,
                                  hipMemcpyDeviceToHost, c->stream));
            HIPCHK(hipStreamSynchronize(c->stream));
            for (int l = 0; l < nl; ++l) {
                const uint32_t* hc = host_counters.data() + (size_t)l * kCounterWords;
                for (uint32_t b = 0; b <= f.max_bounces; ++b) rays_ext += hc[ext_counter(b)];
                for (uint32_t b = 0; b < f.max_bounces; ++b) rays_sh += hc[sh_counter(b + 1)];
            }
        }
        c->sample_index += batch;
        remaining -= batch;
    }
    HIPCHK(hipEventRecord(c->ev_stop, c->stream));
    if (!(render_flags & OHPT_RENDER_ASYNC)) {
        HIPCHK(hipEventSynchronize(c->ev_stop));
        c->stats.ms_total = elapsed(c->ev_start, c->ev_stop);
        c->stats.ms_extend = c->stats.ms_shade = c->stats.ms_connect = 0.0;
        for (const Seg& sg : segs) {
            const double ms = elapsed(sg.a, sg.b);
            if (sg.kind == 0) c->stats.ms_extend += ms;
            else if (sg.kind == 1) c->stats.ms_shade += ms;
            else c->stats.ms_connect += ms;
        }
        c->stats.rays_extend = rays_ext;
        c->stats.rays_shadow = rays_sh;
        c->stats.paths = npix * spp;
        c->stats.extend_launches = n_extend;
        c->stats.node_visits = c->stats.tri_tests = 0;
        if (profile) {
            unsigned long long h[2] = {0, 0};
            HIPCHK(hipMemcpy(h, tstats, 16, hipMemcpyDeviceToHost));
            c->stats.node_visits = h[0];
            c->stats.tri_tests = h[1];
        }
    }
    return OHPT_OK;
}

// ---------------------------------------------------------------- adjoint
int ohpt_zero_gradients(ohpt_context* c) {
    if (!c) return fail(OHPT_ERR_INVALID_ARG, "ohpt_zero_gradients: null context");
    HIPCHK(enter(c));
    std::vector<size_t> off;
    size_t total = 0;
    for (const TexStore& t : c->textures) {
        off.push_back(total);
        total += (t.packed_floats() + 63) & ~size_t(63);
    }
    if (total >= 0xFFFFFFFFull) return fail(OHPT_ERR_UNSUPPORTED, "ohpt_zero_gradients: textures too large");
    const bool changed = off != c->grad_off || !c->grad_arena.p;
    if (changed) {
        HIPCHK(c->grad_arena.ensure(std::max<size_t>(total, 64) * 4));
        c->grad_off = off;
    }
    c->grad_total = total;
    launch_fill_u32(c->grad_arena.as<uint32_t>(), 0u, (uint32_t)std::max<size_t>(total, 64), c->stream);
    HIPCHK(hipGetLastError());
    if (changed) return upload_texdesc(c);
    HIPCHK(hipStreamSynchronize(c->stream));
    return OHPT_OK;
}

int ohpt_read_texture_gradient(ohpt_context* c, int32_t id, float* out, int on_device) {
    if (!c || !out || id < 0 || id >= (int32_t)c->textures.size())
        return fail(OHPT_ERR_INVALID_ARG, "ohpt_read_texture_gradient: bad arguments");
    TexStore& t = c->textures[(size_t)id];
    if (!c->grad_arena.p || (size_t)id >= c->grad_off.size())
        return fail(OHPT_ERR_STATE, "ohpt_read_texture_gradient: no adjoint has run");
    HIPCHK(enter(c));
    const size_t n = (size_t)t.w * t.h, bytes = n * t.c * 4;
    const float* src = c->grad_arena.as<float>() + c->grad_off[(size_t)id];
    const bool padded = t.c == 2 || t.c == 3;
    if (padded && !on_device && n <= kHostGradientTexels) {
        // fewer texels than a launch is worth: 64x64 of three channels 26 us unpacked on the
        // device, 17 here, 129x64 28 and 25; 128x128 32 and 40
        std::vector<float> packed(n * 4);
        HIPCHK(hipMemcpyAsync(packed.data(), src, n * 16, hipMemcpyDeviceToHost, c->stream));
        HIPCHK(hipStreamSynchronize(c->stream));
        for (size_t i = 0; i < n; ++i)
            for (uint32_t k = 0; k < t.c; ++k) out[i * t.c + k] = packed[i * 4 + k];
        return OHPT_OK;
    }
    if (padded) {
        HIPCHK(c->tmp.ensure(bytes));
        launch_texel_unpack(src, n, t.c, c->tmp.as<float>(), c->stream);
        HIPCHK(hipGetLastError());
        src = c->tmp.as<float>();
    }
    if (!on_device) HIPCHK(hipMemcpyAsync(out, src, bytes, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    if (on_device) {
        // on the default stream, behind the caller's earlier work on `out` there
        HIPCHK(hipMemcpy(out, src, bytes, hipMemcpyDefault));
        HIPCHK(hipStreamSynchronize(nullptr));
    }
    if (src == c->tmp.as<float>()) give_back(c, bytes);
    return OHPT_OK;
}

// Path-replay adjoint (Vicini, Speierer, Jakob 2021) of the image made of the
// first `spp` samples after a reset (sample indices seed .. seed+spp-1):
// pass 1 renders each batch forward and records shadow visibility and the
// closest hit of every vertex per path (16 B per vertex in HBM; not with
// OHPT_ADJOINT_RETRACE); pass 2 regenerates the same paths with the same
// random numbers, reads the logged hits (or re-traces every replayed ray),
// and scatters dL/d(texel) into the texture gradient buffers (accumulating:
// call ohpt_zero_gradients first).
int ohpt_adjoint(ohpt_context* c, const float* dl_dimage, int on_device, uint32_t spp, uint32_t flags) {
    if (!c || !dl_dimage) return fail(OHPT_ERR_INVALID_ARG, "ohpt_adjoint: null argument");
    if (int r0 = need_tree(c, "ohpt_adjoint")) return r0;
    if (spp == 0) return OHPT_OK;
    if (c->st.max_bounces > 15) return fail(OHPT_ERR_UNSUPPORTED, "ohpt_adjoint: max_bounces > 15");
    if (c->st.integrator != OHPT_INTEGRATOR_PHYSICAL)
        return fail(OHPT_ERR_UNSUPPORTED, "ohpt_adjoint: only the physically based integrator has an adjoint");
    if (flags & ~(uint32_t)(OHPT_ADJOINT_DETERMINISTIC | OHPT_ADJOINT_RETRACE))
        return fail(OHPT_ERR_INVALID_ARG, "ohpt_adjoint: unknown flags");
    HIPCHK(enter(c));
    if (!c->grad_arena.p || c->grad_off.size() != c->textures.size()) {
        int r = ohpt_zero_gradients(c);
        if (r != OHPT_OK) return r;
    }
    const bool deterministic = (flags & OHPT_ADJOINT_DETERMINISTIC) != 0;
    const bool retrace = (flags & OHPT_ADJOINT_RETRACE) != 0;
    const uint64_t npix = (uint64_t)c->W * c->H;
    HIPCHK(c->adj_dldi.ensure(npix * 16));
    HIPCHK(hipMemcpyAsync(c->adj_dldi.p, dl_dimage, npix * 16,
                          on_device ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice, c->stream));
    uint64_t target = std::max<uint64_t>(npix, 1ull << 22);
    const uint64_t recs_per_path = (uint64_t)std::max(1u, c->st.max_bounces) * kGradRecordsPerVertex;
    if (deterministic) target = std::max<uint64_t>(npix, (1ull << 28) / recs_per_path);
    if (npix * recs_per_path > 0xFFFFFFFFull && deterministic)
        return fail(OHPT_ERR_UNSUPPORTED, "ohpt_adjoint: image too large for the deterministic mode");
    const uint32_t per_batch = (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(spp, target / npix));
    int r = ensure_paths(c, (uint32_t)(npix * per_batch));
    if (r != OHPT_OK) return r;
    HIPCHK(c->adj_vis.ensure((size_t)c->capacity * 4));
    HIPCHK(c->adj_lrem.ensure((size_t)c->capacity * 16));
    if (!retrace) HIPCHK(c->adj_hits.ensure((size_t)c->capacity * (c->st.max_bounces + 1) * 16));
    uint32_t* rec_key = nullptr;
    uint32_t* rec_val = nullptr;
    uint32_t* rec_count = nullptr;
    const uint64_t verts_per_path = std::max(1u, c->st.max_bounces);
    if (deterministic) {
        const size_t nrec = (size_t)npix * per_batch * recs_per_path;
        const size_t nvert = (size_t)npix * per_batch * verts_per_path;
        HIPCHK(c->rec_key.ensure(nrec * 4));
        HIPCHK(c->rec_val.ensure(nrec * 4));
        HIPCHK(c->rec_key2.ensure(nrec * 4));
        HIPCHK(c->rec_val2.ensure(nrec * 4));
        HIPCHK(c->rec_count.ensure(nvert * 4));
        HIPCHK(c->rec_tiles.ensure(((size_t)record_tiles((uint32_t)nvert) + 1) * 4));
        HIPCHK(c->rec_scratch.ensure(radix_sort_scratch_bytes((uint32_t)nrec)));
        rec_key = c->rec_key.as<uint32_t>();
        rec_val = c->rec_val.as<uint32_t>();
        rec_count = c->rec_count.as<uint32_t>();
        HIPCHK(c->rec_flag.ensure(4));
        launch_fill_u32(c->rec_flag.as<uint32_t>(), 0u, 1, c->stream);
    }
    uint32_t* rec_overflow = deterministic ? c->rec_flag.as<uint32_t>() : nullptr;
    const DevScene S = scene_view(c);
    PathState ps = path_state(c);
    ps.hit_log = retrace ? nullptr : c->adj_hits.as<float4>();
    uint32_t* vis = c->adj_vis.as<uint32_t>();
    float4* lrem = c->adj_lrem.as<float4>();
    const float inv_spp = 1.0f / (float)spp;
    HIPCHK(hipEventRecord(c->ev_start, c->stream));
    uint32_t remaining = spp, sample = c->seed;
    while (remaining > 0) {
        const uint32_t batch = std::min(remaining, per_batch);
        FrameParams f{};
        f.cam = c->cam;
        f.width = c->W;
        f.height = c->H;
        f.n_paths = (uint32_t)(npix * batch);
        f.sample_base = sample;
        f.max_bounces = c->st.max_bounces;
        f.rr_start = c->st.rr_start;
        f.sampler = c->st.sampler;
        f.flags = c->st.flags & ~(uint32_t)OHPT_FLAG_AOVS;
        f.firefly_clamp = c->st.firefly_clamp;
        f.ray_eps = c->st.ray_eps;
        const uint32_t nvert = (uint32_t)(f.n_paths * verts_per_path);
        if (deterministic) launch_fill_u32(rec_count, 0u, nvert, c->stream);
        // lanes as in ohpt_render: each runs both passes over its own path range,
        // submitted step by step across the lanes
        const int nl = f.n_paths >= (1u << 18) ? ohpt_context::kLanes : 1;
        const uint32_t part = ((f.n_paths + nl - 1) / nl + 63u) & ~63u;
        f.row_groups = (uint32_t)nl;
        if (nl > 1) HIPCHK(hipEventRecord(c->ev_fork, c->stream));
        struct Lane {
            hipStream_t s;
            FrameParams fl;
            PathState pl;
            uint32_t* ovf;
        };
        Lane ln[ohpt_context::kLanes];
        const uint32_t tblocks = lane_trace_blocks(nl);
        for (int l = 0; l < nl; ++l) {
            Lane& x = ln[l];
            x.s = nl == 1 ? c->stream : c->lane_stream[l];
            if (nl > 1) HIPCHK(hipStreamWaitEvent(x.s, c->ev_fork, 0));
            x.fl = f;
            x.fl.pid_base = std::min<uint32_t>(f.n_paths, (uint32_t)l * part);
            x.fl.n_paths = std::min<uint32_t>(f.n_paths - x.fl.pid_base, part);
            x.pl = lane_view(ps, x.fl.pid_base, l);
            x.ovf = lane_ovf(c, l);
            // pass 1: forward, recording shadow visibility
            launch_clear_counters(x.pl, f.max_bounces + 1, x.s);
            launch_fill_u32(vis + x.fl.pid_base, 0u, x.fl.n_paths, x.s);
            launch_generate(x.fl, x.pl, x.s);
        }
        for (int l = 0; l < nl; ++l) {
            const Lane& x = ln[l];
            launch_extend(S, x.pl.q[0], x.pl.counters, x.fl.n_paths, x.pl.o, x.pl.d, x.pl.hits,
                          fetch_counters(x.pl, 0), x.ovf, nullptr, x.s, tblocks);
        }
        for (uint32_t b = 0; b <= f.max_bounces; ++b) {
            for (int l = 0; l < nl; ++l) launch_shade(S, ln[l].fl, ln[l].pl, b, ln[l].s);
            if (b == f.max_bounces) break;
            for (int l = 0; l < nl; ++l) {
                const Lane& x = ln[l];
                launch_extend_connect(S, x.pl.q[(b + 1) & 1u], x.pl.counters + ext_counter(b + 1), x.fl.n_paths, x.pl.o, x.pl.d,
                                      x.pl.hits, x.pl.counters + sh_counter(b + 1), 2u * x.fl.n_paths,
                                      x.pl.sh_o, x.pl.sh_d, x.pl.sh_c, x.pl.ln0, x.pl.ln1,
                                      fetch_counters(x.pl, b + 1), x.ovf, vis, b, nullptr, x.s,
                                      tblocks);
            }
        }
        // pass 2: replay with the same random numbers, scatter gradients. The
        // replayed vertices come from the hit log, or (retrace) from tracing each
        // replayed ray again: the same origin and direction bit for bit, so the
        // same closest hit.
        for (int l = 0; l < nl; ++l) {
            const Lane& x = ln[l];
            launch_adjoint_init(x.pl, x.fl.pid_base, x.fl.n_paths, lrem, x.s);
            launch_clear_counters(x.pl, f.max_bounces + 1, x.s);
            launch_generate(x.fl, x.pl, x.s);
            if (retrace)
                launch_extend(S, x.pl.q[0], x.pl.counters, x.fl.n_paths, x.pl.o, x.pl.d, x.pl.hits,
                              fetch_counters(x.pl, 0), x.ovf, nullptr, x.s, tblocks);
        }
        for (uint32_t b = 0; b <= f.max_bounces; ++b) {
            for (int l = 0; l < nl; ++l)
                launch_shade_adjoint(S, ln[l].fl, ln[l].pl, b, vis, lrem, c->adj_dldi.as<float4>(), inv_spp, rec_key,
                                     rec_val, rec_count, rec_overflow, ln[l].s);
            if (!retrace || b == f.max_bounces) continue;
            for (int l = 0; l < nl; ++l) {
                const Lane& x = ln[l];
                launch_extend(S, x.pl.q[(b + 1) & 1u], x.pl.counters + ext_counter(b + 1), x.fl.n_paths, x.pl.o, x.pl.d, x.pl.hits,
                              fetch_counters(x.pl, b + 1), x.ovf, nullptr, x.s, tblocks);
            }
        }
        if (nl > 1) {
            for (int l = 0; l < nl; ++l) {
                HIPCHK(hipEventRecord(c->ev_lane[l], ln[l].s));
                HIPCHK(hipStreamWaitEvent(c->stream, c->ev_lane[l], 0));
            }
        }
        if (deterministic) {
            // the written records in vertex order, a stable sort of them by texel (only the key
            // bits the arena needs, whole 8-bit digits), then in-order segment sums
            uint32_t nvalid = 0;
            uint32_t* k2 = c->rec_key2.as<uint32_t>();
            uint32_t* v2 = c->rec_val2.as<uint32_t>();
            hipError_t e = compact_records(rec_count, nvert, rec_key, rec_val, c->rec_tiles.as<uint32_t>(), k2, v2,
                                           &nvalid, c->stream);
            if (e != hipSuccess) return fail_hip("compact_records", e);
            uint32_t key_bits = 8;
            while (key_bits < 32 && (uint64_t)c->grad_total > (1ull << key_bits)) key_bits += 8;
            e = radix_sort_pairs(k2, v2, nvalid, key_bits, c->rec_scratch.p, c->stream);
            if (e != hipSuccess) return fail_hip("radix_sort_pairs", e);
            launch_segment_reduce(k2, v2, nvalid, c->grad_arena.as<float>(), c->stream);
        }
        HIPCHK(hipGetLastError());
        sample += batch;
        remaining -= batch;
    }
    HIPCHK(hipEventRecord(c->ev_stop, c->stream));
    HIPCHK(hipEventSynchronize(c->ev_stop));
    c->stats.ms_total = elapsed(c->ev_start, c->ev_stop);
    c->stats.paths = npix * spp;
    if (rec_overflow) {
        uint32_t ovf = 0;
        HIPCHK(hipMemcpy(&ovf, rec_overflow, 4, hipMemcpyDeviceToHost));
        if (ovf)
            return fail(OHPT_ERR_UNSUPPORTED, "ohpt_adjoint: a path vertex had more texel gradients than the "
                                              "deterministic mode's record slots; the gradients are incomplete");
    }
    return OHPT_OK;
}

int ohpt_synchronize(ohpt_context* c) {
    if (!c) return fail(OHPT_ERR_INVALID_ARG, "ohpt_synchronize: null context");
    HIPCHK(enter(c));
    HIPCHK(hipStreamSynchronize(c->stream));
    return OHPT_OK;
}

int ohpt_get_stats(ohpt_context* c, ohpt_stats* out) {
    if (!c || !out) return fail(OHPT_ERR_INVALID_ARG, "ohpt_get_stats: null argument");
    *out = c->stats;
    return OHPT_OK;
}

extern "C++" {
namespace {
template <class F>
int produce(ohpt_context* c, void* out, size_t bytes, int on_device, F&& kernel) {
    HIPCHK(enter(c));
    if (on_device) {
        kernel(out);
        HIPCHK(hipGetLastError());
        HIPCHK(hipStreamSynchronize(c->stream));
        return OHPT_OK;
    }
    HIPCHK(c->tmp.ensure(bytes));
    kernel(c->tmp.p);
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(out, c->tmp.p, bytes, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    return OHPT_OK;
}
}  // namespace
}  // extern "C++"

int ohpt_read_accum(ohpt_context* c, float* out, int on_device) {
    if (!c || !out) return fail(OHPT_ERR_INVALID_ARG, "ohpt_read_accum: null argument");
    const uint32_t n = c->W * c->H;
    return produce(c, out, (size_t)n * 16, on_device, [&](void* dst) {
        launch_resolve(c->d_accum.as<float4>(), reinterpret_cast<float4*>(dst), n, c->stream);
    });
}

int ohpt_read_moments(ohpt_context* c, float* sum, float* sumsq, int on_device) {
    if (!c || (!sum && !sumsq)) return fail(OHPT_ERR_INVALID_ARG, "ohpt_read_moments: null argument");
    HIPCHK(enter(c));
    const size_t bytes = (size_t)c->W * c->H * 16;
    const hipMemcpyKind k = on_device ? hipMemcpyDeviceToDevice : hipMemcpyDeviceToHost;
    if (sum) HIPCHK(hipMemcpyAsync(sum, c->d_accum.p, bytes, k, c->stream));
    if (sumsq) HIPCHK(hipMemcpyAsync(sumsq, c->d_moments.p, bytes, k, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    return OHPT_OK;
}

int ohpt_read_display_sums(ohpt_context* c, float* out, int on_device) {
    if (!c || !out) return fail(OHPT_ERR_INVALID_ARG, "ohpt_read_display_sums: null argument");
    if (int r0 = need_guides(c, "ohpt_read_display_sums")) return r0;
    HIPCHK(enter(c));
    const hipMemcpyKind k = on_device ? hipMemcpyDeviceToDevice : hipMemcpyDeviceToHost;
    HIPCHK(hipMemcpyAsync(out, c->d_disp.p, (size_t)c->W * c->H * 16, k, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    return OHPT_OK;
}

int ohpt_read_pixels(ohpt_context* c, uint8_t* out, int on_device) {
    if (!c || !out) return fail(OHPT_ERR_INVALID_ARG, "ohpt_read_pixels: null argument");
    const uint32_t n = c->W * c->H;
    return produce(c, out, (size_t)n * 4, on_device, [&](void* dst) {
        launch_tonemap(c->d_accum.as<float4>(), reinterpret_cast<uint8_t*>(dst), n, c->stream);
    });
}

int ohpt_read_aovs(ohpt_context* c, float* albedo, float* normal, float* depth, int on_device) {
    if (!c) return fail(OHPT_ERR_INVALID_ARG, "ohpt_read_aovs: null context");
    if (int r0 = need_guides(c, "ohpt_read_aovs")) return r0;
    HIPCHK(enter(c));
    const uint32_t n = c->W * c->H;
    if (on_device) {
        launch_resolve_aovs(c->d_accum.as<float4>(), c->d_aov_albedo.as<float4>(), c->d_aov_normal.as<float4>(),
                            albedo, normal, depth, n, c->stream);
        HIPCHK(hipGetLastError());
        HIPCHK(hipStreamSynchronize(c->stream));
        return OHPT_OK;
    }
    HIPCHK(c->tmp.ensure((size_t)n * 36));
    float* ta = c->tmp.as<float>();
    float* tn = ta + (size_t)n * 4;
    float* td = tn + (size_t)n * 4;
    launch_resolve_aovs(c->d_accum.as<float4>(), c->d_aov_albedo.as<float4>(), c->d_aov_normal.as<float4>(), ta, tn,
                        td, n, c->stream);
    HIPCHK(hipGetLastError());
    if (albedo) HIPCHK(hipMemcpyAsync(albedo, ta, (size_t)n * 16, hipMemcpyDeviceToHost, c->stream));
    if (normal) HIPCHK(hipMemcpyAsync(normal, tn, (size_t)n * 16, hipMemcpyDeviceToHost, c->stream));
    if (depth) HIPCHK(hipMemcpyAsync(depth, td, (size_t)n * 4, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    return OHPT_OK;
}

// ---------------------------------------------------------------- denoise
int ohpt_denoise(ohpt_context* c, ohpt_denoiser* dn, float* out, int on_device) {
    if (!c || !dn || !out) return fail(OHPT_ERR_INVALID_ARG, "ohpt_denoise: null argument");
    if (int r0 = need_guides(c, "ohpt_denoise")) return r0;
    HIPCHK(enter(c));
    const uint32_t n = c->W * c->H;
    HIPCHK(c->dn_guides.ensure((size_t)n * 52));
    float* rad = c->dn_guides.as<float>();
    float* alb = rad + (size_t)n * 4;
    float* nrm = alb + (size_t)n * 4;
    float* dep = nrm + (size_t)n * 4;
    launch_resolve(c->d_accum.as<float4>(), reinterpret_cast<float4*>(rad), n, c->stream);
    launch_resolve_aovs(c->d_accum.as<float4>(), c->d_aov_albedo.as<float4>(), c->d_aov_normal.as<float4>(), alb,
                        nrm, dep, n, c->stream);
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(c->stream));
    float* dst = out;
    if (!on_device) {
        HIPCHK(c->dn_out.ensure((size_t)n * 16));
        dst = c->dn_out.as<float>();
    }
    const int rc = denoiser_infer_device(dn, rad, alb, nrm, dep, dst, c->W, c->H);
    if (rc != OHPT_OK) return rc;
    if (!on_device) HIPCHK(hipMemcpy(out, dst, (size_t)n * 16, hipMemcpyDeviceToHost));
    return OHPT_OK;
}

int ohpt_denoise_atrous(ohpt_context* c, float* out, int on_device) {
    if (!c || !out) return fail(OHPT_ERR_INVALID_ARG, "ohpt_denoise_atrous: null argument");
    if (int r0 = need_guides(c, "ohpt_denoise_atrous")) return r0;
    if (!(c->st.flags & OHPT_FLAG_AOVS))
        return fail(OHPT_ERR_STATE, "ohpt_denoise_atrous: the edge stops need OHPT_FLAG_AOVS");
    HIPCHK(enter(c));
    HIPCHK(c->dn_guides.ensure(svgf_scratch_bytes(c->W, c->H)));
    const uint32_t n = c->W * c->H;
    hipError_t ferr = hipSuccess;
    const int r = produce(c, out, (size_t)n * 16, on_device, [&](void* dst) {
        ferr = svgf_atrous(c->d_accum.as<float4>(), c->d_disp.as<float4>(), c->d_aov_albedo.as<float4>(),
                           c->d_aov_normal.as<float4>(), c->W, c->H, reinterpret_cast<float4*>(dst),
                           c->dn_guides.p, c->stream);
    });
    if (ferr != hipSuccess) return fail_hip("svgf_atrous", ferr);
    return r;
}

// ---------------------------------------------------------------- ray batches
extern "C++" {
namespace {
int ray_batch(ohpt_context* c, const float* rays, void* out, uint32_t n, int on_device, bool occl) {
    if (!c || !rays || !out) return fail(OHPT_ERR_INVALID_ARG, "ray batch: null argument");
    if (int r0 = need_tree(c, "ray batch")) return r0;
    if (n == 0) return OHPT_OK;
    HIPCHK(enter(c));
    DevBuf dr, dout;
    HIPCHK(ensure_trace_scratch(c, 1));
    const float4* r = reinterpret_cast<const float4*>(rays);
    void* o = out;
    const size_t out_bytes = (size_t)n * (occl ? 4 : 16);
    if (!on_device) {
        HIPCHK(dr.ensure((size_t)n * 32));
        HIPCHK(dout.ensure(out_bytes));
        HIPCHK(hipMemcpyAsync(dr.p, rays, (size_t)n * 32, hipMemcpyHostToDevice, c->stream));
        r = dr.as<float4>();
        o = dout.p;
    }
    const DevScene S = scene_view(c);
    uint32_t* const fetch = trace_fetch(c);
    uint32_t* const ovf = lane_ovf(c, 0);
    if (occl) launch_occluded_rays(S, r, reinterpret_cast<uint32_t*>(o), n, fetch, ovf, c->stream);
    else launch_trace_rays(S, r, reinterpret_cast<float4*>(o), n, fetch, ovf, c->stream);
    HIPCHK(hipGetLastError());
    if (!on_device) HIPCHK(hipMemcpyAsync(out, dout.p, out_bytes, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    return OHPT_OK;
}
}  // namespace
}  // extern "C++"

int ohpt_trace_rays(ohpt_context* c, const float* rays, float* hits, uint32_t n, int on_device) {
    return ray_batch(c, rays, hits, n, on_device, false);
}

int ohpt_occluded_rays(ohpt_context* c, const float* rays, uint32_t* out, uint32_t n, int on_device) {
    return ray_batch(c, rays, out, n, on_device, true);
}

// ohpt_trace_rays with device buffers and the per-device `scratch` array in
// place of the context's counters and overflow stacks that ray_batch uses: no allocation,
// no synchronisation, launches on the context's stream only.
int ohpt_trace_rays_noalloc(ohpt_context* c, const float* rays, float* hits, uint32_t n) {
    if (!c || (n && (!rays || !hits))) return fail(OHPT_ERR_INVALID_ARG, "ohpt_trace_rays_noalloc: null argument");
    if (int r0 = need_tree(c, "ohpt_trace_rays_noalloc")) return r0;
    if (n > kNoAllocMaxRays)
        return fail(OHPT_ERR_INVALID_ARG, "ohpt_trace_rays_noalloc: more than 2^31 rays in one call");
    if ((reinterpret_cast<uintptr_t>(rays) | reinterpret_cast<uintptr_t>(hits)) & 15u)
        return fail(OHPT_ERR_INVALID_ARG, "ohpt_trace_rays_noalloc: buffers must be 16-byte aligned");
    if (n == 0) return OHPT_OK;
    HIPCHK(enter(c));
    unsigned char* base = static_cast<unsigned char*>(noalloc_scratch(c->device));
    if (!base) return fail(OHPT_ERR_STATE, "ohpt_trace_rays_noalloc: scratch not resolved for this device");
    uint32_t* fetch = reinterpret_cast<uint32_t*>(base);          // kFetchWords, zeroed by a kernel at launch
    uint32_t* ovf = reinterpret_cast<uint32_t*>(base + kFetchWords * 4);
    launch_trace_rays(scene_view(c), reinterpret_cast<const float4*>(rays), reinterpret_cast<float4*>(hits), n,
                      fetch, ovf, c->stream, kNoAllocBlocks);
    HIPCHK(hipGetLastError());
    return OHPT_OK;
}

int ohpt_scene_tree_depth(ohpt_context* c, uint32_t* out) {
    if (!c || !out) return fail(OHPT_ERR_INVALID_ARG, "ohpt_scene_tree_depth: null argument");
    *out = c->tree_depth;
    return OHPT_OK;
}

}  // extern "C"
