/*
 * ohpt.h — C-ABI of the MI355X path-tracing core.
 *
 * Plain C types only: pointers, sizes, PODs. No exceptions cross this
 * boundary. Every function returns OHPT_OK (0) or a negative error code and
 * leaves a message for ohpt_last_error() on the calling thread.
 *
 * One context owns one HIP stream on one device. Contexts are not
 * thread-safe; use one per host thread (the reference renderer is
 * single-threaded: ohao/gpu/vulkan/renderer.cpp:729-733).
 *
 * Reference interfaces replaced (paths relative to the reference tree):
 *   VulkanRenderer façade        ohao/gpu/vulkan/renderer.hpp:114-292
 *   IRTRendererProfile plugin    ohao/render/rt/rt_profile_renderer.hpp:7-86
 *   PathTracer::render           ohao/render/rt/path_tracer_render.cpp:38-1281
 *   scene→RT upload              ohao/gpu/vulkan/rt_build.cpp:825-906,
 *                                ohao/gpu/vulkan/light_upload.cpp:153-501
 */
#ifndef OHPT_H
#define OHPT_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define OHPT_ABI_VERSION 1

/* ---- status codes ---------------------------------------------------- */
enum {
    OHPT_OK = 0,
    OHPT_ERR_INVALID_ARG = -1,   /* null handle/pointer, bad size          */
    OHPT_ERR_HIP = -2,           /* a HIP runtime call failed              */
    OHPT_ERR_NO_SCENE = -3,      /* render before a scene was committed    */
    OHPT_ERR_OUT_OF_MEMORY = -4,
    OHPT_ERR_UNSUPPORTED = -5,
    OHPT_ERR_STATE = -6          /* call out of order (e.g. adjoint without forward state) */
};

/* ---- samplers (ohao/render/rt/sampler_types.hpp; shaders/includes/rt/sampler_api.glsl:16-41) */
enum {
    OHPT_SAMPLER_PCG32 = 0,      /* O'Neill PCG32, stream = pixel, state seeded from (seed, sample, vertex) */
    OHPT_SAMPLER_SOBOL_OWEN = 1  /* padded-4D Sobol + Burley-2020 Owen scramble (reference default) */
};

/* ---- render flags ------------------------------------------------------ */
enum {
    OHPT_FLAG_AOVS = 1u << 0,          /* write first-hit albedo/normal/depth AOVs (PT_FLAG_ENABLE_AOVS)
                                          and the display-space sums (ohpt_read_display_sums) */
    OHPT_FLAG_FIREFLY_CLAMP = 1u << 2, /* luminance clamp per sample (PT_FLAG_ENABLE_FIREFLY_CLAMP) */
    OHPT_FLAG_NO_ENV_NEE = 1u << 8,    /* disable env importance sampling (BSDF sampling only) */
    OHPT_FLAG_NO_LIGHT_NEE = 1u << 9   /* disable light/emitter NEE (BSDF sampling only) */
};

/* ---- integrators (ohpt_settings.integrator) ----------------------------- */
enum {
    /* Lambert + GGX-VNDF with NEE to lights, emitters and the environment,
       balance-heuristic MIS and Russian roulette (the default) */
    OHPT_INTEGRATOR_PHYSICAL = 0,
    /* the reference's own estimator, shaders/rt/pt_raygen_offline.rgen:129-1355
       with pt_closesthit.rchit and pt_miss.rmiss: a specular and a diffuse chain
       after the first hit, NEE-only lights, the 1x1 sRGB8 base-colour texture;
       Sobol dimensions consumed as the shader consumes them. Beauty and moments
       only: an accumulation holding its samples has no first-hit guides, so
       ohpt_read_aovs, ohpt_read_display_sums, ohpt_denoise and
       ohpt_denoise_atrous return OHPT_ERR_STATE until the next reset;
       ohpt_adjoint refuses it (OHPT_ERR_UNSUPPORTED), as ohpt_render does
       max_bounces above 30. */
    OHPT_INTEGRATOR_REFERENCE = 1,
    /* as OHPT_INTEGRATOR_REFERENCE with the revision of the shader the
       reference's committed golden images were rendered with (the diffuse
       chain's specular bounce weighted by mix(1, albedo, metallic), where
       pt_raygen_offline.rgen:1172 now has albedo * (1 - metallic)) */
    OHPT_INTEGRATOR_REFERENCE_GOLDEN = 2
};

/* ---- light types (ohao/scene/component/light_component.hpp:10-15) ------- */
enum {
    OHPT_LIGHT_SPHERE = 0,
    OHPT_LIGHT_DIRECTIONAL = 1,
    OHPT_LIGHT_SPOT = 2,
    OHPT_LIGHT_AREA_RECT = 3
};

/*
 * Light record: byte-for-byte the reference GPULight (80 B, std430),
 * ohao/render/rt/gpu_light.hpp:10-16, filled as in
 * ohao/gpu/vulkan/light_upload.cpp:157-181.
 */
typedef struct ohpt_light {
    float position_type[4];        /* xyz position, w = type                    */
    float color_intensity[4];      /* rgb color, w = intensity                  */
    float dir_param[4];            /* xyz direction, w = radius / inner angle   */
    float extra[4];                /* area: xyz edge1; spot: w = outer angle    */
    float extra2[4];               /* area: xyz edge2, w = area                 */
} ohpt_light;

/*
 * Material record (64 B). Mirrors the reference Material fields that reach
 * the ray-traced path (ohao/gpu/vulkan/material.hpp:11-41, packed in
 * ohao/gpu/vulkan/rt_build.cpp:236-257). `emissive` is uploaded here although
 * the reference drops it on this path; `specular_f0` is the dielectric F0
 * the reference hard-codes to 0.04 (0 gives a pure Lambert surface).
 * Texture ids index textures uploaded with ohpt_upload_texture; -1 = none.
 * Textures hold linear values (the reference samples UNORM textures and
 * raises albedo/emissive texels to the power 2.2 itself,
 * shaders/rt/pt_closesthit.rchit:108-113, :150-157; a caller converting
 * such images does that once at upload).
 */
typedef struct ohpt_material {
    float base_color[3];
    float roughness;
    float metallic;
    float specular_f0;
    float emissive[3];             /* emitted radiance; with emissive_tex, multiplies the texture */
    int32_t albedo_tex;            /* RGB texture, multiplies base_color        */
    int32_t roughness_tex;         /* channel 0 multiplies roughness            */
    int32_t metallic_tex;          /* channel 0 multiplies metallic             */
    /* tangent-space normal map, RGB in [0,1] -> normalize(2t-1), applied in
       the Frisvad basis of the interpolated normal (pt_closesthit.rchit:115-133) */
    int32_t normal_tex;
    /* packed occlusion/roughness/metallic: G multiplies roughness, B multiplies
       metallic, R (ambient occlusion) is not used by the path tracer
       (pt_closesthit.rchit:138-148) */
    int32_t orm_tex;
    /* RGB emission texture times `emissive` (pt_closesthit.rchit:150-157) */
    int32_t emissive_tex;
    int32_t reserved;
} ohpt_material;

/*
 * Render settings (subset of RTRenderSettings, ohao/render/rt/rt_settings.hpp:17-35,
 * that affects the offline integrator).
 */
typedef struct ohpt_settings {
    uint32_t max_bounces;          /* indirect bounces; extend rays per path = max_bounces + 1 */
    uint32_t rr_start;             /* first bounce index that applies Russian roulette */
    uint32_t sampler;              /* OHPT_SAMPLER_*                            */
    uint32_t flags;                /* OHPT_FLAG_*                               */
    float firefly_clamp;           /* luminance clamp when OHPT_FLAG_FIREFLY_CLAMP */
    float ray_eps;                 /* relative origin offset for secondary rays (0 = default 1e-4) */
    uint32_t integrator;           /* OHPT_INTEGRATOR_*                         */
    uint32_t reserved;
} ohpt_settings;

/* Pinhole camera in the reference's convention
 * (shaders/rt/pt_raygen_offline.rgen:144-162, render_dispatch.cpp:161-163):
 * dir = normalize(fwd + right*ndc.x*tan_y*aspect - up*ndc.y*tan_y). */
typedef struct ohpt_camera {
    float position[3];
    float forward[3];
    float right[3];
    float up[3];
    float tan_half_fov_y;
} ohpt_camera;

/* GPU timing of the last ohpt_render / ohpt_adjoint call (HIP events). */
typedef struct ohpt_stats {
    double ms_total;               /* generate -> accumulate                    */
    double ms_extend;              /* traversal kernels: closest-hit rays and, in ohpt_render,
                                      the shadow rays traced in the same launches */
    double ms_shade;
    double ms_connect;             /* separate shadow-ray kernels (ohpt_adjoint) */
    double ms_build;               /* last LBVH build                           */
    uint64_t rays_extend;          /* closest-hit rays traced                   */
    uint64_t rays_shadow;          /* shadow rays traced                        */
    uint64_t paths;
    uint64_t node_visits;          /* traversal BVH node visits, all rays (OHPT_RENDER_PROFILE only) */
    uint64_t tri_tests;            /* ray/triangle tests, all rays (OHPT_RENDER_PROFILE only) */
    uint32_t extend_launches;      /* traversal launches in the last call       */
    uint32_t reserved;
} ohpt_stats;

typedef struct ohpt_context ohpt_context;

/* ---- lifecycle -------------------------------------------------------------
 * replaces VulkanRenderer(W,H) + initialize() (renderer.hpp:116-121),
 * resize (renderer.hpp:125), shutdown (renderer.hpp:122). */
int ohpt_create(ohpt_context** out, int device, uint32_t width, uint32_t height);
int ohpt_destroy(ohpt_context* ctx);
int ohpt_resize(ohpt_context* ctx, uint32_t width, uint32_t height);
const char* ohpt_last_error(void);
int ohpt_abi_version(void);

/* ---- scene upload ------------------------------------------------------------
 * replaces updateSceneBuffers/buildBLASTLAS (scene_upload.cpp:21-190,
 * rt_build.cpp:825-906). Meshes are transformed to world space with the
 * column-major 4x4 `world` matrix (glm convention) and flattened into one
 * LBVH built on the GPU at commit. normals/uvs/mat_ids may be NULL
 * (geometric normal, zero uv, material 0). mat_ids are local to the mesh and
 * offset by material_base. */
int ohpt_scene_begin(ohpt_context* ctx);
int ohpt_scene_add_mesh(ohpt_context* ctx,
                        const float* positions, const float* normals, const float* uvs,
                        uint32_t num_vertices,
                        const uint32_t* indices, uint32_t num_triangles,
                        const uint32_t* mat_ids, uint32_t material_base,
                        const float* world /* 16 floats or NULL */);
int ohpt_scene_commit(ohpt_context* ctx);
/* Transform change without a rebuild (the TLAS instance-transform update of
 * rt_acceleration_structure.cpp:419-535): mesh = index in add order, world as
 * in ohpt_scene_add_mesh (NULL = identity). ohpt_scene_refit then refits the
 * committed tree: same topology and leaf order, every box recomputed from the
 * new triangles, the 4-wide nodes re-collapsed. Large motions degrade the
 * tree's quality, not its correctness; commit again to rebuild. */
int ohpt_scene_set_mesh_transform(ohpt_context* ctx, uint32_t mesh, const float* world);
int ohpt_scene_refit(ohpt_context* ctx);
int ohpt_scene_triangle_count(ohpt_context* ctx, uint64_t* out);
/* Maximum leaf depth of the committed LBVH (root = 1). */
int ohpt_scene_tree_depth(ohpt_context* ctx, uint32_t* out);

/* Device-side scene arrays after commit, for inspection/tests. Buffers are
 * host pointers; sizes in elements as documented in the implementation. */
int ohpt_scene_export_bvh(ohpt_context* ctx, void* nodes_out /* (n-1)*64 B */,
                          void* tris_out /* n*48 B */, uint32_t* leaf_prims_out /* n */);
/* The 4-wide nodes every ray query traverses (the binary LBVH collapsed two
 * levels per node): *count_out = node count; nodes4_out (count*128 B, may be
 * NULL to query the count) receives them when capacity >= count. */
int ohpt_scene_export_bvh4(ohpt_context* ctx, void* nodes4_out, uint32_t capacity, uint32_t* count_out);

/* Materials and textures: updateRTMaterialParams (rt_build.cpp:313-389)
 * rewrites materials without touching the BVH. Texels (and the vertices of
 * larger meshes) pass through a device staging buffer, of which the context
 * keeps up to 256 MB for the next upload. */
int ohpt_upload_materials(ohpt_context* ctx, const ohpt_material* materials, uint32_t count);
int ohpt_upload_texture(ohpt_context* ctx, int32_t* out_id, const float* texels,
                        uint32_t width, uint32_t height, uint32_t channels);
int ohpt_update_texture(ohpt_context* ctx, int32_t id, const float* texels, int texels_on_device);
int ohpt_texture_info(ohpt_context* ctx, int32_t id, uint32_t* width, uint32_t* height,
                      uint32_t* channels);
/* Releases every uploaded texture (ids restart at 0). Materials keep their
 * constants and lose their texture bindings until ohpt_upload_materials is
 * called again. Replaces the bindless array rebuild of a scene upload
 * (rt_build.cpp:391-823), which recreates the texture set instead of growing it. */
int ohpt_clear_textures(ohpt_context* ctx);

/* Lights: uploadLightBuffer / updateRTLightParams (light_upload.cpp:145-284). */
int ohpt_upload_lights(ohpt_context* ctx, const ohpt_light* lights, uint32_t count);

/* Environment: RGBA32F equirect, row 0 = +Y (light_upload.cpp:307-501);
 * the marginal/conditional CDF is built on the GPU (env_cdf.cpp:13-61).
 * pixels may be NULL with width=height=0 to clear the environment. */
int ohpt_upload_env(ohpt_context* ctx, const float* rgba, uint32_t width, uint32_t height);
int ohpt_set_env_intensity(ohpt_context* ctx, float scale);   /* setEnvIntensityScale */
int ohpt_export_env_cdf(ohpt_context* ctx, float* marginal /* H */, float* conditional /* W*H */,
                        float* integral);
/* Environment importance samples as the integrator draws them
 * (shaders/includes/rt/env_sampling.glsl:16-74), for inspection: u = n pairs in
 * [0,1)^2 (host), out = n x (dir.x, dir.y, dir.z, pdf) (host); pdf 0 where no
 * sample is produced. */
int ohpt_env_sample(ohpt_context* ctx, const float* u, float* out, uint32_t n);

/* ---- per-frame state --------------------------------------------------- */
int ohpt_set_camera(ohpt_context* ctx, const ohpt_camera* cam);
int ohpt_set_settings(ohpt_context* ctx, const ohpt_settings* settings);
int ohpt_get_settings(ohpt_context* ctx, ohpt_settings* settings);
/* resetAccumulation (path_tracer.cpp:189-191): sample index <- seed, count <- 0 */
int ohpt_reset_accumulation(ohpt_context* ctx);
/* setRenderSeed (renderer.hpp:160): base sample index after reset */
int ohpt_set_render_seed(ohpt_context* ctx, uint32_t seed);

/* ---- rendering -------------------------------------------------------------
 * Traces `spp` samples per pixel into the running-mean accumulation buffer
 * (pt_raygen_offline.rgen:1211-1262). Synchronous with respect to the host
 * unless OHPT_RENDER_ASYNC is given; unlike the reference's 3-deep frame ring
 * (render_dispatch.cpp:139-141) results are visible right after the call.
 * Consecutive calls with OHPT_RENDER_ASYNC and no other call in between
 * overlap on the GPU (each of a frame's wavefront lanes starts the next frame
 * when it is done with its part of this one); any other call on the context
 * is ordered after every render before it, and a render after it waits for it.
 * The accumulated result is the same, bit for bit, however the calls overlap. */
enum {
    OHPT_RENDER_ASYNC = 1u << 0,    /* return without waiting for the GPU          */
    OHPT_RENDER_PROFILE = 1u << 1   /* time every kernel with HIP events and count node
                                       visits; the frame then runs as one wavefront on
                                       the context stream (no concurrent lanes)    */
};
int ohpt_render(ohpt_context* ctx, uint32_t spp, uint32_t render_flags);
int ohpt_synchronize(ohpt_context* ctx);
int ohpt_get_stats(ohpt_context* ctx, ohpt_stats* out);
/* Accumulated HDR beauty, RGBA32F: the per-pixel mean radiance (w = sample count). `on_device` != 0 means
 * `out` is a device pointer on this context's device. */
int ohpt_read_accum(ohpt_context* ctx, float* out, int on_device);
/* Raw per-pixel sums since the last reset: sum = (sum r, g, b, sample count),
 * sumsq = (sum r^2, g^2, b^2, 0), RGBA32F each. Either may be NULL. Used for
 * per-pixel variance (no reference counterpart: the reference keeps only the
 * running mean). */
int ohpt_read_moments(ohpt_context* ctx, float* sum, float* sumsq, int on_device);
/* Display-space sums since the last reset, recorded with OHPT_FLAG_AOVS:
 * (sum of the per-sample display value (ACES(x*0.5))^(1/2.2) per channel,
 * sum of its squared luminance), RGBA32F: the colour and luminance moments
 * the reference's SVGF temporal pass accumulates (rt_svgf_temporal.comp:87-99),
 * read by ohpt_denoise_atrous. */
int ohpt_read_display_sums(ohpt_context* ctx, float* out, int on_device);
/* RGBA8: (ACES(x*0.5))^(1/2.2) as pt_raygen_offline.rgen:1338-1354. */
int ohpt_read_pixels(ohpt_context* ctx, uint8_t* out, int on_device);
/* First-hit AOVs (readbackHDRBuffers, render_dispatch.cpp:536-626):
 * albedo RGBA32F, normal RGBA32F (world normal, w=1 on hit), depth F32. Any may be NULL. */
int ohpt_read_aovs(ohpt_context* ctx, float* albedo, float* normal, float* depth, int on_device);

/* ---- differentiation ---------------------------------------------------------
 * Path-replay adjoint of the image formed by the first `spp` samples after a
 * reset (sample indices seed .. seed+spp-1). dl_dimage is dL/d(mean radiance)
 * per pixel, RGBA32F (alpha ignored). Gradients with respect to every texel of
 * every texture bound as albedo (RGB), roughness or metallic (channel 0)
 * accumulate into per-texture buffers. Replaces the coordinate finite
 * differences of StagedFitter::runStage (ohao/inverse/staged_fit.hpp:296-357)
 * and turns IInverseImageFormation::supportsAnalyticGrads
 * (ohao/inverse/backend/image_formation.hpp:53) on for the path tracer.
 * Requires max_bounces <= 15. With OHPT_ADJOINT_DETERMINISTIC the texel sums
 * are order-independent (bit-reproducible); otherwise FP32 atomics. The replay
 * reads the closest hit of every vertex from a log the forward pass writes
 * (16 B per path vertex); with OHPT_ADJOINT_RETRACE it re-traces each path
 * with the same random numbers instead, as path replay is published, storing
 * nothing per vertex (same gradients, one more traversal per vertex). */
enum { OHPT_ADJOINT_DETERMINISTIC = 1u << 0, OHPT_ADJOINT_RETRACE = 1u << 1 };
int ohpt_adjoint(ohpt_context* ctx, const float* dl_dimage, int on_device, uint32_t spp, uint32_t flags);
int ohpt_zero_gradients(ohpt_context* ctx);
/* dL/d(texel) of texture `id`, w*h*channels floats (the upload layout). */
int ohpt_read_texture_gradient(ohpt_context* ctx, int32_t id, float* out, int on_device);

/* Trace a batch of caller-supplied rays (closest hit). rays: n x 8 floats
 * (ox,oy,oz,tmin, dx,dy,dz,tmax); hits: n x 4 (t, prim as uint bits, u, v),
 * prim = 0xFFFFFFFF on miss. prim is the caller's global triangle numbering
 * (mesh order, then triangle order). Device pointers when on_device != 0. The
 * first query allocates the traversal's stack slots, which the context keeps
 * (about 100 MB on a 256-CU device); renders keep three times as many and
 * queries share them. */
int ohpt_trace_rays(ohpt_context* ctx, const float* rays, float* hits, uint32_t n, int on_device);
/* Occlusion query: out[i] = 1 if any hit in (tmin, tmax). */
int ohpt_occluded_rays(ohpt_context* ctx, const float* rays, uint32_t* out, uint32_t n, int on_device);

/* ohpt_trace_rays without any allocation. No counterpart in the reference: it
 * is for callers that cannot allocate device memory — code under HIP graph
 * capture, tight serving loops, harnesses that forbid hipMalloc. rays and hits
 * are device pointers on the context's device (16-byte aligned, same layouts
 * as ohpt_trace_rays); results equal ohpt_trace_rays's bit for bit. The
 * traversal's fetch counter and stack-overflow slots live in one fixed array
 * per device (36 MiB + 8 KiB, held until the process ends), the counters
 * cleared by a kernel at each call of more than 131,072 rays (fewer need
 * none). The call only enqueues work on the context's stream
 * (ohpt_synchronize before reading hits on the host). Calls that overlap on
 * one device — from any contexts or threads — race on that array and must be
 * serialised by the caller. n above 2^31 is rejected (OHPT_ERR_INVALID_ARG). */
int ohpt_trace_rays_noalloc(ohpt_context* ctx, const float* rays, float* hits, uint32_t n);

/* ---- learned denoiser ----------------------------------------------------------
 * Kernel-predicting U-Net: 10 input channels (log1p radiance, albedo, normal,
 * log1p depth) in bfloat16, five levels of 3x3 convolutions with 32/64/96/128/160
 * channels, 2x2 max-pool down, bilinear x2 up with skip concatenation, and a
 * head predicting per-pixel 5x5 softmax filter weights applied to the noisy
 * radiance. Convolutions run on the matrix cores in BF16 with FP32 accumulation;
 * parameters and Adam state are FP32. Images of any size are padded to a
 * multiple of 16 by edge replication.
 *
 * Takes the place of the reference's denoise stage: oidnDenoise
 * (ohao/render/rt/denoise/oidn_denoise.hpp:14-17, same beauty/albedo/normal
 * guides), selected through VulkanRenderer::setDenoiseMode
 * (ohao/gpu/vulkan/renderer.hpp:182) and applied lazily by getPixels
 * (renderer.hpp:255-258). One denoiser owns one HIP stream; not thread-safe. */
typedef struct ohpt_denoiser ohpt_denoiser;

/* Guide images of `batch` images, each width*height pixels, row-major.
 * radiance, albedo, normal: RGBA32F (alpha ignored); depth: F32. albedo,
 * normal and depth may be NULL (that channel group is then zero). */
typedef struct ohpt_denoise_inputs {
    const float* radiance;
    const float* albedo;
    const float* normal;
    const float* depth;
} ohpt_denoise_inputs;

typedef struct ohpt_denoiser_stats {
    float ms_total;          /* GPU time of the last infer / train call         */
    float ms_conv;           /* of which 3x3 convolution kernels (when profiled) */
    double conv_flops;       /* algorithmic 3x3-convolution FLOPs of that call   */
    uint32_t padded_width, padded_height, batch, reserved;
} ohpt_denoiser_stats;

/* Parameters are initialised from `seed` (He-normal convolutions, zero bias,
 * near-zero head so the untrained filter is a 5x5 box). */
int ohpt_denoiser_create(ohpt_denoiser** out, int device, uint64_t seed);
int ohpt_denoiser_destroy(ohpt_denoiser* dn);
/* FP32 parameters: for each convolution in network order, W[tap][cin][cout]
 * then bias[cout]. set_params resets the Adam moments and step count. */
int ohpt_denoiser_param_count(ohpt_denoiser* dn, uint64_t* n);
int ohpt_denoiser_get_params(ohpt_denoiser* dn, float* out, uint64_t n);
int ohpt_denoiser_set_params(ohpt_denoiser* dn, const float* in, uint64_t n);
/* Gradient of the last forward_backward / train_step, same layout. */
int ohpt_denoiser_get_grads(ohpt_denoiser* dn, float* out, uint64_t n);
/* Loss = mean over pixels and RGB of |T(out) - T(target)| with
 * T(x) = (ACES(0.5 x) + 1e-3)^(1/2.2); target RGBA32F. Computes the gradient
 * of every parameter; *loss receives the loss (host pointer, may be NULL). */
int ohpt_denoiser_forward_backward(ohpt_denoiser* dn, const ohpt_denoise_inputs* in, const float* target,
                                   uint32_t batch, uint32_t width, uint32_t height, float* loss, int on_device);
/* One Adam step (beta1 0.9, beta2 0.999, eps 1e-8, bias-corrected) with the
 * stored gradient. */
int ohpt_denoiser_adam_step(ohpt_denoiser* dn, float lr);
int ohpt_denoiser_train_step(ohpt_denoiser* dn, const ohpt_denoise_inputs* in, const float* target,
                             uint32_t batch, uint32_t width, uint32_t height, float lr, float* loss, int on_device);
/* Denoised RGBA32F (alpha = 1) of `batch` images. */
int ohpt_denoiser_infer(ohpt_denoiser* dn, const ohpt_denoise_inputs* in, float* out, uint32_t batch,
                        uint32_t width, uint32_t height, int on_device);
/* Intermediate tensor `index` of the last call as FP32, for tests: 0..26 are
 * the network activations in evaluation order (NHWC, padded size), 27 the
 * head logits (32 channels, 25 used), 100+i the gradient of activation i,
 * 127 the gradient of the logits. n = element count of `out` (host).
 * Inference computes the input features (x0), the decoder's upsampled inputs
 * (u3, u2, u1, u0) and the head logits inside the convolutions without
 * storing them; they are stored by forward_backward / train_step. */
int ohpt_denoiser_read_tensor(ohpt_denoiser* dn, uint32_t index, float* out, uint64_t n);
int ohpt_denoiser_get_stats(ohpt_denoiser* dn, ohpt_denoiser_stats* out);
/* on != 0: time every convolution launch with HIP events (fills ms_conv). */
int ohpt_denoiser_set_profiling(ohpt_denoiser* dn, int on);
/* Denoise the context's current accumulation (mean beauty + first-hit AOVs)
 * into out (width*height RGBA32F of the context). */
int ohpt_denoise(ohpt_context* ctx, ohpt_denoiser* dn, float* out, int on_device);

/* Variance-guided a-trous filter (the SVGF spatial pass) of the context's
 * current accumulation into out (width*height RGBA32F display values in
 * [0,1], alpha 1): replaces AtrousDenoiser::dispatch
 * (ohao/render/rt/denoise/atrous_denoise.hpp:59-60) with
 * shaders/rt/rt_svgf_atrous.comp:49-115 over 5 iterations (steps 1..16,
 * sigmaL 0.4, sigmaNormal 0.3, sigmaDepth 2.0, atrous_denoise.cpp:29-40).
 * Input colour = the mean per-sample display value, variance = the
 * per-sample display-luminance variance (raised to the 3x3 spatial variance
 * below 4 samples, rt_svgf_temporal.comp:105-120), normal/depth = the
 * first-hit AOVs (OHPT_FLAG_AOVS must be set, else OHPT_ERR_STATE). */
int ohpt_denoise_atrous(ohpt_context* ctx, float* out, int on_device);

#ifdef __cplusplus
}
#endif

#endif /* OHPT_H */
