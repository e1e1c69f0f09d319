// The reference's own estimator on the GPU (ohpt_settings.integrator =
// OHPT_INTEGRATOR_REFERENCE / _REFERENCE_GOLDEN): main() of
// shaders/rt/pt_raygen_offline.rgen in the offline profile with the closest-hit
// shader pt_closesthit.rchit and the miss shader pt_miss.rmiss, as the oracle
// restates it (oracle/oracle_compat.cpp):
//   * after the first hit a specular-sampled chain (:570-895), then a
//     diffuse-sampled chain (:897-1201), both added with no lobe weight; the
//     sample dimension index runs on from the first chain into the second;
//   * jittered-reflection "specular" directions with a GGX pdf for MIS;
//   * untextured materials sample the 1x1 UNORM sRGB8(baseColor) texture the
//     reference makes (rt_build.cpp:446-470): albedo = base * (srgb8/255)^2.2;
//   * lights are next-event only; surfaces emit only through emissive textures;
//   * the environment is read at v = asin(y)/pi + 0.5 and sampled at texel centres.
// In wavefront form, as ohpt_render's physically based path: every sample's
// rays are traced by the persistent traversal kernels (traverse.hip's node step,
// so hits match the oracle), a shading kernel runs the shader's arithmetic
// between two rays, and each pixel's samples are summed into the accumulation
// buffers (sum, count, sum of squares; readback divides).
// Beauty only: no first-hit guides, no adjoint.
#include "ohpt_trace.h"

namespace ohpt {
namespace {

using namespace trace;

// The same vector arithmetic as the oracle's restatement: normalize divides by
// the length (the product's f3 normalize multiplies by a reciprocal).
__device__ __forceinline__ f3 nrm(f3 a) {
    const float l = sqrtf(dot(a, a));
    return mk(a.x / l, a.y / l, a.z / l);
}
__device__ __forceinline__ f3 div(f3 a, float s) { return mk(a.x / s, a.y / s, a.z / s); }
__device__ __forceinline__ f3 mixv(f3 a, f3 b, float t) { return a * (1.0f - t) + b * t; }
__device__ __forceinline__ float mixf(float a, float b, float t) { return a * (1.0f - t) + b * t; }
__device__ __forceinline__ f3 reflect(f3 i, f3 n) { return i - n * (2.0f * dot(n, i)); }
__device__ __forceinline__ float clampf(float x, float lo, float hi) { return fminf(fmaxf(x, lo), hi); }
__device__ __forceinline__ f3 pow3(f3 a, float e) { return mk(powf(a.x, e), powf(a.y, e), powf(a.z, e)); }
__device__ __forceinline__ float pow5(float b) { return powf(fmaxf(b, 0.0f), 5.0f); }
__device__ __forceinline__ f3 s3(float s) { return mk(s, s, s); }
__device__ __forceinline__ float3 to3(f3 a) { return make_float3(a.x, a.y, a.z); }

constexpr float kPi = 3.14159265358979f;      // OHPT_PI of env_sampling.glsl
constexpr float kTwoPi = 6.28318530717959f;

// sampler_sobol.glsl (padded Owen-scrambled Sobol) or sampler_pcg.glsl's stateful hash-LCG
struct Sampler {
    bool sobol;
    uint32_t pixel_seed, index, pcg;
    __device__ __forceinline__ float s1(uint32_t dim) {
        if (sobol) return sobol_owen(pixel_seed, index, dim);
        pcg = pcg * 747796405u + 2891336453u;
        uint32_t w = ((pcg >> ((pcg >> 28u) + 4u)) ^ pcg) * 277803737u;
        w = (w >> 22u) ^ w;
        return (float)w / 4294967296.0f;
    }
};

// rt_build.cpp:458-461 (a float std::pow on the host: a double pow rounded to
// float gives the same correctly rounded value)
__device__ __forceinline__ float srgb8_unorm(float v) {
    const float p = (float)pow((double)v, (double)(1.0f / 2.4f));
    const float s = (v <= 0.0031308f) ? v * 12.92f : 1.055f * p - 0.055f;
    const uint32_t byte = (uint32_t)(clampf(s, 0.0f, 1.0f) * 255.0f + 0.5f);
    return (float)byte / 255.0f;
}

struct Hit {
    bool hit;
    f3 color;               // emissive at a hit, environment radiance at a miss
    f3 pos, normal, albedo;
    float rough, metal, env_pdf;
};

struct Ctx {
    const DevScene& S;
    bool env_on;
};

__device__ __forceinline__ float texel_density(const DevScene& S, int x, int y) {
    const int W = (int)S.env_w, H = (int)S.env_h;
    const float* cond = S.env_cond + (size_t)y * W;
    const float condDiff = cond[x] - (x > 0 ? cond[x - 1] : 0.0f);
    const float margDiff = S.env_marg[y] - (y > 0 ? S.env_marg[y - 1] : 0.0f);
    return condDiff * margDiff * (float)W * (float)H;
}

__device__ __forceinline__ int cdf_search(const float* cdf, int n, float u) {
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi) / 2;
        if (cdf[mid] < u) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

// sampleEnvMap / pdfEnvMap, env_sampling.glsl:52-95
__device__ __forceinline__ void env_sample_ref(const DevScene& S, float u1, float u2, f3& dir, float& pdf) {
    const int W = (int)S.env_w, H = (int)S.env_h;
    const int y = cdf_search(S.env_marg, H, u1);
    const int x = cdf_search(S.env_cond + (size_t)y * W, W, u2);
    const float uu = ((float)x + 0.5f) / (float)W, vv = ((float)y + 0.5f) / (float)H;
    const float phi = (uu - 0.5f) * kTwoPi, theta = vv * kPi;
    const float sinT = sinf(theta);
    dir = mk(sinT * cosf(phi), cosf(theta), sinT * sinf(phi));
    const float th = ((float)y + 0.5f) / (float)H * kPi;
    pdf = fmaxf(texel_density(S, x, y) / (kTwoPi * kPi * fmaxf(sinf(th), 1e-4f)), 0.0f);
}

__device__ __forceinline__ float env_pdf_ref(const DevScene& S, f3 dir) {
    const int W = (int)S.env_w, H = (int)S.env_h;
    const float theta = acosf(clampf(dir.y, -1.0f, 1.0f));
    const float phi = atan2f(dir.z, dir.x);
    const float u = phi / kTwoPi + 0.5f, v = theta / kPi;
    const int x = min(max((int)(u * (float)W), 0), W - 1);
    const int y = min(max((int)(v * (float)H), 0), H - 1);
    return fmaxf(texel_density(S, x, y) / (kTwoPi * kPi * fmaxf(sinf(theta), 1e-4f)), 0.0f);
}

// pt_miss.rmiss:51-81: the environment bilinear at v = asin(y)/pi + 0.5, REPEAT addressing
__device__ __forceinline__ void miss(const Ctx& c, f3 d, Hit& h) {
    h.hit = false;
    h.color = s3(0.0f);
    h.env_pdf = 0.0f;
    if (!c.env_on) return;
    const f3 dir = nrm(d);
    const float u = atan2f(dir.z, dir.x) / 6.2831853f + 0.5f;
    const float v = asinf(clampf(dir.y, -1.0f, 1.0f)) / 3.1415926f + 0.5f;
    const TexDesc t{reinterpret_cast<const float*>(c.S.env), nullptr, c.S.env_w, c.S.env_h, 4u, 0u};
    const float4 e = tex_bilinear(t, u, v);
    const float sc = c.S.env_intensity > 0.0f ? c.S.env_intensity : 1.0f;
    h.color = mk(e.x, e.y, e.z) * sc;
    h.env_pdf = env_pdf_ref(c.S, dir);
}

// The payload of traceRayEXT with the closest-hit shader (pt_closesthit.rchit:37-161)
// or the miss shader, from the closest hit r of the ray (o, d) over t in [0.001, 10000].
// srgb: the untextured materials' 1x1 sRGB8 texels, when a caller has them at hand.
__device__ __forceinline__ Hit hit_from(const Ctx& c, float4 r, f3 o, f3 d, const float4* srgb = nullptr) {
    Hit h;
    const DevScene& S = c.S;
    const uint32_t slot = __float_as_uint(r.y);
    if (slot == kMiss) {
        miss(c, d, h);
        return h;
    }
    h.hit = true;
    h.pos = o + d * r.x;
    const float u = r.z, v = r.w, w = 1.0f - u - v;
    const float4* ap = S.attrs + (size_t)slot * 4;
    const float4 a0 = ap[0], a1 = ap[1], a2 = ap[2], a3 = ap[3];
    const f3 n0 = mk(a0.x, a0.y, a0.z), n1 = mk(a0.w, a1.x, a1.y), n2 = mk(a1.z, a1.w, a2.x);
    const f3 interp = n0 * w + n1 * u + n2 * v;
    f3 N;
    if (dot(interp, interp) > 0.0001f) {
        N = nrm(nrm(interp));
    } else {
        const float4* tp = S.tris + (size_t)slot * 3;
        const f3 v0 = xyz(tp[0]);
        N = nrm(cross(xyz(tp[1]) - v0, xyz(tp[2]) - v0));
        if (dot(N, d) > 0.0f) N = -N;
    }
    const float tu = w * a2.y + u * a2.w + v * a3.y;
    const float tv = w * a2.z + u * a3.x + v * a3.z;
    const uint32_t m = min(__float_as_uint(a3.w), S.n_materials - 1u);
    const float4 m0 = S.mats[m * 4 + 0], m1 = S.mats[m * 4 + 1], m2 = S.mats[m * 4 + 2], m3 = S.mats[m * 4 + 3];
    f3 albedo = xyz(m0), tex;
    const int at = __float_as_int(m2.y), nt = __float_as_int(m3.x), ot = __float_as_int(m3.y);
    const int et = __float_as_int(m3.z);
    if (at >= 0) {
        const float4 t = tex_bilinear(S.tex[at], tu, tv);
        tex = mk(t.x, t.y, t.z);
    } else if (srgb) {
        tex = xyz(srgb[m]);
    } else {
        tex = mk(srgb8_unorm(albedo.x), srgb8_unorm(albedo.y), srgb8_unorm(albedo.z));
    }
    albedo = albedo * pow3(tex, 2.2f);
    if (nt >= 0) {
        const float4 t = tex_bilinear(S.tex[nt], tu, tv);
        const f3 mapN = nrm(mk(t.x, t.y, t.z) * 2.0f - s3(1.0f));
        f3 T, B;
        if (N.z < -0.9999f) {
            T = mk(0.0f, -1.0f, 0.0f);
            B = mk(-1.0f, 0.0f, 0.0f);
        } else {
            const float a = 1.0f / (1.0f + N.z);
            const float dd = -N.x * N.y * a;
            T = mk(1.0f - N.x * N.x * a, dd, -N.x);
            B = mk(dd, 1.0f - N.y * N.y * a, -N.y);
        }
        N = nrm(T * mapN.x + B * mapN.y + N * mapN.z);
    }
    h.normal = N;
    h.albedo = albedo;
    float rough = m0.w, metal = m1.x;
    if (ot >= 0) {
        const float4 t = tex_bilinear(S.tex[ot], tu, tv);
        rough *= t.y;
        metal *= t.z;
    }
    rough = fmaxf(rough, 0.04f);
    h.color = s3(0.0f);
    if (et >= 0) {
        const float4 t = tex_bilinear(S.tex[et], tu, tv);
        h.color = pow3(mk(t.x, t.y, t.z), 2.2f);
    }
    h.rough = fmaxf(fabsf(rough), 0.01f);          // unpackHitPbr, pbr_unpack.glsl:8-20
    h.metal = clampf(metal, 0.0f, 1.0f);
    h.env_pdf = 0.0f;
    return h;
}

// cosineHemisphere, pt_raygen_offline.rgen:93-100
__device__ __forceinline__ f3 cosine_hemisphere(f3 N, float u0, float u1) {
    const f3 up = fabsf(N.y) < 0.999f ? mk(0, 1, 0) : mk(1, 0, 0);
    const f3 T = nrm(cross(up, N));
    const f3 B = cross(N, T);
    const float r = sqrtf(u0);
    const float phi = 6.2831853f * u1;
    return nrm(T * r * cosf(phi) + B * r * sinf(phi) + N * sqrtf(fmaxf(0.0f, 1.0f - r * r)));
}

__device__ __forceinline__ float ggx_d(float NdotH, float rough, float pi) {
    const float a = rough * rough, a2 = a * a;
    const float denom = NdotH * NdotH * (a2 - 1.0f) + 1.0f;
    return a2 / (pi * denom * denom + 0.0001f);
}

struct LightSample {
    f3 L, Le;
    float shadow_dist, weight;
};

// :311-389 (and the copies at the later vertices)
__device__ LightSample sample_light(const DevScene& S, uint32_t k, f3 hitPos, Sampler& smp, uint32_t& dim) {
    LightSample s;
    const float4* rec = S.lights + (size_t)k * 5;
    const float4 pt = rec[0], ci = rec[1], dp = rec[2], ex = rec[3], ex2 = rec[4];
    const float type = pt.w;
    const f3 center = xyz(pt);
    const f3 lightDir = nrm(xyz(dp));
    const float r = fmaxf(dp.w, 0.01f);
    const float area = 4.0f * 3.14159f * r * r;
    s.Le = div(xyz(ci) * ci.w, fmaxf(area, 0.01f));
    s.L = s3(0.0f);
    s.shadow_dist = 0.0f;
    s.weight = 0.0f;
    if (type < 0.5f || (type >= 1.5f && type < 2.5f)) {
        const float u1 = smp.s1(dim), u2 = smp.s1(dim + 1u);
        dim += 2u;
        const float cosTheta = 1.0f - 2.0f * u1;
        const float sinTheta = sqrtf(fmaxf(0.0f, 1.0f - cosTheta * cosTheta));
        const float phi = 6.2831853f * u2;
        const f3 offset = mk(sinTheta * cosf(phi), sinTheta * sinf(phi), cosTheta) * r;
        const f3 toLight = center + offset - hitPos;
        const float lightDist = length(toLight);
        s.L = div(toLight, lightDist);
        s.shadow_dist = lightDist - 0.02f;
        const float lightArea = 4.0f * 3.14159f * r * r;
        if (type < 0.5f) {
            const float lightCos = fmaxf(dot(-s.L, nrm(offset)), 0.0f);
            s.weight = lightCos * lightArea / (lightDist * lightDist);
        } else {
            const float deg = 3.14159265358979f / 180.0f;
            const float innerCos = cosf(dp.w * deg), outerCos = cosf(ex.w * deg);
            float spot = clampf((dot(-s.L, lightDir) - outerCos) / (innerCos - outerCos + 0.001f), 0.0f, 1.0f);
            spot *= spot;
            s.weight = lightArea / (lightDist * lightDist) * spot;
        }
    } else if (type < 1.5f) {
        s.L = -lightDir;
        s.weight = 1.0f;
        s.shadow_dist = 10000.0f;
    } else {
        const f3 e1 = xyz(ex), e2 = xyz(ex2);
        const float au = smp.s1(dim), av = smp.s1(dim + 1u);
        dim += 2u;
        const f3 toLight = center + e1 * au + e2 * av - hitPos;
        const float lightDist = length(toLight);
        s.L = div(toLight, lightDist);
        const float lightCos = fmaxf(dot(-s.L, nrm(cross(e1, e2))), 0.0f);
        s.weight = lightCos * ex2.w / (lightDist * lightDist);
        s.shadow_dist = lightDist - 0.02f;
    }
    return s;
}

__device__ __forceinline__ f3 clamp_lum(f3 c, bool on, float limit) {
    if (on) {
        const float l = c.x * 0.2126f + c.y * 0.7152f + c.z * 0.0722f;
        if (l > limit) c = c * (limit / l);
    }
    return c;
}

// ------------------------------------------------------------ wavefront form
// The estimator path by path in the shader's order of arithmetic and sample
// dimensions, split at its rays: a shading step adds the
// contributions whose shadow rays the previous step traced unoccluded, takes the
// closest hit of the path's ray, emits the vertex's light and environment
// shadow rays (their contributions pending) and the next ray of the chain.
// Per-path state between steps: see RefFrame (ohpt_internal.h).
constexpr uint32_t kRefShadeBlock = 256;
constexpr uint32_t kRefChainMask = 3u;          // 0 camera ray, 1 specular chain, 2 diffuse chain
constexpr uint32_t kRefBounceShift = 2;         // 6 bits
constexpr uint32_t kRefDeltaBit = 1u << 8;      // the last direction was a delta (mirror) one
constexpr uint32_t kRefFinishBit = 1u << 9;     // the path only waits for its shadow rays
constexpr float kRefTmax = 10000.0f;

__device__ __forceinline__ Sampler ref_sampler(const RefFrame& f, uint32_t px, uint32_t py, uint32_t sidx) {
    return Sampler{f.sampler == OHPT_SAMPLER_SOBOL_OWEN, hash_pixel(px, py), sidx,
                   px * 1973u + py * 9277u + sidx * 26699u + 1u};
}

// :129-162: the camera ray; consumes dimensions 0 and 1 of smp
__device__ __forceinline__ f3 ref_camera_dir(const RefFrame& f, uint32_t px, uint32_t py, Sampler& smp) {
    const float jx = smp.s1(0) - 0.5f, jy = smp.s1(1) - 0.5f;
    const float uvx = ((float)px + 0.5f + jx + 0.0f) / (float)f.width;
    const float uvy = ((float)py + 0.5f + jy + 0.0f) / (float)f.height;
    const float ndcx = uvx * 2.0f - 1.0f, ndcy = uvy * 2.0f - 1.0f;
    const f3 fwd = mk(f.cam.forward[0], f.cam.forward[1], f.cam.forward[2]);
    const f3 right = mk(f.cam.right[0], f.cam.right[1], f.cam.right[2]);
    const f3 up = mk(f.cam.up[0], f.cam.up[1], f.cam.up[2]);
    const float tanY = fabsf(f.cam.tan_half_fov_y), tanX = tanY * ((float)f.width / (float)f.height);
    return nrm(fwd + right * ndcx * tanX - up * ndcy * tanY);
}

__global__ __launch_bounds__(256) void k_ref_generate(RefFrame f, PathState ps) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i == 0) ps.counters[0] = f.n_paths;
    if (i >= f.n_paths) return;
    const uint32_t pid = f.pid_base + i;
    const uint32_t npix = f.width * f.height;
    const uint32_t pixel = pixel_of_slot(pid % npix, f.width, f.height, f.row_groups);
    const uint32_t px = pixel % f.width, py = pixel / f.width;
    Sampler smp = ref_sampler(f, px, py, f.sample_base + pid / npix);
    const f3 dir = ref_camera_dir(f, px, py, smp);
    ps.o[pid] = make_float4(f.cam.position[0], f.cam.position[1], f.cam.position[2], kRefTmax);
    ps.d[pid] = f4(dir, 0.0f);
    ps.T[pid] = make_float4(1.0f, 1.0f, 1.0f, __uint_as_float(0u));
    ps.L[pid] = make_float4(0.0f, 0.0f, 0.0f, __uint_as_float(2u));
    ps.ln0[pid] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    ps.ln1[pid] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    ps.aov0[pid] = make_float4(0.0f, 0.0f, 0.0f, __uint_as_float(smp.pcg));
    ps.q[0][i] = pid;
}

// One path's registers during a shading step.
struct RefStep {
    Sampler smp;
    uint32_t dim, chain, bounce;
    bool lastDelta;
    float lastPdf;
    f3 thr, radiance;
    // emitted this step
    bool emit_l, emit_e, emit_next;
    float4 shl_o, shl_d, shl_c, she_o, she_d, she_c;
    f3 next_o, next_d;
};

// Next-event estimation at vertex v reached along inDir (:311-568 at the first
// hit, the copies at the chain vertices): the picked light's and the
// environment sample's shadow rays, with the contributions they add if unoccluded.
__device__ __forceinline__ void ref_nee(const Ctx& c, RefStep& P, const Hit& v, f3 inDir, bool first, uint32_t pid) {
    const DevScene& S = c.S;
    const uint32_t n = S.n_lights;
    const f3 F0 = mixv(s3(0.04f), v.albedo, v.metal);
    if (n > 0) {
        uint32_t sel = (uint32_t)(P.smp.s1(P.dim) * (float)n);
        P.dim += 1u;
        sel = min(sel, n - 1u);
        const LightSample ls = sample_light(S, sel, v.pos, P.smp, P.dim);
        const float NdotL = fmaxf(dot(v.normal, ls.L), 0.0f);
        if (NdotL > 0.0f && ls.weight > 0.0f) {
            const f3 V = nrm(-inDir);
            const f3 H = nrm(ls.L + V);
            const float NdotH = fmaxf(dot(v.normal, H), 0.001f);
            const float NdotV = fmaxf(dot(v.normal, V), 0.001f);
            const float VdotH = fmaxf(dot(V, H), 0.001f);
            const float D = ggx_d(NdotH, v.rough, first ? 3.14159265f : 3.14159f);
            const f3 F = F0 + (s3(1.0f) - F0) * pow5(1.0f - VdotH);
            const float k = (v.rough + 1.0f) * (v.rough + 1.0f) / 8.0f;
            const float G = (NdotL / (NdotL * (1.0f - k) + k)) * (NdotV / (NdotV * (1.0f - k) + k));
            const f3 spec = div(F * D * G, 4.0f * NdotV * NdotL + 0.001f);
            const f3 diff = div((s3(1.0f) - F) * (1.0f - v.metal) * v.albedo, 3.14159f);
            const f3 cl = first ? ls.Le * (diff * NdotL + spec * NdotL) * ls.weight * (float)n
                                : P.thr * ls.Le * (diff + spec) * NdotL * ls.weight * (float)n;
            P.shl_o = f4(v.pos + v.normal * 0.01f, ls.shadow_dist);
            P.shl_d = f4(ls.L, __uint_as_float(pid * 2u));
            P.shl_c = f4(cl, 1.0f);
            P.emit_l = true;
        }
    }
    if (!c.env_on) return;
    const float u1 = P.smp.s1(P.dim), u2 = P.smp.s1(P.dim + 1u);
    P.dim += 2u;
    f3 envDir;
    float envPdf;
    env_sample_ref(S, u1, u2, envDir, envPdf);
    const float NdotL = fmaxf(dot(v.normal, envDir), 0.0f);
    if (!(NdotL > 0.0f && envPdf > 0.0f)) return;
    Hit m;
    miss(c, envDir, m);
    const f3 V = nrm(-inDir);
    const f3 H = nrm(envDir + V);
    const float NdotH = fmaxf(dot(v.normal, H), 0.001f);
    const float NdotV = fmaxf(dot(v.normal, V), 0.001f);
    const float VdotH = fmaxf(dot(V, H), 0.001f);
    const float D = ggx_d(NdotH, v.rough, first ? 3.14159265f : kPi);
    const f3 F = F0 + (s3(1.0f) - F0) * pow5(1.0f - VdotH);
    const float k = (v.rough + 1.0f) * (v.rough + 1.0f) / 8.0f;
    const float G = (NdotL / (NdotL * (1.0f - k) + k)) * (NdotV / (NdotV * (1.0f - k) + k));
    const f3 spec = div(F * D * G, 4.0f * NdotV * NdotL + 0.001f);
    const f3 diff = div((s3(1.0f) - F) * (1.0f - v.metal) * v.albedo, kPi);
    const f3 brdf = diff + spec;
    const float cosI = fabsf(dot(nrm(inDir), v.normal));
    const f3 fresnel = F0 + (s3(1.0f) - F0) * pow5(1.0f - cosI);
    const float specProbMIS = mixf(maxc(fresnel) * (1.0f - v.rough * 0.9f), 1.0f, v.metal);
    const float bsdfPdf = mixf(NdotL / kPi, D * NdotH / (4.0f * VdotH + 1e-4f), specProbMIS);
    const float w = envPdf / fmaxf(envPdf + bsdfPdf, 1e-6f);
    const f3 cl = first ? div(m.color * brdf * NdotL * w, envPdf) : div(P.thr * m.color * brdf * NdotL * w, envPdf);
    P.she_o = f4(v.pos + v.normal * 0.01f, 10000.0f);
    P.she_d = f4(envDir, __uint_as_float(pid * 2u + 1u));
    P.she_c = f4(cl, 1.0f);
    P.emit_e = true;
}

// The first ray of a chain; false: the chain is empty (no bounces).
__device__ __forceinline__ bool ref_start_chain(const RefFrame& f, RefStep& P, uint32_t chain, f3 origin, f3 dir,
                                                f3 thr, float lastPdf, bool lastDelta) {
    P.chain = chain;
    P.bounce = 1u;
    P.thr = thr;
    P.lastPdf = lastPdf;
    P.lastDelta = lastDelta;
    if (f.max_bounces < 1u) return false;
    P.next_o = origin;
    P.next_d = dir;
    P.emit_next = true;
    return true;
}

// :570-615: the specular chain's first direction from the first hit
__device__ __forceinline__ bool ref_spec_start(const RefFrame& f, RefStep& P, const Hit& v, f3 rayDir) {
    f3 refl = reflect(rayDir, v.normal);
    if (v.rough > 0.01f) {
        const float j0 = P.smp.s1(P.dim), j1 = P.smp.s1(P.dim + 1u);
        P.dim += 2u;
        refl = nrm(refl + cosine_hemisphere(refl, j0, j1) * v.rough);
        if (dot(refl, v.normal) < 0.0f) {
            const float f0 = P.smp.s1(P.dim), f1 = P.smp.s1(P.dim + 1u);
            P.dim += 2u;
            refl = cosine_hemisphere(v.normal, f0, f1);
        }
    }
    float lastPdf = 1.0f;
    bool lastDelta = true;
    if (!(v.rough < 0.05f)) {
        const f3 Hs = nrm(-rayDir + refl);
        const float NdotHs = fmaxf(dot(v.normal, Hs), 0.001f);
        const float VdotHs = fmaxf(dot(-rayDir, Hs), 0.001f);
        lastPdf = ggx_d(NdotHs, v.rough, 3.14159265f) * NdotHs / (4.0f * VdotHs + 1e-4f);
        lastDelta = false;
    }
    return ref_start_chain(f, P, 1u, v.pos + v.normal * 0.01f, refl, mixv(s3(1.0f), v.albedo, v.metal), lastPdf,
                           lastDelta);
}

// :833-895 / :1139-1201: Russian roulette and the next direction at a chain
// vertex; false: the chain has ended.
__device__ __forceinline__ bool ref_continue(const RefFrame& f, RefStep& P, const Hit& v, f3 dir) {
    if (P.bounce > 1u) {
        const float q = maxc(P.thr);
        const float rr = P.smp.s1(P.dim);
        P.dim += 1u;
        if (q < 0.01f || rr > q) return false;
        P.thr = div(P.thr, q);
    }
    const f3 F0 = mixv(s3(0.04f), v.albedo, v.metal);
    const float cosI = fabsf(dot(nrm(dir), v.normal));
    const f3 fresnel = F0 + (s3(1.0f) - F0) * pow5(1.0f - cosI);
    float specProb = maxc(fresnel);
    specProb *= (1.0f - v.rough * 0.9f);
    specProb = mixf(specProb, 1.0f, v.metal);
    const float choice = P.smp.s1(P.dim);
    P.dim += 1u;
    f3 ndir;
    if (choice < specProb || v.rough < 0.05f) {
        f3 refl = reflect(dir, v.normal);
        if (v.rough > 0.01f) {
            const float j0 = P.smp.s1(P.dim), j1 = P.smp.s1(P.dim + 1u);
            P.dim += 2u;
            refl = nrm(refl + cosine_hemisphere(refl, j0, j1) * v.rough);
            if (dot(refl, v.normal) < 0.0f) {
                const float f0 = P.smp.s1(P.dim), f1 = P.smp.s1(P.dim + 1u);
                P.dim += 2u;
                refl = cosine_hemisphere(v.normal, f0, f1);
            }
        }
        ndir = refl;
        if (P.chain == 2u && f.revision == 0u) P.thr = P.thr * (v.albedo * (1.0f - v.metal));
        else P.thr = P.thr * mixv(s3(1.0f), v.albedo, v.metal);
        P.thr = div(P.thr, fmaxf(specProb, 0.01f));
        if (v.rough < 0.05f) {
            P.lastPdf = 1.0f;
            P.lastDelta = true;
        } else {
            const f3 Hs = nrm(-dir + ndir);
            const float NdotHs = fmaxf(dot(v.normal, Hs), 0.001f);
            const float VdotHs = fmaxf(dot(-dir, Hs), 0.001f);
            P.lastPdf = specProb * (ggx_d(NdotHs, v.rough, kPi) * NdotHs / (4.0f * VdotHs + 1e-4f));
            P.lastDelta = false;
        }
    } else {
        const float d0 = P.smp.s1(P.dim), d1 = P.smp.s1(P.dim + 1u);
        P.dim += 2u;
        ndir = cosine_hemisphere(v.normal, d0, d1);
        P.thr = P.thr * v.albedo;
        P.thr = div(P.thr, fmaxf(1.0f - specProb, 0.01f));
        P.lastPdf = (1.0f - specProb) * fmaxf(dot(ndir, v.normal), 0.0f) / kPi;
        P.lastDelta = false;
    }
    if (++P.bounce > f.max_bounces) return false;
    P.next_o = v.pos + v.normal * 0.01f;
    P.next_d = ndir;
    P.emit_next = true;
    return true;
}

// Queue entry j of step `step` (j >= count: the lane only takes part in the
// block's appends).
__device__ __forceinline__ void ref_shade_one(const DevScene& S, const RefFrame& f, const PathState& ps,
                                              uint32_t step, uint32_t j, uint32_t count, const float4* srgb,
                                              uint32_t* app) {
    const uint32_t* __restrict__ qin = ps.q[step & 1u];
    uint32_t* __restrict__ qout = ps.q[(step + 1u) & 1u];
    const bool active = j < count;
    RefStep P;
    P.emit_l = P.emit_e = P.emit_next = false;
    uint32_t pid = 0;
    if (active) {
        pid = qin[j];
        const Ctx c{S, S.env_w > 0 && S.env_h > 0};
        const bool clamp_on = (f.flags & OHPT_FLAG_FIREFLY_CLAMP) && f.firefly_clamp > 0.0f;
        const uint32_t npix = f.width * f.height;
        const uint32_t pixel = pixel_of_slot(pid % npix, f.width, f.height, f.row_groups);
        const uint32_t px = pixel % f.width, py = pixel / f.width, sidx = f.sample_base + pid / npix;
        const float4 o4 = ps.o[pid], d4 = ps.d[pid], T4 = ps.T[pid], L4 = ps.L[pid];
        const uint32_t bits = __float_as_uint(T4.w);
        P.smp = ref_sampler(f, px, py, sidx);
        if (!P.smp.sobol) P.smp.pcg = __float_as_uint(ps.aov0[pid].w);   // the PCG sampler's state
        P.dim = __float_as_uint(L4.w);
        P.chain = bits & kRefChainMask;
        P.bounce = (bits >> kRefBounceShift) & 63u;
        P.lastDelta = (bits & kRefDeltaBit) != 0;
        P.lastPdf = d4.w;
        P.thr = xyz(T4);
        P.radiance = xyz(L4);
        // what the previous step's shadow rays found unoccluded, in the shader's order
        const float4 p0 = ps.ln0[pid], p1 = ps.ln1[pid];
        if (p0.w == 2.0f) P.radiance = P.radiance + clamp_lum(xyz(p0), clamp_on, f.firefly_clamp);
        if (p1.w == 2.0f) P.radiance = P.radiance + clamp_lum(xyz(p1), clamp_on, f.firefly_clamp);
        bool done = (bits & kRefFinishBit) != 0, finishing = false;
        f3 value = clamp_lum(P.radiance, clamp_on, f.firefly_clamp);
        if (!done) {
            const f3 rd = xyz(d4);
            const float4 r = ps.hits[j];
            const Hit h = hit_from(c, r, xyz(o4), rd, srgb);
            bool chain_ended = false;
            if (P.chain == 0u) {   // the camera ray
                if (!h.hit) {
                    done = true;
                    value = clamp_lum(h.color, clamp_on, f.firefly_clamp);
                } else {
                    ps.aov1[pid] = r;
                    if (length(h.color) > 0.001f) P.radiance = P.radiance + h.color;
                    P.thr = s3(1.0f);
                    ref_nee(c, P, h, rd, true, pid);
                    chain_ended = !ref_spec_start(f, P, h, rd);
                }
            } else if (!h.hit) {
                float w = 1.0f;
                if (h.env_pdf > 0.0f && c.env_on && !P.lastDelta) w = P.lastPdf / fmaxf(P.lastPdf + h.env_pdf, 1e-6f);
                P.radiance = P.radiance + P.thr * h.color * w;
                chain_ended = true;
            } else {
                if (length(h.color) > 0.001f) P.radiance = P.radiance + P.thr * h.color;
                ref_nee(c, P, h, rd, false, pid);
                chain_ended = !ref_continue(f, P, h, rd);
            }
            if (!done && chain_ended && P.chain == 1u) {
                // :897-922: the diffuse chain from the first hit, rebuilt from the camera ray's hit
                Sampler cs = ref_sampler(f, px, py, sidx);
                const f3 cdir = ref_camera_dir(f, px, py, cs);
                const f3 cpos = mk(f.cam.position[0], f.cam.position[1], f.cam.position[2]);
                const Hit v0 = hit_from(c, ps.aov1[pid], cpos, cdir, srgb);
                const float d0 = P.smp.s1(P.dim), d1 = P.smp.s1(P.dim + 1u);
                P.dim += 2u;
                const f3 dir = cosine_hemisphere(v0.normal, d0, d1);
                chain_ended = !ref_start_chain(f, P, 2u, v0.pos + v0.normal * 0.01f, dir, v0.albedo,
                                               fmaxf(dot(dir, v0.normal), 0.0f) / kPi, false);
            }
            if (!done && chain_ended) {
                value = clamp_lum(P.radiance, clamp_on, f.firefly_clamp);
                if (P.emit_l || P.emit_e) {   // wait one step for the last vertex's shadow rays
                    finishing = true;
                    P.emit_next = true;
                } else {
                    done = true;
                }
            }
        }
        if (done) {
            if (!(value.x == value.x) || !(value.y == value.y) || !(value.z == value.z)) value = s3(0.0f);
            ps.L[pid] = f4(value, 1.0f);
        } else {
            const uint32_t nb = P.chain | (P.bounce << kRefBounceShift) | (P.lastDelta ? kRefDeltaBit : 0u) |
                                (finishing ? kRefFinishBit : 0u);
            ps.T[pid] = f4(P.thr, __uint_as_float(nb));
            ps.L[pid] = f4(P.radiance, __uint_as_float(P.dim));
            if (!P.smp.sobol) ps.aov0[pid] = make_float4(0.0f, 0.0f, 0.0f, __uint_as_float(P.smp.pcg));
            if (finishing) {
                ps.o[pid] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);   // t in [0.001, 0]: hits nothing
                ps.d[pid] = make_float4(0.0f, 1.0f, 0.0f, P.lastPdf);
            } else {
                ps.o[pid] = f4(P.next_o, kRefTmax);
                ps.d[pid] = f4(P.next_d, P.lastPdf);
            }
            ps.ln0[pid] = P.emit_l ? P.shl_c : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            ps.ln1[pid] = P.emit_e ? P.she_c : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
    }
    // queue appends (every thread of the block takes part)
    const QueueSlots at = block_append<kRefShadeBlock / 64>(ps.counters + ext_counter(step + 1u), P.emit_next,
                                                            P.emit_l, P.emit_e, app);
    if (P.emit_l) { ps.sh_o[at.sh_l] = P.shl_o; ps.sh_d[at.sh_l] = P.shl_d; }
    if (P.emit_e) { ps.sh_o[at.sh_e] = P.she_o; ps.sh_d[at.sh_e] = P.she_d; }
    if (P.emit_next) qout[at.next] = pid;
}

// Persistent over the step's queue (its length is known only on the device):
// blocks take 256 entries at a time. Each block first converts the materials'
// base colours to their sRGB8 texels (a double-precision pow per channel, as the
// reference's upload computes them) into LDS, once instead of at every hit.
constexpr uint32_t kRefSrgbMax = 256;
__global__ __launch_bounds__(kRefShadeBlock) void k_ref_shade(DevScene S, RefFrame f, PathState ps, uint32_t step) {
    __shared__ float4 srgb[kRefSrgbMax];
    __shared__ uint32_t app[2 * (kRefShadeBlock / 64) + 2];
    const uint32_t count = ps.counters[ext_counter(step)];
    if (blockIdx.x * kRefShadeBlock >= count) return;   // uniform per block
    const bool table = S.n_materials <= kRefSrgbMax;
    if (table) {
        for (uint32_t m = threadIdx.x; m < S.n_materials; m += kRefShadeBlock) {
            const float4 m0 = S.mats[m * 4];
            srgb[m] = make_float4(srgb8_unorm(m0.x), srgb8_unorm(m0.y), srgb8_unorm(m0.z), 0.0f);
        }
        __syncthreads();
    }
    for (uint32_t base = blockIdx.x * kRefShadeBlock; base < count; base += gridDim.x * kRefShadeBlock) {
        ref_shade_one(S, f, ps, step, base + threadIdx.x, count, table ? srgb : nullptr, app);
        __syncthreads();   // app is read before the next entries' appends
    }
}

// Per pixel, the batch's samples in sample order into the accumulation.
__global__ __launch_bounds__(256) void k_ref_accumulate(RefFrame f, const float4* __restrict__ L,
                                                        float4* __restrict__ accum, float4* __restrict__ moments) {
    const uint32_t npix = f.width * f.height;
    const uint32_t pixel = blockIdx.x * 256 + threadIdx.x;
    if (pixel >= npix) return;
    const uint32_t spp = f.n_paths / npix;
    const uint32_t slot = slot_of_pixel(pixel, f.width, f.height, f.row_groups);
    float sx = 0, sy = 0, sz = 0, qx = 0, qy = 0, qz = 0;
    for (uint32_t k = 0; k < spp; ++k) {
        const float4 r = L[k * npix + slot];
        sx += r.x; sy += r.y; sz += r.z;
        qx += r.x * r.x; qy += r.y * r.y; qz += r.z * r.z;
    }
    float4 acc = accum[pixel];
    acc.x += sx; acc.y += sy; acc.z += sz; acc.w += (float)spp;
    accum[pixel] = acc;
    float4 mo = moments[pixel];
    mo.x += qx; mo.y += qy; mo.z += qz;
    moments[pixel] = mo;
}

}  // namespace

void launch_ref_generate(const RefFrame& f, const PathState& ps, hipStream_t s) {
    if (f.n_paths == 0) return;
    k_ref_generate<<<(f.n_paths + 255) / 256, 256, 0, s>>>(f, ps);
}

void launch_ref_shade(const DevScene& S, const RefFrame& f, const PathState& ps, uint32_t step, hipStream_t s) {
    if (f.n_paths == 0) return;
    static uint32_t resident = 0;
    if (!resident) {
        int dev = 0, cus = 0, per_cu = 0;
        (void)hipGetDevice(&dev);
        (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
        (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_ref_shade, kRefShadeBlock, 0);
        resident = (uint32_t)(std::max(cus, 1) * std::max(per_cu, 1));
    }
    const uint32_t grid = std::min(resident, (f.n_paths + kRefShadeBlock - 1) / kRefShadeBlock);
    k_ref_shade<<<grid, kRefShadeBlock, 0, s>>>(S, f, ps, step);
}

void launch_ref_accumulate(const RefFrame& f, const PathState& ps, float4* accum, float4* moments, hipStream_t s) {
    const uint32_t npix = f.width * f.height;
    k_ref_accumulate<<<(npix + 255) / 256, 256, 0, s>>>(f, ps.L, accum, moments);
}

}  // namespace ohpt
