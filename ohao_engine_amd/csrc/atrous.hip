// Variance-guided a-trous wavelet filter (SVGF's spatial pass), the reference's
// DenoiseMode::Atrous comparator (AtrousDenoiser, ohao/render/rt/denoise/
// atrous_denoise.hpp:44-67; shaders/rt/rt_svgf_atrous.comp:42-114), run on the
// accumulated frame. Its inputs are what the reference's temporal pass
// (rt_svgf_temporal.comp:87-120) hands over for a still camera, one sample per
// frame:
//   * colour = the mean of the per-sample display values (ACES(x/2)^(1/2.2)),
//   * variance = E[l^2] - E[l]^2 of the per-sample display luminance l,
//     raised to the 3x3 spatial luminance variance while fewer than 4 samples
//     are in (the temporal pass's bootstrap, rt_svgf_temporal.comp:105-120);
//   * normal / depth = the first-hit AOVs (mean normal, mean hit distance
//     over the hits; background 1e30 when fewer than half the samples hit);
//   * 5 iterations, steps 1, 2, 4, 8, 16, B3-spline taps, the reference's
//     sigmaL 0.4, sigmaNormal 0.3, sigmaDepth 2.0 (atrous_denoise.cpp:38-40).
// The colour and moments are exact means over all samples where the
// reference's exponential average caps the history at 20 frames (alpha 0.05).
#include "ohpt_internal.h"

namespace ohpt {
namespace {

constexpr float kLw[3] = {0.2126f, 0.7152f, 0.0722f};

__device__ __forceinline__ float luma(float4 c) { return kLw[0] * c.x + kLw[1] * c.y + kLw[2] * c.z; }

// Blocks of 64 x 4: a wave reads one row segment of 64 records per tap.
constexpr int kBX = 64, kBY = 4;

// Per-pixel records: cv = (display colour rgb, luminance variance), geo =
// (normal xyz, depth): one 16-byte load each per filter tap. While a pixel has
// fewer than 4 samples its moment variance is unreliable, so the variance is at
// least the 3x3 luminance variance of the display image (taps clamped to the edge,
// 9 of them), rt_svgf_temporal.comp:105-120.
// Bounded by HBM (96 B per pixel, the neighbours hit the caches): 1920x1080 in 41 us
// where a record pass and a variance pass over its output took 29 + 20 us.
__global__ __launch_bounds__(256) void k_svgf_prep(const float4* __restrict__ acc, const float4* __restrict__ disp,
                                                   const float4* __restrict__ aa, const float4* __restrict__ an, int W,
                                                   int H, float4* __restrict__ cv, float4* __restrict__ geo) {
    const int x = blockIdx.x * kBX + (threadIdx.x % kBX), y = blockIdx.y * kBY + (threadIdx.x / kBX);
    if (x >= W || y >= H) return;
    const int p = y * W + x;
    auto colour = [&](int q, float inv) {
        const float4 d = disp[q];
        return make_float4(d.x * inv, d.y * inv, d.z * inv, d.w * inv);
    };
    const float cnt = acc[p].w;
    const float4 al = aa[p], nm = an[p];
    const float inv = cnt > 0.0f ? 1.0f / cnt : 0.0f;
    float4 c = colour(p, inv);
    const float m1 = luma(c);
    c.w = fmaxf(0.0f, c.w - m1 * m1);
    if (cnt < 4.0f) {
        float s = 0.0f, s2 = 0.0f;
#pragma unroll
        for (int dy = -1; dy <= 1; ++dy)
#pragma unroll
            for (int dx = -1; dx <= 1; ++dx) {
                const int q = min(max(y + dy, 0), H - 1) * W + min(max(x + dx, 0), W - 1);
                const float qc = acc[q].w;
                const float l = luma(colour(q, qc > 0.0f ? 1.0f / qc : 0.0f));
                s += l;
                s2 += l * l;
            }
        const float mm = s / 9.0f;
        c.w = fmaxf(c.w, fmaxf(0.0f, s2 / 9.0f - mm * mm));
    }
    cv[p] = c;
    float nx = nm.x * inv, ny = nm.y * inv, nz = nm.z * inv;
    const float len = sqrtf(nx * nx + ny * ny + nz * nz);
    if (len > 0.0f) { nx /= len; ny /= len; nz /= len; }
    const float hits = nm.w;   // samples whose primary ray hit (the AOV hit flag summed)
    const float depth = (hits * 2.0f > cnt && hits > 0.0f) ? al.w / hits : 1e30f;
    geo[p] = make_float4(nx, ny, nz, depth);
}

// One iteration, rt_svgf_atrous.comp:49-115. The three edge stops are one
// exponential of the summed exponents. The last iteration writes alpha 1.
//
// A thread filters R pixels of its column, `step` rows apart: they share tap rows,
// so R + 4 rows of five taps are loaded for R outputs (10 taps per pixel at R = 4
// where one pixel per thread loads 25), and a tap's luminance is taken once. Rows
// are uniform per wave (scalar row addresses). Bounded by vector issue, about 16
// operations and a quarter-rate exponential per tap and output; one pixel per
// thread was bounded by the 50 16-byte L1 reads per pixel. 1920x1080:
// 121 us an iteration with one pixel per thread, 54 us now; the whole filter 0.64 -> 0.30 ms.
//
// The exponential is the hardware's base-2 one (error below 1 ulp) of an exponent summed in
// base 2, log2(e) folded into the three factors. expf carries e log2(e) as two floats,
// but e already is off by several roundings of its products, so that buys nothing: over 16
// frames (97x63 to 1920x1080, 1 to 8 samples) the result's relative error against 64 bits is
// 6.3e-7 to 4.0e-6, mean 1.9552e-6, and with expf 6.4e-7 to 4.0e-6, mean 1.9557e-6 (one pixel
// per thread with expf 1.9560e-6); expf takes 367 us for the whole 1920x1080 filter where this
// takes 330.
template <int R>
__global__ __launch_bounds__(256, 4) void k_svgf_atrous(const float4* __restrict__ cvin, const float4* __restrict__ geo,
                                                     int W, int H, int step, int last, float sigma_l, float sigma_n,
                                                     float sigma_d, float4* __restrict__ cvout) {
    const int x = blockIdx.x * kBX + (threadIdx.x % kBX);
    // row group j: rows y0, y0 + step, .. of a band of R * step rows
    const int j = __builtin_amdgcn_readfirstlane((int)(blockIdx.y * kBY + threadIdx.x / kBX));
    const int band = j / step;
    const int y0 = band * R * step + (j - band * step);
    if (x >= W || y0 >= H) return;
    const float kLog2e = 1.4426950408889634f;
    const float inv_n = kLog2e / (sigma_n * sigma_n + 1e-4f);
    const float inv_d = kLog2e / (sigma_d * sigma_d + 1e-4f);
    int xq[5];
#pragma unroll
    for (int dx = 0; dx < 5; ++dx) xq[dx] = min(max(x + (dx - 2) * step, 0), W - 1);
    const int xm = max(x - 1, 0), xp = min(x + 1, W - 1);
    float4 cg[R];
    float cl[R], cvar[R], inv_l[R];
    float sr[R], sg[R], sb[R], ws[R], vs[R];
#pragma unroll
    for (int k = 0; k < R; ++k) {
        const int y = min(y0 + k * step, H - 1);   // rows below the image are not written
        cg[k] = geo[(size_t)y * W + x];
        cl[k] = luma(cvin[(size_t)y * W + x]);
        // 3x3 Gaussian prefilter of the variance for the luminance edge stop (weights sum to 1)
        const float gk[3] = {0.25f, 0.5f, 0.25f};
        float v = 0.0f;
#pragma unroll
        for (int dy = -1; dy <= 1; ++dy) {
            const float4* row = cvin + (size_t)min(max(y + dy, 0), H - 1) * W;
            v += gk[dy + 1] * (gk[0] * row[xm].w + gk[1] * row[x].w + gk[2] * row[xp].w);
        }
        cvar[k] = v;
        inv_l[k] = kLog2e / (sqrtf(fmaxf(v, 1e-8f)) * sigma_l + 1e-6f);
        sr[k] = sg[k] = sb[k] = ws[k] = vs[k] = 0.0f;
    }
    const float kb[5] = {1.0f / 16.0f, 4.0f / 16.0f, 6.0f / 16.0f, 4.0f / 16.0f, 1.0f / 16.0f};
#pragma unroll
    for (int m = 0; m < R + 4; ++m) {
        int qy = min(max(y0 + (m - 2) * step, 0), H - 1);
        // a row's loads stay behind the last row's sums: 10 records in registers, not 40
#pragma unroll
        for (int k = 0; k < R; ++k)
            asm volatile("" : "+v"(sr[k]), "+v"(sg[k]), "+v"(sb[k]), "+v"(ws[k]), "+v"(vs[k]));
        asm volatile("" : "+s"(qy));
        const float4* crow = cvin + (size_t)qy * W;
        const float4* grow = geo + (size_t)qy * W;
#pragma unroll
        for (int dx = 0; dx < 5; ++dx) {
            const float4 sc = crow[xq[dx]], sgeo = grow[xq[dx]];
            const float sl = luma(sc);
#pragma unroll
            for (int k = 0; k < R; ++k) {
                const int dy = m - k;
                if (dy < 0 || dy > 4) continue;
                const float nd = fmaxf(1.0f - (cg[k].x * sgeo.x + cg[k].y * sgeo.y + cg[k].z * sgeo.z), 0.0f);
                const float e = fabsf(cl[k] - sl) * inv_l[k] + nd * inv_n + fabsf(cg[k].w - sgeo.w) * inv_d;
                const float w = kb[dx] * kb[dy] * __builtin_amdgcn_exp2f(-e);
                sr[k] += sc.x * w;
                sg[k] += sc.y * w;
                sb[k] += sc.z * w;
                ws[k] += w;
                vs[k] += w * w * sc.w;
            }
        }
    }
#pragma unroll
    for (int k = 0; k < R; ++k) {
        const int y = y0 + k * step;
        if (y >= H) break;
        float4 o;
        if (ws[k] > 1e-6f) {
            const float iw = 1.0f / ws[k];
            o = make_float4(sr[k] * iw, sg[k] * iw, sb[k] * iw, vs[k] * iw * iw);
        } else {
            const float4 cc = cvin[(size_t)y * W + x];
            o = make_float4(cc.x, cc.y, cc.z, cvar[k]);
        }
        if (last) o.w = 1.0f;
        cvout[(size_t)y * W + x] = o;
    }
}

template <int R>
void launch_atrous(const float4* ci, const float4* geo, int W, int H, int step, int last, float4* co, hipStream_t s) {
    const int groups = (H + R * step - 1) / (R * step) * step;
    const dim3 grid((W + kBX - 1) / kBX, (groups + kBY - 1) / kBY);
    k_svgf_atrous<R><<<grid, 256, 0, s>>>(ci, geo, W, H, step, last, kSvgfSigmaL, kSvgfSigmaN, kSvgfSigmaD, co);
}

}  // namespace

hipError_t svgf_atrous(const float4* accum, const float4* disp, const float4* aov_albedo,
                       const float4* aov_normal, uint32_t W, uint32_t H, float4* out, void* scratch,
                       hipStream_t s) {
    const uint32_t n = W * H;
    if (n == 0) return hipSuccess;
    float4* c0 = reinterpret_cast<float4*>(scratch);
    float4* geo = c0 + n;
    const dim3 grid((W + kBX - 1) / kBX, (H + kBY - 1) / kBY);
    k_svgf_prep<<<grid, 256, 0, s>>>(accum, disp, aov_albedo, aov_normal, (int)W, (int)H, c0, geo);
    // ping-pong c0 -> out -> c0 -> out -> c0 -> out: the odd count of 5 ends in `out`
    static_assert(kSvgfIterations % 2 == 1, "the ping-pong below ends in `out` for an odd count");
    // Four pixels per thread leave small images with too few waves and a longer chain per
    // thread: whole filter with one / four, 320x200 46 / 78 us, 512x512 73 / 79 us,
    // 800x600 123 / 117 us, 1920x1080 390 / 301 us.
    const bool wide = n >= 400000;
    for (int it = 0; it < kSvgfIterations; ++it) {
        const float4* ci = (it % 2 == 0) ? c0 : out;
        float4* co = (it % 2 == 0) ? out : c0;
        const int last = it == kSvgfIterations - 1 ? 1 : 0;
        if (wide) launch_atrous<4>(ci, geo, (int)W, (int)H, 1 << it, last, co, s);
        else launch_atrous<1>(ci, geo, (int)W, (int)H, 1 << it, last, co, s);
    }
    return hipGetLastError();
}

size_t svgf_scratch_bytes(uint32_t W, uint32_t H) { return (size_t)W * H * 32; }

}  // namespace ohpt
