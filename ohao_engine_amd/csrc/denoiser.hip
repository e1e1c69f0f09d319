// Learned kernel-predicting denoiser (include/ohpt.h, "learned denoiser").
//
// Network: 5-level U-Net over NHWC bfloat16 activations.
//   encoder  x0(16) -> a0,e0(32) -pool-> a1,e1(64) -pool-> a2,e2(96) -pool-> a3,e3(128) -pool-> a4,e4(160)
//   decoder  up(e4)|e3 -> b3,d3(128) ; up(d3)|e2 -> b2,d2(96) ; up(d2)|e1 -> b1,d1(64) ; up(d1)|e0 -> b0,d0(32)
//   head     d0 -> 25 logits (FP32) -> softmax -> 5x5 filter applied to the noisy radiance
// Every 3x3 convolution (forward, input gradient and weight gradient) is an
// implicit GEMM on the gfx950 matrix cores, v_mfma_f32_16x16x32_bf16, FP32
// accumulation; bias + ReLU are fused into the forward epilogue.
//
// Kernel shapes (wave64):
//   k_conv3x3<CC,MX,RW,NC,UPS> one block (RW/2 waves) = (16*MX)xRW output pixels x
//                  32*NC output channels (RW = 16: 8 waves sharing one weight
//                  stage; NC = 2 where the layer has a multiple of 64).
//                  Per input-channel chunk of CC channels the (16*MX+2)x(RW+2)
//                  input halo and the chunk's packed weights are staged in
//                  LDS; each wave owns two rows of 16*MX pixels x 32 channels
//                  (2*MX x 2 MFMA tiles, each weight fragment used 2*MX times)
//                  and walks K = 9 taps x CC channels in steps of 32; the bf16
//                  result is transposed through LDS so each output pixel's 32
//                  channels are written as four 16-byte stores.
//   k_wgrad<CC>    (256 threads) one block = (pixel-tile range, 32 output channels, CC
//                  input channels) and all nine taps; K = pixels, 32 per MFMA step,
//                  split over the block's waves; per-block partial sums go to a buffer
//                  that a fixed-order reduction sums (deterministic weight gradients).
//   k_conv_dma     k_conv3x3's tiling for the layers without an upsampled or
//                  feature input, each chunk's halo and weights staged by
//                  global->LDS loads into a second pair of LDS buffers while the
//                  previous chunk's MFMAs run; k_conv_ring is its persistent form.
//   k_conv_stream, k_conv_features: the full-resolution layers of inference.
// The input gradient reuses these kernels with the weights flipped and transposed.
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "ohpt_internal.h"

using namespace ohpt;

namespace {

#define DNCHK(x)                                             \
    do {                                                     \
        hipError_t e_ = (x);                                 \
        if (e_ != hipSuccess) return set_hip_error(#x, e_); \
    } while (0)

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------- bf16 helpers
// Round to nearest even (gfx950 v_cvt_pk_bf16_f32); a NaN stays a quiet NaN.
__device__ inline uint16_t f2bf(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }
__device__ inline float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

__device__ inline bf16x8 as_bf16x8(uint4 v) { return __builtin_bit_cast(bf16x8, v); }

inline uint32_t cdiv(uint64_t a, uint64_t b) { return (uint32_t)((a + b - 1) / b); }

// Bilinear source taps of output coordinate X for a x2 upsample of n samples
// (half-pixel centres, clamped at the low edge and the high edge).
__device__ inline void up_taps(int X, int n, int& i0, int& i1, float& l1) {
    const float s = fmaxf(0.5f * ((float)X + 0.5f) - 0.5f, 0.0f);
    i0 = (int)s;
    i1 = i0 + (i0 < n - 1 ? 1 : 0);
    l1 = s - (float)i0;
}

// One linear interpolation step of the x2 upsample, (1 - l) * a + l * b, with
// every product and sum rounded on its own (no fused multiply-add), so the
// separable form in the convolution's halo load rounds like the direct one.
__device__ inline float up_lerp(float a, float b, float l) {
    return __fadd_rn(__fmul_rn(1.0f - l, a), __fmul_rn(l, b));
}

// Eight bf16 channels of output pixel (Y, X) of the x2 bilinear upsample of an
// h x w NHWC image (`base` points at the image's first pixel, channel offset
// applied, `cs` channels per pixel): the horizontal interpolation of both
// source rows, then the vertical one. k_up_fwd stores it; the convolution's
// halo load computes the same values separably.
__device__ inline uint4 up8(const uint16_t* base, int Y, int X, int h, int w, int cs) {
    int y0, y1, x0, x1;
    float ly, lx;
    up_taps(Y, h, y0, y1, ly);
    up_taps(X, w, x0, x1, lx);
    const uint4 q00 = *reinterpret_cast<const uint4*>(base + ((size_t)y0 * w + x0) * cs);
    const uint4 q01 = *reinterpret_cast<const uint4*>(base + ((size_t)y0 * w + x1) * cs);
    const uint4 q10 = *reinterpret_cast<const uint4*>(base + ((size_t)y1 * w + x0) * cs);
    const uint4 q11 = *reinterpret_cast<const uint4*>(base + ((size_t)y1 * w + x1) * cs);
    uint4 o;
    uint16_t* oe = reinterpret_cast<uint16_t*>(&o);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const float top = up_lerp(bf2f(reinterpret_cast<const uint16_t*>(&q00)[e]),
                                  bf2f(reinterpret_cast<const uint16_t*>(&q01)[e]), lx);
        const float bot = up_lerp(bf2f(reinterpret_cast<const uint16_t*>(&q10)[e]),
                                  bf2f(reinterpret_cast<const uint16_t*>(&q11)[e]), lx);
        oe[e] = f2bf(up_lerp(top, bot, ly));
    }
    return o;
}

// Guide images (FP32, W x H per image) at padded pixel (y, x) -> the network's
// 16 input features, edge replication beyond the image: log1p radiance (3),
// albedo (3), normal (3), log1p depth (1), zeros (6). half = 0 gives features
// 0-7, half = 1 features 8-15, as eight bf16.
struct FeatureSrc {
    const float4* rad;
    const float4* alb;   // may be null (zeros), as nrm and dep
    const float4* nrm;
    const float* dep;
    int H, W;            // image size (the padded size is the convolution's)
};

// The guide values one features8 call needs (loaded by feat_load, converted by
// feat_mix; split so a caller can issue the loads early and convert later).
struct Feat8 {
    float4 r, a, n;   // half 0: radiance, albedo, normal; half 1: normal in n, depth in r.x
};

__device__ inline Feat8 feat_load(const FeatureSrc& f, int b, int y, int x, int half) {
    const size_t s = ((size_t)b * f.H + min(y, f.H - 1)) * f.W + min(x, f.W - 1);
    Feat8 q;
    q.n = f.nrm ? f.nrm[s] : make_float4(0, 0, 0, 0);
    if (half == 0) {
        q.r = f.rad[s];
        q.a = f.alb ? f.alb[s] : make_float4(0, 0, 0, 0);
    } else {
        q.r = make_float4(f.dep ? f.dep[s] : 0.0f, 0, 0, 0);
        q.a = make_float4(0, 0, 0, 0);
    }
    return q;
}

__device__ inline uint4 feat_mix(const FeatureSrc& f, const Feat8& q, int half) {
    float v[8];
    if (half == 0) {
        v[0] = log1pf(fmaxf(q.r.x, 0.0f));
        v[1] = log1pf(fmaxf(q.r.y, 0.0f));
        v[2] = log1pf(fmaxf(q.r.z, 0.0f));
        v[3] = q.a.x; v[4] = q.a.y; v[5] = q.a.z;
        v[6] = q.n.x; v[7] = q.n.y;
    } else {
        v[0] = q.n.z;
        v[1] = f.dep ? log1pf(fmaxf(q.r.x, 0.0f)) : 0.0f;
#pragma unroll
        for (int k = 2; k < 8; ++k) v[k] = 0.0f;
    }
    uint4 o;
    uint16_t* oe = reinterpret_cast<uint16_t*>(&o);
#pragma unroll
    for (int k = 0; k < 8; ++k) oe[k] = f2bf(v[k]);
    return o;
}

__device__ inline uint4 features8(const FeatureSrc& f, int b, int y, int x, int half) {
    return feat_mix(f, feat_load(f, b, y, x, half), half);
}

// Max of each bf16 element over four vectors, the first maximum kept in scan
// order (the pooled value is one of the inputs, bit for bit).
__device__ inline uint4 max4_bf16(const uint4 q[4]) {
    uint4 o;
    uint16_t* oe = reinterpret_cast<uint16_t*>(&o);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        uint16_t best = reinterpret_cast<const uint16_t*>(&q[0])[e];
        float bv = bf2f(best);
#pragma unroll
        for (int k = 1; k < 4; ++k) {
            const uint16_t cand = reinterpret_cast<const uint16_t*>(&q[k])[e];
            if (bf2f(cand) > bv) { bv = bf2f(cand); best = cand; }
        }
        oe[e] = best;
    }
    return o;
}

// Kernel prediction at image pixel (y, x) of image b (H x W, RGBA32F radiance):
// softmax of the 25 logits lg[0..24], 5x5 filter of the radiance (edge
// clamped). s receives the weights, rk the 25 radiance samples (k_kpn keeps
// them for the backward pass; k_conv_stream's inference head splits the taps
// over four lanes, another summation order).
__device__ inline float3 kpn_apply(const float* lg, const float4* __restrict__ rad, int b, int y, int x, int H, int W,
                                   float s[25], float3 rk[25]) {
    float mx = lg[0];
#pragma unroll
    for (int k = 1; k < 25; ++k) mx = fmaxf(mx, lg[k]);
    float z = 0.0f;
#pragma unroll
    for (int k = 0; k < 25; ++k) { s[k] = expf(lg[k] - mx); z += s[k]; }
    const float iz = 1.0f / z;
    float3 o = make_float3(0, 0, 0);
#pragma unroll
    for (int k = 0; k < 25; ++k) {
        s[k] *= iz;
        const int yy = min(max(y + k / 5 - 2, 0), H - 1), xx = min(max(x + k % 5 - 2, 0), W - 1);
        const float4 r = rad[((size_t)b * H + yy) * W + xx];
        rk[k] = make_float3(r.x, r.y, r.z);
        o.x += s[k] * r.x; o.y += s[k] * r.y; o.z += s[k] * r.z;
    }
    return o;
}

// ------------------------------------------------------------- 3x3 convolution
struct ConvArgs {
    const uint16_t* in0;   // NHWC, c0 channels
    const uint16_t* in1;   // NHWC, c1 channels (second half of a concatenation) or null
    int c0, c1;
    const uint16_t* wp;    // packed weights [cin/CC][KS][np][32]
    int np;                // output channels, multiple of 32
    const float* bias;     // [nb] or null
    int nb;
    uint16_t* out0;        // channels [0, oc0) with row stride oc0
    uint16_t* out1;        // channels [oc0, oc0+oc1) with row stride oc1
    int oc0, oc1;
    float* outf;           // FP32 output with np channels (replaces out0/out1)
    int relu;
    // input gradient: out0 is zeroed where this tensor (its layout) is not positive, or null
    const uint16_t* mask0;
    int B, H, W;
    // in0 is the (H/2) x (W/2) image whose x2 bilinear upsample is the input
    // (the upsample is computed in the halo load instead of being stored)
    int up0;
    // with a bf16 output: also write its 2x2 max-pool, (H/2) x (W/2) x np
    uint16_t* pool_out;
    // feat.rad != null: the input is the 16 features of these guide images,
    // computed in the halo load (c0 = 16, CC = 16)
    FeatureSrc feat;
    // head layer in inference (k_conv_stream, np = 32): instead of storing the
    // logits, apply the kernel prediction to kpn_rad (img_H x img_W images) and
    // write the filtered radiance to kpn_out
    const float4* kpn_rad;
    float4* kpn_out;
    int img_H, img_W;
    // k_conv_stream: 16x16 tiles per image row / column, tiles per block
    int tiles_x, tiles_y, per_block;
};

// 16-byte vector slot of logical vector v of halo pixel p (CC channels per pixel):
// unpadded halo rows with the vectors XOR-swizzled by the pixel index, so a
// 16-lane fragment read spreads over the LDS banks
template <int CC>
__device__ inline int halo_slot(int p, int v) {
    return CC == 32 ? (v ^ ((p >> 1) & 3)) : (v ^ ((p >> 2) & 1));
}

template <int CC, int MX, int RW, int NC, bool UPS>
__global__ __launch_bounds__(32 * RW) void k_conv3x3(ConvArgs a) {
    constexpr int NT = 32 * RW;              // threads: RW / 2 waves of two output rows each
    constexpr int NO = 32 * NC;              // output channels per block
    constexpr int KS = (9 * CC + 31) / 32;   // K steps of 32 per input chunk
    // LDS strides (bf16 elements): halo pixels and weight rows unpadded, their
    // 16-byte vectors XOR-swizzled by the pixel / row (halo_slot), so fragment
    // reads spread over the banks and the 32-channel blocks fit four per CU
    constexpr int XS = CC;                   // halo pixel stride
    constexpr int WS = 32;                   // weight row stride
    constexpr int VPP = CC / 8;              // 16-byte vectors per halo pixel
    constexpr int TX = 16 * MX;              // output pixels per block row
    constexpr int HX = TX + 2;               // halo row length
    constexpr int HP = HX * (RW + 2);        // halo pixels
    __shared__ __align__(16) uint16_t xs[HP * XS];
    __shared__ __align__(16) uint16_t ws[KS * NO * WS];
    // UPS (layers whose first input is upsampled): the horizontal interpolation of the
    // SR source rows the halo reads
    constexpr int SR = RW / 2 + 2;
    __shared__ __align__(16) float hs[UPS ? SR * HX * VPP * 8 : 4];
    static_assert(!UPS || CC == 32, "upsampled inputs come in 32-channel chunks");

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int g = lane >> 4, r16 = lane & 15;
    const int ncout = a.np / NO;
    const int b = blockIdx.z / ncout, nc = blockIdx.z - b * ncout;
    const int x0 = blockIdx.x * TX, y0 = blockIdx.y * RW;
    const int nchunk = (a.c0 + a.c1) / CC;

    // this wave: rows 2*wave, 2*wave+1; MX 16-pixel tiles per row; 2*NC tiles of 16 output channels
    f32x4 acc[2][MX][2 * NC];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int m = 0; m < MX; ++m)
#pragma unroll
            for (int j = 0; j < 2 * NC; ++j) acc[i][m][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    for (int c = 0; c < nchunk; ++c) {
        const int cb = c * CC;
        const uint16_t* src;
        int cs, co;
        if (cb < a.c0) { src = a.in0; cs = a.c0; co = cb; }
        else { src = a.in1; cs = a.c1; co = cb - a.c0; }
        __syncthreads();
        {
            // thread -> (halo pixel p, 16-byte vector v); p advances by 256 / VPP per step
            constexpr int PSTEP = NT / VPP, DY = PSTEP / HX, DX = PSTEP - DY * HX;
            const int v = tid % VPP;
            int p = tid / VPP;
            int hy = p / HX, hx = p - hy * HX;
            const bool up = UPS && a.up0 && cb < a.c0;   // uniform per chunk
            const int sh = up ? a.H / 2 : a.H, sw = up ? a.W / 2 : a.W;
            const uint16_t* img = src + (size_t)b * sh * sw * cs + co + v * 8;
            if (UPS && up) {
                // x2 bilinear upsample, separably: the horizontal interpolation of the source
                // rows y0/2 - 1 .. y0/2 + RW/2 once per (row, halo column) into LDS (FP32),
                // then the vertical one per halo pixel; the same rounding as up8
                const int sy0 = y0 / 2 - 1;
                for (int i = tid; i < SR * HX * VPP; i += NT) {   // NT % VPP == 0: i % VPP == v
                    const int hc = (i / VPP) % HX, k = i / (VPP * HX);
                    const int sr = sy0 + k, gx = x0 - 1 + hc;
                    if (sr < 0 || sr >= sh || gx < 0 || gx >= a.W) continue;   // never read
                    int xa, xb;
                    float lx;
                    up_taps(gx, sw, xa, xb, lx);
                    const uint4 qa = *reinterpret_cast<const uint4*>(img + ((size_t)sr * sw + xa) * cs);
                    const uint4 qb = *reinterpret_cast<const uint4*>(img + ((size_t)sr * sw + xb) * cs);
                    float hv[8];
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        hv[e] = up_lerp(bf2f(reinterpret_cast<const uint16_t*>(&qa)[e]),
                                        bf2f(reinterpret_cast<const uint16_t*>(&qb)[e]), lx);
                    float4* hp = reinterpret_cast<float4*>(hs + ((k * HX + hc) * VPP + v) * 8);
                    hp[0] = make_float4(hv[0], hv[1], hv[2], hv[3]);
                    hp[1] = make_float4(hv[4], hv[5], hv[6], hv[7]);
                }
                __syncthreads();   // uniform: the chunk is upsampled for every thread
                for (; p < HP; p += PSTEP) {
                    const int gy = y0 - 1 + hy, gx = x0 - 1 + hx;
                    uint4 val = make_uint4(0u, 0u, 0u, 0u);
                    if (gy >= 0 && gy < a.H && gx >= 0 && gx < a.W) {
                        int ya, yb;
                        float ly;
                        up_taps(gy, sh, ya, yb, ly);
                        const float* ta = hs + (((ya - sy0) * HX + hx) * VPP + v) * 8;
                        const float* tb = hs + (((yb - sy0) * HX + hx) * VPP + v) * 8;
                        uint16_t* oe = reinterpret_cast<uint16_t*>(&val);
#pragma unroll
                        for (int e = 0; e < 8; ++e) oe[e] = f2bf(up_lerp(ta[e], tb[e], ly));
                    }
                    *reinterpret_cast<uint4*>(&xs[p * XS + (halo_slot<CC>(p, v) << 3)]) = val;
                    hy += DY;
                    hx += DX;
                    if (hx >= HX) { hx -= HX; ++hy; }
                }
            } else {
                for (; p < HP; p += PSTEP) {
                    const int gy = y0 - 1 + hy, gx = x0 - 1 + hx;
                    uint4 val = make_uint4(0u, 0u, 0u, 0u);
                    if (gy >= 0 && gy < a.H && gx >= 0 && gx < a.W) {
                        if (CC == 16 && a.feat.rad) val = features8(a.feat, b, gy, gx, v);
                        else val = *reinterpret_cast<const uint4*>(img + ((size_t)gy * a.W + gx) * cs);
                    }
                    *reinterpret_cast<uint4*>(&xs[p * XS + (halo_slot<CC>(p, v) << 3)]) = val;
                    hy += DY;
                    hx += DX;
                    if (hx >= HX) { hx -= HX; ++hy; }
                }
            }
        }
        const uint16_t* wsrc = a.wp + ((size_t)c * KS * a.np + (size_t)nc * NO) * 32;
        for (int i = tid; i < KS * NO * 4; i += NT) {
            const int s = i / (NO * 4), n = (i >> 2) % NO, v = i & 3;
            *reinterpret_cast<uint4*>(&ws[(s * NO + n) * WS + ((v ^ ((n >> 1) & 3)) << 3)]) =
                *reinterpret_cast<const uint4*>(wsrc + ((size_t)s * a.np + n) * 32 + v * 8);
        }
        __syncthreads();
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            const int kf = s * 32 + g * 8;
            const int tap = kf / CC, ci0 = kf - tap * CC;
            const int dy = tap / 3, dx = tap - dy * 3;
            bf16x8 bfr[2 * NC];
#pragma unroll
            for (int ni = 0; ni < 2 * NC; ++ni)
                bfr[ni] = as_bf16x8(
                    *reinterpret_cast<const uint4*>(&ws[(s * NO + ni * 16 + r16) * WS + ((g ^ ((r16 >> 1) & 3)) << 3)]));
#pragma unroll
            for (int mi = 0; mi < 2; ++mi) {
                const int row = wave * 2 + mi;
#pragma unroll
                for (int m = 0; m < MX; ++m) {
                    const int p = (row + dy) * HX + m * 16 + r16 + dx;
                    uint4 v = make_uint4(0u, 0u, 0u, 0u);
                    if (tap < 9) v = *reinterpret_cast<const uint4*>(&xs[p * XS + (halo_slot<CC>(p, ci0 >> 3) << 3)]);
                    const bf16x8 af = as_bf16x8(v);
#pragma unroll
                    for (int ni = 0; ni < 2 * NC; ++ni)
                        acc[mi][m][ni] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, bfr[ni], acc[mi][m][ni], 0, 0, 0);
                }
            }
        }
    }

    // D layout of a 16x16 tile: lane (g, r16), register i -> pixel x = 4g + i, channel r16.
    // FP32 logits are written directly; bf16 activations go through LDS below.
    if (a.outf) {
#pragma unroll
        for (int mi = 0; mi < 2; ++mi) {
            const int y = y0 + wave * 2 + mi;
            if (y >= a.H) continue;
#pragma unroll
            for (int m = 0; m < MX; ++m) {
#pragma unroll
                for (int ni = 0; ni < 2 * NC; ++ni) {
                    const int n = nc * NO + ni * 16 + r16;
                    const float bias = (a.bias && n < a.nb) ? a.bias[n] : 0.0f;
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int x = x0 + m * 16 + g * 4 + i;
                        if (x >= a.W) continue;
                        float v = acc[mi][m][ni][i] + bias;
                        if (a.relu) v = fmaxf(v, 0.0f);
                        const size_t pix = (size_t)(b * a.H + y) * a.W + x;
                        if (a.outf) a.outf[pix * a.np + n] = v;
                        else if (n < a.oc0) a.out0[pix * a.oc0 + n] = f2bf(v);
                        else a.out1[pix * a.oc1 + (n - a.oc0)] = f2bf(v);
                    }
                }
            }
        }
        return;
    }
    // bf16 outputs: transpose the tile through LDS ([pixel][NO channels], padded) so each
    // pixel's channels leave as 16-byte stores
    constexpr int OS = NO + 8;
    constexpr bool kStageInWeights = RW * TX * OS <= KS * NO * WS;
    static_assert(kStageInWeights || RW * TX * OS <= HP * XS, "output staging fits a shared buffer");
    uint16_t* os = kStageInWeights ? ws : xs;
    __syncthreads();
#pragma unroll
    for (int mi = 0; mi < 2; ++mi) {
#pragma unroll
        for (int m = 0; m < MX; ++m) {
#pragma unroll
            for (int ni = 0; ni < 2 * NC; ++ni) {
                const int nl = ni * 16 + r16, n = nc * NO + nl;
                const float bias = (a.bias && n < a.nb) ? a.bias[n] : 0.0f;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    float v = acc[mi][m][ni][i] + bias;
                    if (a.relu) v = fmaxf(v, 0.0f);
                    os[((wave * 2 + mi) * TX + m * 16 + g * 4 + i) * OS + nl] = f2bf(v);
                }
            }
        }
    }
    __syncthreads();
    for (int i = tid; i < RW * TX * 4 * NC; i += NT) {
        const int pl = i / (4 * NC), v = i % (4 * NC);
        const int y = y0 + pl / TX, x = x0 + pl % TX;
        if (y >= a.H || x >= a.W) continue;
        const uint4 val = *reinterpret_cast<const uint4*>(&os[pl * OS + v * 8]);
        const int n = nc * NO + v * 8;
        const size_t pix = (size_t)(b * a.H + y) * a.W + x;
        if (n < a.oc0) *reinterpret_cast<uint4*>(&a.out0[pix * a.oc0 + n]) = val;
        else *reinterpret_cast<uint4*>(&a.out1[pix * a.oc1 + (n - a.oc0)]) = val;
    }
    if (a.pool_out) {
        // 2x2 max-pool of the staged tile (block origins and H, W are even)
        const int h2 = a.H >> 1, w2 = a.W >> 1;
        for (int i = tid; i < (RW / 2) * (TX / 2) * 4 * NC; i += NT) {
            const int pl = i / (4 * NC), v = i % (4 * NC);
            const int py = pl / (TX / 2), px = pl % (TX / 2);
            const int y = (y0 >> 1) + py, x = (x0 >> 1) + px;
            if (y >= h2 || x >= w2) continue;
            uint4 q[4];
#pragma unroll
            for (int k = 0; k < 4; ++k)
                q[k] = *reinterpret_cast<const uint4*>(&os[((2 * py + (k >> 1)) * TX + 2 * px + (k & 1)) * OS + v * 8]);
            const size_t pix = (size_t)(b * h2 + y) * w2 + x;
            *reinterpret_cast<uint4*>(&a.pool_out[pix * a.np + nc * NO + v * 8]) = max4_bf16(q);
        }
    }
}

// ------------------------------------------ shared parts of the persistent convolutions
// Fragments are multiplied with the weights as the first operand, and row r of tile ni
// is output channel 8 (r / 4) + 4 ni + r % 4: lane (g, r16), register i of tile ni then
// is channel 8 g + 4 ni + i of pixel r16, so a lane stores eight channels of its pixel
// as 16 bytes and a row needs no transpose through LDS.
__device__ __forceinline__ int w_row(int ni, int r16) { return (r16 >> 2) * 8 + ni * 4 + (r16 & 3); }
// 16-byte slot of vector v in the LDS row of output channel n: the rows that a fragment
// read takes from one bank group (n % 4 alike) differ in n / 8
__device__ __forceinline__ int w_slot(int n, int v) { return v ^ ((n >> 3) & 3); }

// This lane's biases of the 32 output channels from n0.
__device__ __forceinline__ void load_bias(const ConvArgs& a, int n0, int g, float bias[2][4]) {
#pragma unroll
    for (int ni = 0; ni < 2; ++ni)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int n = n0 + g * 8 + ni * 4 + i;
            bias[ni][i] = (a.bias && n < a.nb) ? a.bias[n] : 0.0f;
        }
}

// A 16x16 tile's image and tile coordinates, advanced tile by tile.
struct Tile { int b, y, x; };
__device__ __forceinline__ Tile tile_at(const ConvArgs& a, int t) {
    const int tpi = a.tiles_x * a.tiles_y, b = t / tpi, r = t - b * tpi, y = r / a.tiles_x;
    return Tile{b, y, r - y * a.tiles_x};
}
__device__ __forceinline__ void advance(const ConvArgs& a, Tile& t) {
    if (++t.x == a.tiles_x) {
        t.x = 0;
        if (++t.y == a.tiles_y) { t.y = 0; ++t.b; }
    }
}

__device__ __forceinline__ uint2 pack4(const float v[4]) {
    return make_uint2((uint32_t)f2bf(v[0]) | (uint32_t)f2bf(v[1]) << 16, (uint32_t)f2bf(v[2]) | (uint32_t)f2bf(v[3]) << 16);
}

// The gradients g of eight channels whose activations y are positive, the others 0. The
// kernel that writes a gradient last masks it: a pass over each tensor took 238 us of a
// 16 x 256^2 training step of 2.75 ms.
__device__ __forceinline__ uint4 relu_masked(uint4 g, uint4 y) {
    uint16_t* ge = reinterpret_cast<uint16_t*>(&g);
    const uint16_t* ye = reinterpret_cast<const uint16_t*>(&y);
#pragma unroll
    for (int k = 0; k < 8; ++k)
        if (!(bf2f(ye[k]) > 0.0f)) ge[k] = 0;
    return g;
}

// Biased (and rectified) values of one pixel's channels n0 + 8 g + 4 ni + i, stored;
// returned as bf16 for the pooling.
__device__ __forceinline__ void store_row(const ConvArgs& a, int b, int y, int x, int n0, int g, const f32x4 acc[2],
                                          const float bias[2][4], uint4& q) {
    float v[2][4];
#pragma unroll
    for (int ni = 0; ni < 2; ++ni)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[ni][i] = acc[ni][i] + bias[ni][i];
            if (a.relu) v[ni][i] = fmaxf(v[ni][i], 0.0f);
        }
    const uint2 lo = pack4(v[0]), hi = pack4(v[1]);
    q = make_uint4(lo.x, lo.y, hi.x, hi.y);
    if (y >= a.H || x >= a.W) return;
    const size_t pix = (size_t)(b * a.H + y) * a.W + x;
    const int n = n0 + g * 8;
    if (a.outf) {
        float4* o = reinterpret_cast<float4*>(&a.outf[pix * a.np + n]);
        o[0] = make_float4(v[0][0], v[0][1], v[0][2], v[0][3]);
        o[1] = make_float4(v[1][0], v[1][1], v[1][2], v[1][3]);
    } else if (n < a.oc0) {
        uint4 o = q;
        if (a.mask0) o = relu_masked(q, *reinterpret_cast<const uint4*>(&a.mask0[pix * a.oc0 + n]));
        *reinterpret_cast<uint4*>(&a.out0[pix * a.oc0 + n]) = o;
    } else {
        *reinterpret_cast<uint4*>(&a.out1[pix * a.oc1 + (n - a.oc0)]) = q;
    }
}

// 2x2 max-pool of two rows' stored values (top, bot: this lane's pixel), by the lanes
// of even pixels; y, x: the pooled pixel. Origins, H and W are even.
__device__ __forceinline__ void store_pooled(const ConvArgs& a, int b, int y, int x, int n0, int g, int r16,
                                             const uint4& top, const uint4& bot) {
    const int h2 = a.H >> 1, w2 = a.W >> 1;
    auto other = [](const uint4& v) {
        return make_uint4((uint32_t)__shfl_xor((int)v.x, 1), (uint32_t)__shfl_xor((int)v.y, 1),
                          (uint32_t)__shfl_xor((int)v.z, 1), (uint32_t)__shfl_xor((int)v.w, 1));
    };
    const uint4 q[4] = {top, other(top), bot, other(bot)};
    if ((r16 & 1) || y >= h2 || x >= w2) return;
    *reinterpret_cast<uint4*>(&a.pool_out[((size_t)(b * h2 + y) * w2 + x) * a.np + n0 + g * 8]) = max4_bf16(q);
}

// One 32-channel input chunk for a wave's two output rows (from halo row row0) of 16
// pixels x 32 output channels: a fragment of an input row serves both output rows that
// it lies under, 12 + 18 LDS reads for 36 MFMAs. Per accumulator the taps run in
// order (dy, then dx).
__device__ __forceinline__ void conv_rows(const uint16_t* xs, const uint16_t* ws, int row0, int g, int r16,
                                          f32x4 acc[2][2]) {
    constexpr int HX = 18;
    bf16x8 w[9][2];
#pragma unroll
    for (int ry = 0; ry < 4; ++ry) {
        if (ry < 3) {
#pragma unroll
            for (int t = ry * 3; t < ry * 3 + 3; ++t)
#pragma unroll
                for (int ni = 0; ni < 2; ++ni)
                    w[t][ni] = as_bf16x8(*reinterpret_cast<const uint4*>(
                        &ws[(t * 32 + w_row(ni, r16)) * 32 + (w_slot(w_row(ni, r16), g) << 3)]));
        }
#pragma unroll
        for (int dx = 0; dx < 3; ++dx) {
            const int p = (row0 + ry) * HX + r16 + dx;
            const bf16x8 x = as_bf16x8(*reinterpret_cast<const uint4*>(&xs[p * 32 + (halo_slot<32>(p, g) << 3)]));
#pragma unroll
            for (int dy = 0; dy < 3; ++dy) {
                const int r = ry - dy;
                if (r < 0 || r > 1) continue;
#pragma unroll
                for (int ni = 0; ni < 2; ++ni)
                    acc[r][ni] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[dy * 3 + dx][ni], x, acc[r][ni], 0, 0, 0);
            }
        }
    }
}

__device__ __forceinline__ void zero_rows(f32x4 acc[2][2]) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
}

// ------------------------------------- double-buffered convolution (LDS-direct loads)
// Zero vector read by halo slots outside the image (an LDS-direct load cannot write
// zeros of its own).
__device__ __align__(16) uint32_t g_zero_vec[4] = {0u, 0u, 0u, 0u};

// k_conv_dma: k_conv3x3<32, 1, 16, 1, false> with the staging of input chunk
// c + 1 (its 18x18 halo and packed weights) issued as global->LDS loads
// (global_load_lds_dwordx4) into a second pair of LDS buffers before chunk c's
// MFMAs, so the loads' latency hides behind the matrix work instead of
// stalling the block between two barriers. Lane l of wave load i fills the
// 16-byte slot 64 i + l, so each lane fetches the vector that the XOR-swizzled
// layouts of k_conv3x3 keep in that slot. The MFMA order per accumulator
// (chunks, then K steps) and the epilogue are k_conv3x3's: bit-identical outputs.
// kMask: an input gradient with a ReLU mask (a.mask0); the other layers run without its test.
template <bool kMask>
__global__ __launch_bounds__(512) void k_conv_dma(ConvArgs a) {
    constexpr int CC = 32, RW = 16, TX = 16, NT = 512, NO = 32, KS = 9;
    constexpr int HX = TX + 2, HP = HX * (RW + 2);   // 18 x 18 halo pixels
    constexpr int HSLOT = HP * 4;                    // 16-byte halo slots
    constexpr int WSLOT = KS * NO * 4;               // 16-byte weight slots
    constexpr int HI = (HSLOT + 63) / 64, WI = WSLOT / 64;
    constexpr int NW = NT / 64;
    __shared__ __align__(16) uint16_t xa[HP * CC];
    __shared__ __align__(16) uint16_t xb[HP * CC];
    __shared__ __align__(16) uint16_t wa[KS * NO * 32];
    __shared__ __align__(16) uint16_t wb[KS * NO * 32];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int g = lane >> 4, r16 = lane & 15;
    const int ncout = a.np / NO;
    const int b = blockIdx.z / ncout, nc = blockIdx.z - b * ncout;
    const int x0 = blockIdx.x * TX, y0 = blockIdx.y * RW;
    const int nchunk = (a.c0 + a.c1) / CC;

    auto issue = [&](int c, uint16_t* xd, uint16_t* wd) {
        const int cb = c * CC;
        const uint16_t* src;
        int cs, co;
        if (cb < a.c0) { src = a.in0; cs = a.c0; co = cb; }
        else { src = a.in1; cs = a.c1; co = cb - a.c0; }
        const uint16_t* img = src + (size_t)b * a.H * a.W * cs + co;
#pragma unroll
        for (int i = wave; i < HI; i += NW) {
            const int s = i * 64 + lane;
            if (s < HSLOT) {
                const int p = s >> 2, v = (s & 3) ^ ((p >> 1) & 3);
                const int hy = p / HX, hx = p - hy * HX;
                const int gy = y0 - 1 + hy, gx = x0 - 1 + hx;
                const void* gp = g_zero_vec;
                if (gy >= 0 && gy < a.H && gx >= 0 && gx < a.W) gp = img + ((size_t)gy * a.W + gx) * cs + v * 8;
                __builtin_amdgcn_global_load_lds(gp, xd + i * 64 * 8, 16, 0, 0);
            }
        }
        const uint16_t* wsrc = a.wp + ((size_t)c * KS * a.np + (size_t)nc * NO) * 32;
#pragma unroll
        for (int i = wave; i < WI; i += NW) {
            const int s = i * 64 + lane;
            const int row = s >> 2, st = row / NO, n = row - st * NO;
            const int v = (s & 3) ^ ((n >> 1) & 3);
            __builtin_amdgcn_global_load_lds(wsrc + ((size_t)st * a.np + n) * 32 + v * 8, wd + i * 64 * 8, 16, 0, 0);
        }
    };

    f32x4 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    auto compute = [&](const uint16_t* xsb, const uint16_t* wsb) {
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            const int dy = s / 3, dx = s - dy * 3;   // 32-channel chunks: one tap per K step
            bf16x8 bfr[2];
#pragma unroll
            for (int ni = 0; ni < 2; ++ni)
                bfr[ni] = as_bf16x8(
                    *reinterpret_cast<const uint4*>(&wsb[(s * NO + ni * 16 + r16) * 32 + ((g ^ ((r16 >> 1) & 3)) << 3)]));
#pragma unroll
            for (int mi = 0; mi < 2; ++mi) {
                const int p = (wave * 2 + mi + dy) * HX + r16 + dx;
                const bf16x8 af = as_bf16x8(*reinterpret_cast<const uint4*>(&xsb[p * CC + ((g ^ ((p >> 1) & 3)) << 3)]));
#pragma unroll
                for (int ni = 0; ni < 2; ++ni)
                    acc[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, bfr[ni], acc[mi][ni], 0, 0, 0);
            }
        }
    };

    // This wave's LDS-direct loads have landed before it reaches a barrier, so after
    // the barrier the whole buffer is written.
    auto loads_then_barrier = [&]() {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    };

    issue(0, xa, wa);
    int c = 0;
    for (; c + 1 < nchunk; c += 2) {
        loads_then_barrier();          // chunk c in (xa, wa); (xb, wb) no longer read
        issue(c + 1, xb, wb);
        compute(xa, wa);
        loads_then_barrier();          // chunk c + 1 in (xb, wb); (xa, wa) no longer read
        if (c + 2 < nchunk) issue(c + 2, xa, wa);
        compute(xb, wb);
    }
    if (c < nchunk) {
        loads_then_barrier();
        compute(xa, wa);
    }

    if (a.outf) {
#pragma unroll
        for (int mi = 0; mi < 2; ++mi) {
            const int y = y0 + wave * 2 + mi;
            if (y >= a.H) continue;
#pragma unroll
            for (int ni = 0; ni < 2; ++ni) {
                const int n = nc * NO + ni * 16 + r16;
                const float bias = (a.bias && n < a.nb) ? a.bias[n] : 0.0f;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int x = x0 + g * 4 + i;
                    if (x >= a.W) continue;
                    float v = acc[mi][ni][i] + bias;
                    if (a.relu) v = fmaxf(v, 0.0f);
                    const size_t pix = (size_t)(b * a.H + y) * a.W + x;
                    a.outf[pix * a.np + n] = v;
                }
            }
        }
        return;
    }
    // bf16 outputs: the tile transposed through LDS ([pixel][NO channels], padded)
    constexpr int OS = NO + 8;
    static_assert(RW * TX * OS <= HP * CC, "output staging fits its buffer");
    uint16_t* os = xa;
    __syncthreads();
#pragma unroll
    for (int mi = 0; mi < 2; ++mi) {
#pragma unroll
        for (int ni = 0; ni < 2; ++ni) {
            const int nl = ni * 16 + r16, n = nc * NO + nl;
            const float bias = (a.bias && n < a.nb) ? a.bias[n] : 0.0f;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float v = acc[mi][ni][i] + bias;
                if (a.relu) v = fmaxf(v, 0.0f);
                os[((wave * 2 + mi) * TX + g * 4 + i) * OS + nl] = f2bf(v);
            }
        }
    }
    __syncthreads();
    for (int i = tid; i < RW * TX * 4; i += NT) {
        const int pl = i / (4), v = i % (4);
        const int y = y0 + pl / TX, x = x0 + pl % TX;
        if (y >= a.H || x >= a.W) continue;
        uint4 val = *reinterpret_cast<const uint4*>(&os[pl * OS + v * 8]);
        const int n = nc * NO + v * 8;
        const size_t pix = (size_t)(b * a.H + y) * a.W + x;
        if (kMask && n < a.oc0) val = relu_masked(val, *reinterpret_cast<const uint4*>(&a.mask0[pix * a.oc0 + n]));
        if (n < a.oc0) *reinterpret_cast<uint4*>(&a.out0[pix * a.oc0 + n]) = val;
        else *reinterpret_cast<uint4*>(&a.out1[pix * a.oc1 + (n - a.oc0)]) = val;
    }
    if (a.pool_out) {
        const int h2 = a.H >> 1, w2 = a.W >> 1;
        for (int i = tid; i < (RW / 2) * (TX / 2) * 4; i += NT) {
            const int pl = i / (4), v = i % (4);
            const int py = pl / (TX / 2), px = pl % (TX / 2);
            const int y = (y0 >> 1) + py, x = (x0 >> 1) + px;
            if (y >= h2 || x >= w2) continue;
            uint4 q[4];
#pragma unroll
            for (int k = 0; k < 4; ++k)
                q[k] = *reinterpret_cast<const uint4*>(&os[((2 * py + (k >> 1)) * TX + 2 * px + (k & 1)) * OS + v * 8]);
            const size_t pix = (size_t)(b * h2 + y) * w2 + x;
            *reinterpret_cast<uint4*>(&a.pool_out[pix * a.np + nc * NO + v * 8]) = max4_bf16(q);
        }
    }
}

// k_conv_ring: k_conv_dma's tile and staging, persistent: a block keeps its 32 output
// channels and walks a range of tiles, and the (tile, chunk) steps take the two pairs of
// LDS buffers in turn across tile borders, so a layer of one chunk overlaps its loads
// too and a tile's stores drain behind the next step's MFMAs. With one or two chunks
// the weights stay in LDS; halo addresses are kept per lane, border checks only where
// a tile has a border. Bounded by the latency of the halo loads (two blocks per CU,
// 78 KB each) and the LDS reads. 1920x1080 with / without: 32 -> 64 channels at half
// size 34 / 43 us, 64 -> 64 47 / 63 us (817 TFLOP/s), 96 -> 96 at a quarter 28 / 36 us.
// Where a block gets one tile its longer prologue costs 0.5-1.5 us a layer; launch_conv
// says from where on it runs.
__global__ __launch_bounds__(512, 4) void k_conv_ring(ConvArgs a) {
    constexpr int CC = 32, RW = 16, TX = 16, NO = 32, KS = 9;
    constexpr int HX = TX + 2, HP = HX * (RW + 2);   // 18 x 18 halo pixels
    constexpr int HSLOT = HP * 4;                    // 16-byte halo slots
    constexpr int WSLOT = KS * NO * 4;               // 16-byte weight slots
    constexpr int HI = (HSLOT + 63) / 64, WI = WSLOT / 64;
    constexpr int NW = 8;
    __shared__ __align__(16) uint16_t xa[HP * CC];
    __shared__ __align__(16) uint16_t xb[HP * CC];
    __shared__ __align__(16) uint16_t wa[KS * NO * 32];
    __shared__ __align__(16) uint16_t wb[KS * NO * 32];

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, r16 = lane & 15;
    const int ncout = a.np / NO;
    const int nchunk = (a.c0 + a.c1) / CC;
    // XCD-banded order (workgroups are dealt round-robin to the 8 XCDs): the blocks of a
    // tile range, one per 32 output channels, run on one XCD and share its L2
    int lb = blockIdx.x;
    if ((gridDim.x & 7) == 0) lb = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    const int range = lb / ncout, nc = lb - range * ncout;
    const int t_begin = range * a.per_block, t_end = min(t_begin + a.per_block, a.B * a.tiles_x * a.tiles_y);
    if (t_begin >= t_end) return;   // whole block: before any barrier
    const int nsteps = (t_end - t_begin) * nchunk;
    Tile nt = tile_at(a, t_begin);   // tile of the next step to stage

    // where this lane's slots of a halo and of a chunk's weights lie: the same for every tile
    constexpr int HK = (HI + NW - 1) / NW, WK = (WI + NW - 1) / NW;
    int hpix[HK], hyx[HK], woff[WK];   // pixel offset from the halo's corner * 4 + vector; hy << 8 | hx
#pragma unroll
    for (int k = 0; k < HK; ++k) {
        const int s = (wave + k * NW) * 64 + lane, p = s >> 2, v = (s & 3) ^ ((p >> 1) & 3);
        const int hy = p / HX, hx = p - hy * HX;
        hpix[k] = (hy * a.W + hx) * 4 + v;
        hyx[k] = hy << 8 | hx;
    }
#pragma unroll
    for (int k = 0; k < WK; ++k) {
        const int s = (wave + k * NW) * 64 + lane, row = s >> 2, st = row / NO, n = row - st * NO;
        woff[k] = (st * a.np + n) * 32 + w_slot(n, s & 3) * 8;
    }
    Tile ct = nt;           // tile of the computed step
    int nch = 0, cch = 0;   // their chunks
    auto issue = [&](bool weights, uint16_t* xd, uint16_t* wd) __attribute__((always_inline)) {
        const int cb = nch * CC;
        const uint16_t* src;
        int cs, co;
        if (cb < a.c0) { src = a.in0; cs = a.c0; co = cb; }
        else { src = a.in1; cs = a.c1; co = cb - a.c0; }
        const int x0 = nt.x * TX - 1, y0 = nt.y * RW - 1;   // the halo's corner
        const uint16_t* img = src + ((int64_t)nt.b * a.H * a.W + (int64_t)y0 * a.W + x0) * cs + co;
        const bool inside = x0 >= 0 && y0 >= 0 && x0 + HX <= a.W && y0 + RW + 2 <= a.H;
#pragma unroll
        for (int k = 0; k < HK; ++k) {
            const int i = wave + k * NW;
            if (i * 64 + lane >= HSLOT) continue;
            const void* gp = img + ((uint32_t)(hpix[k] >> 2) * (uint32_t)cs + (hpix[k] & 3) * 8);
            if (!inside) {
                const int gy = y0 + (hyx[k] >> 8), gx = x0 + (hyx[k] & 255);
                if (gy < 0 || gy >= a.H || gx < 0 || gx >= a.W) gp = g_zero_vec;
            }
            __builtin_amdgcn_global_load_lds(gp, xd + i * 64 * 8, 16, 0, 0);
        }
        if (weights) {
            const uint16_t* wsrc = a.wp + ((size_t)nch * KS * a.np + (size_t)nc * NO) * 32;
#pragma unroll
            for (int k = 0; k < WK; ++k) {
                const int i = wave + k * NW;
                if (i >= WI) continue;
                const void* wp = wsrc + woff[k];
                __builtin_amdgcn_global_load_lds(wp, wd + i * 64 * 8, 16, 0, 0);
            }
        }
        if (++nch == nchunk) { nch = 0; advance(a, nt); }
    };
    // This wave's LDS-direct loads have landed before it reaches a barrier, so after
    // the barrier the whole buffer is written.
    auto loads_then_barrier = [&]() {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    };

    float bias[2][4];
    f32x4 acc[2][2];
    zero_rows(acc);
    auto step = [&](int j, const uint16_t* xs, const uint16_t* ws, uint16_t* xn, uint16_t* wn)
                    __attribute__((always_inline)) {
        // with one or two chunks each buffer keeps its chunk's weights
        if (j + 1 < nsteps) issue(j == 0 || nchunk > 2, xn, wn);
        conv_rows(xs, ws, wave * 2, g, r16, acc);
        loads_then_barrier();   // step j + 1 staged; (xs, ws) no longer read
        if (++cch == nchunk) {   // the stores drain behind the next step's MFMAs
            const int y = ct.y * RW + wave * 2, x = ct.x * TX + r16;
            uint4 q[2];
#pragma unroll
            for (int r = 0; r < 2; ++r) store_row(a, ct.b, y + r, x, nc * NO, g, acc[r], bias, q[r]);
            if (a.pool_out) store_pooled(a, ct.b, y >> 1, x >> 1, nc * NO, g, r16, q[0], q[1]);
            zero_rows(acc);
            cch = 0;
            advance(a, ct);
        }
    };

    issue(true, xa, wa);
    load_bias(a, nc * NO, g, bias);
    loads_then_barrier();
    int j = 0;
    for (; j + 1 < nsteps; j += 2) {
        step(j, xa, wa, xb, wb);
        step(j + 1, xb, wb, xa, wa);
    }
    if (j < nsteps) step(j, xa, wa, xb, wb);
}

// ------------------------------------------- streaming full-resolution convolution
// LDS writes of this wave are visible to its other lanes after this (no block barrier).
__device__ inline void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// k_conv_stream<EPI>: inference convolutions 32 -> 32 channels on the full-resolution
// 16-aligned grid. Persistent: a block (8 waves, 512 threads) stages the layer's
// packed weights in LDS once and walks a contiguous range of 16x16 output tiles. Each
// tile's 18x18 halo goes to one of two LDS buffers; the global loads of the next tile
// are issued before this tile's MFMAs, so HBM latency hides behind the matrix work
// with one block barrier per tile. Each wave owns two output rows and finishes its
// tile in a private LDS stage (bf16 transpose to 16-byte stores, 2x2 max-pool, or the
// kernel-prediction filter) without a block barrier. Halo pixels and weight rows are
// stored unpadded with their 16-byte vectors XOR-swizzled by the pixel (row) index, so
// a 16-lane fragment read spreads over the banks and two blocks fit per CU. The
// per-accumulator MFMA order is k_conv3x3's, so the outputs are bit-identical to it.
//   EPI 0: bf16 store, 1: + 2x2 max-pool, 2: the head (25 logits) with the kernel
//   prediction applied to a.kpn_rad (the tile's 20x20 radiance window is staged in
//   LDS; four lanes per pixel share the 25 taps).
// The decoder's upsampling layers stay on k_conv3x3 (measured faster there:
// the interpolation registers and three chunks of weights leave one block per CU).
constexpr int kStreamNT = 512;

template <int EPI>
__global__ __launch_bounds__(kStreamNT) void k_conv_stream(ConvArgs a) {
    constexpr int CC = 32, NT = kStreamNT, TX = 16, RW = 16, HX = TX + 2, HP = HX * (RW + 2);
    constexpr int KS = 9;
    constexpr int VPP = CC / 8;
    constexpr int PSTEP = NT / VPP, NPF = (HP + PSTEP - 1) / PSTEP;
    constexpr int XB = HP * CC;                                      // halo buffer (bf16 units)
    constexpr int OS = 40;                                           // staged pixel stride (bf16)
    constexpr int OSW = EPI == 2 ? TX * 25 * 2 : 2 * TX * OS;        // per-wave stage (bf16 units)
    constexpr int WL = KS * 32 * 32;
    __shared__ __align__(16) uint16_t xs[2 * XB];
    __shared__ __align__(16) uint16_t os[(NT / 64) * OSW];
    __shared__ __align__(16) uint16_t ws[WL];
    // head: the tile's 20x20 radiance window (edge-clamped); written after the step's
    // barrier and read after a second one, so one buffer serves (79 KB: two blocks per CU)
    constexpr int RWN = 20 * 20;
    __shared__ __align__(16) float4 rwin[EPI == 2 ? RWN : 1];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int g = lane >> 4, r16 = lane & 15;
    // XCD-banded order: workgroups are dealt round-robin to the 8 XCDs, so logical block
    // k*(n/8)+i runs on XCD k and each XCD's L2 holds one band of adjacent tile ranges
    int lb = blockIdx.x;
    if ((gridDim.x & 7) == 0) lb = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    const int tpi = a.tiles_x * a.tiles_y;
    const int t_begin = lb * a.per_block, t_end = min(t_begin + a.per_block, a.B * tpi);
    if (t_begin >= t_end) return;   // whole block: before any barrier
    const int nsteps = t_end - t_begin;

    // packed weights [step][n][32] -> LDS rows of 32 bf16, vectors swizzled by the row
    for (int i = tid; i < KS * 32 * 4; i += NT) {
        const int sn = i >> 2, v = i & 3;   // sn = step * 32 + output channel
        *reinterpret_cast<uint4*>(&ws[sn * 32 + ((v ^ ((sn >> 1) & 3)) << 3)]) =
            *reinterpret_cast<const uint4*>(a.wp + ((size_t)(sn >> 5) * a.np + (sn & 31)) * 32 + v * 8);
    }
    float bias[2];
#pragma unroll
    for (int ni = 0; ni < 2; ++ni) {
        const int n = ni * 16 + r16;
        bias[ni] = (a.bias && n < a.nb) ? a.bias[n] : 0.0f;
    }

    // halo slots of this thread: pixel tid / VPP + k * PSTEP, 16-byte vector tid % VPP
    const int hv = tid % VPP;
    uint4 pv[NPF];
    uint32_t inb = 0;      // bit k: slot k inside the image
    float4 pr = make_float4(0.f, 0.f, 0.f, 0.f);   // head: this thread's radiance window texel

    auto tile_origin = [&](int t, int& b, int& x0, int& y0) {
        b = t / tpi;
        const int r = t - b * tpi, ty = r / a.tiles_x;
        x0 = (r - ty * a.tiles_x) * TX;
        y0 = ty * RW;
    };
    // issue the global loads of step j
    auto issue = [&](int j) {
        int b, x0, y0;
        tile_origin(t_begin + j, b, x0, y0);
        const uint16_t* img = a.in0 + (size_t)b * a.H * a.W * CC + hv * 8;
        inb = 0;
#pragma unroll
        for (int k = 0; k < NPF; ++k) {
            const int p = tid / VPP + k * PSTEP;
            const int hy = p / HX, hx = p - hy * HX;
            const int gy = y0 - 1 + hy, gx = x0 - 1 + hx;
            const bool in = p < HP && gy >= 0 && gy < a.H && gx >= 0 && gx < a.W;
            inb |= (uint32_t)in << k;
            if (in) pv[k] = *reinterpret_cast<const uint4*>(img + ((size_t)gy * a.W + gx) * CC);
        }
        if constexpr (EPI == 2) {
            if (tid < RWN) {
                const int yy = min(max(y0 - 2 + tid / 20, 0), a.img_H - 1);
                const int xx = min(max(x0 - 2 + tid % 20, 0), a.img_W - 1);
                pr = a.kpn_rad[((size_t)b * a.img_H + yy) * a.img_W + xx];
            }
        }
    };
    auto finish = [&]() {
#pragma unroll
        for (int k = 0; k < NPF; ++k)
            if (!((inb >> k) & 1u)) pv[k] = make_uint4(0u, 0u, 0u, 0u);
    };

    issue(0);
    finish();
    f32x4 acc[2][2];
    for (int j = 0; j < nsteps; ++j) {
        uint16_t* xb = xs + (j & 1) * XB;
#pragma unroll
        for (int k = 0; k < NPF; ++k) {
            const int p = tid / VPP + k * PSTEP;
            if (p < HP) *reinterpret_cast<uint4*>(&xb[p * CC + (halo_slot<CC>(p, hv) << 3)]) = pv[k];
        }
        __syncthreads();   // halo j (and, at j = 0, the weights) complete; step j - 1's buffer is free
        if constexpr (EPI == 2) {
            // every wave has finished step j - 1's filter: the window of tile j replaces it
            if (tid < RWN) rwin[tid] = pr;
        }
        if (j + 1 < nsteps) issue(j + 1);
        zero_rows(acc);
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            const int dy = s / 3, dx = s - dy * 3;
            bf16x8 bfr[2];
#pragma unroll
            for (int ni = 0; ni < 2; ++ni)
                bfr[ni] = as_bf16x8(*reinterpret_cast<const uint4*>(
                    &ws[(s * 32 + ni * 16 + r16) * 32 + ((g ^ ((r16 >> 1) & 3)) << 3)]));
#pragma unroll
            for (int mi = 0; mi < 2; ++mi) {
                const int p = (wave * 2 + mi + dy) * HX + r16 + dx;
                const bf16x8 af = as_bf16x8(*reinterpret_cast<const uint4*>(&xb[p * CC + (halo_slot<CC>(p, g) << 3)]));
#pragma unroll
                for (int ni = 0; ni < 2; ++ni)
                    acc[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, bfr[ni], acc[mi][ni], 0, 0, 0);
            }
        }
        {
            int b, x0, y0;
            tile_origin(t_begin + j, b, x0, y0);
            uint16_t* st = os + wave * OSW;
            if constexpr (EPI == 2) {
                // one row at a time: its 16 pixels' 25 logits through this wave's LDS stage,
                // then four lanes per pixel (taps 0-6, 7-12, 13-18, 19-24) take the softmax and
                // filter the radiance window, combined by cross-lane sums
                __syncthreads();   // the radiance window of this tile is complete
                float* lg = reinterpret_cast<float*>(st);
                const int px = lane & 15, qt = lane >> 4;
                const int k0 = qt == 0 ? 0 : 1 + 6 * qt, nk = qt == 0 ? 7 : 6;
#pragma unroll
                for (int mi = 0; mi < 2; ++mi) {
#pragma unroll
                    for (int ni = 0; ni < 2; ++ni) {
                        const int n = ni * 16 + r16;
                        if (n >= 25) continue;
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            float v = acc[mi][ni][i] + bias[ni];
                            if (a.relu) v = fmaxf(v, 0.0f);
                            lg[(g * 4 + i) * 25 + n] = v;
                        }
                    }
                    wave_lds_sync();
                    const float* lp = lg + px * 25 + k0;
                    float e[7];
                    float mx = -INFINITY;
#pragma unroll
                    for (int k = 0; k < 7; ++k) {
                        e[k] = k < nk ? lp[k] : -INFINITY;
                        mx = fmaxf(mx, e[k]);
                    }
                    mx = fmaxf(mx, __shfl_xor(mx, 16));
                    mx = fmaxf(mx, __shfl_xor(mx, 32));
                    float z = 0.0f;
#pragma unroll
                    for (int k = 0; k < 7; ++k) {
                        e[k] = k < nk ? expf(e[k] - mx) : 0.0f;
                        z += e[k];
                    }
                    z += __shfl_xor(z, 16);
                    z += __shfl_xor(z, 32);
                    const float iz = 1.0f / z;
                    const float4* win = rwin + (wave * 2 + mi) * 20 + px;
                    float ox = 0.0f, oy = 0.0f, oz = 0.0f;
#pragma unroll
                    for (int k = 0; k < 7; ++k) {
                        if (k < nk) {
                            const int t = k0 + k;
                            const float4 r = win[(t / 5) * 20 + t % 5];
                            const float w = e[k] * iz;
                            ox += w * r.x; oy += w * r.y; oz += w * r.z;
                        }
                    }
                    ox += __shfl_xor(ox, 16);
                    oy += __shfl_xor(oy, 16);
                    oz += __shfl_xor(oz, 16);
                    ox += __shfl_xor(ox, 32);
                    oy += __shfl_xor(oy, 32);
                    oz += __shfl_xor(oz, 32);
                    const int y = y0 + wave * 2 + mi, x = x0 + px;
                    if (qt == 0 && y < a.img_H && x < a.img_W)
                        a.kpn_out[((size_t)b * a.img_H + y) * a.img_W + x] = make_float4(ox, oy, oz, 1.0f);
                    wave_lds_sync();   // this row's logits are read before the next row's replace them
                }
            } else {
#pragma unroll
                for (int mi = 0; mi < 2; ++mi)
#pragma unroll
                    for (int ni = 0; ni < 2; ++ni)
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            float v = acc[mi][ni][i] + bias[ni];
                            if (a.relu) v = fmaxf(v, 0.0f);
                            st[(mi * TX + g * 4 + i) * OS + ni * 16 + r16] = f2bf(v);
                        }
                wave_lds_sync();
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    const int idx = lane + 64 * k, pl = idx >> 2, v = idx & 3;
                    const int y = y0 + wave * 2 + pl / TX, x = x0 + pl % TX;
                    if (y < a.H && x < a.W) {
                        const size_t pix = (size_t)(b * a.H + y) * a.W + x;
                        *reinterpret_cast<uint4*>(&a.out0[pix * a.oc0 + v * 8]) =
                            *reinterpret_cast<const uint4*>(&st[pl * OS + v * 8]);
                    }
                }
                if constexpr (EPI == 1) {
                    // 2x2 max-pool of the wave's two rows (origins and H, W are even)
                    if (lane < TX * 2) {
                        const int px = lane >> 2, v = lane & 3;
                        const int h2 = a.H >> 1, w2 = a.W >> 1;
                        const int y = (y0 >> 1) + wave, x = (x0 >> 1) + px;
                        if (y < h2 && x < w2) {
                            uint4 q[4];
#pragma unroll
                            for (int k = 0; k < 4; ++k)
                                q[k] = *reinterpret_cast<const uint4*>(&st[((k >> 1) * TX + 2 * px + (k & 1)) * OS + v * 8]);
                            const size_t pix = (size_t)(b * h2 + y) * w2 + x;
                            *reinterpret_cast<uint4*>(&a.pool_out[pix * a.np + v * 8]) = max4_bf16(q);
                        }
                    }
                }
            }
        }
        if (j + 1 < nsteps) finish();
    }
}

// The input layer of inference: k_conv_stream's persistent form over the 16 guide
// features. A thread loads the guides of one halo pixel and converts all of them (a
// thread per half pixel made every wave run both halves, twice), the fragments are
// multiplied as in conv_rows. 1920x1080: 118 -> 97 us; HBM 45 us (273 MB).
__global__ __launch_bounds__(kStreamNT, 4) void k_conv_features(ConvArgs a) {
    constexpr int CC = 16, NT = kStreamNT, HX = 18, HP = HX * 18, KS = 5;
    __shared__ __align__(16) uint16_t xs[2 * HP * CC];
    __shared__ __align__(16) uint16_t ws[KS * 32 * 32];
    static_assert(NT >= HP, "a halo pixel per thread");

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int g = lane >> 4, r16 = lane & 15;
    int lb = blockIdx.x;   // XCD-banded order, as k_conv_stream
    if ((gridDim.x & 7) == 0) lb = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    const int t_begin = lb * a.per_block, t_end = min(t_begin + a.per_block, a.B * a.tiles_x * a.tiles_y);
    if (t_begin >= t_end) return;   // whole block: before any barrier
    const int nsteps = t_end - t_begin;

    for (int i = tid; i < KS * 32 * 4; i += NT) {
        const int sn = i >> 2, v = i & 3;   // sn = step * 32 + output channel
        *reinterpret_cast<uint4*>(&ws[sn * 32 + (w_slot(sn & 31, v) << 3)]) =
            *reinterpret_cast<const uint4*>(a.wp + ((size_t)(sn >> 5) * a.np + (sn & 31)) * 32 + v * 8);
    }
    float bias[2][4];
    load_bias(a, 0, g, bias);

    const int hy = tid / HX, hx = tid - hy * HX;   // this thread's halo pixel
    float4 fr, fa, fn;                             // its guides
    float fd = 0.0f;
    bool in = false;                               // inside the image
    Tile nt = tile_at(a, t_begin), ct = nt;        // the next tile to load, the computed one
    auto issue = [&]() {
        const int gy = nt.y * 16 - 1 + hy, gx = nt.x * 16 - 1 + hx;
        in = tid < HP && gy >= 0 && gy < a.H && gx >= 0 && gx < a.W;
        if (in) {
            const size_t q = ((size_t)nt.b * a.feat.H + min(gy, a.feat.H - 1)) * a.feat.W + min(gx, a.feat.W - 1);
            fr = a.feat.rad[q];
            fa = a.feat.alb ? a.feat.alb[q] : make_float4(0, 0, 0, 0);
            fn = a.feat.nrm ? a.feat.nrm[q] : make_float4(0, 0, 0, 0);
            fd = a.feat.dep ? a.feat.dep[q] : 0.0f;
        }
        advance(a, nt);
    };
    auto stage = [&](int buf) {
        if (tid >= HP) return;
        uint16_t* xb = xs + buf * HP * CC;
        uint4 lo = make_uint4(0u, 0u, 0u, 0u), hi = lo;
        if (in) {
            lo = feat_mix(a.feat, Feat8{fr, fa, fn}, 0);
            hi = feat_mix(a.feat, Feat8{make_float4(fd, 0, 0, 0), fa, fn}, 1);
        }
        *reinterpret_cast<uint4*>(&xb[tid * CC + (halo_slot<CC>(tid, 0) << 3)]) = lo;
        *reinterpret_cast<uint4*>(&xb[tid * CC + (halo_slot<CC>(tid, 1) << 3)]) = hi;
    };

    issue();
    stage(0);
    for (int j = 0; j < nsteps; ++j) {
        const uint16_t* xb = xs + (j & 1) * HP * CC;
        __syncthreads();   // tile j staged; the other buffer is no longer read
        if (j + 1 < nsteps) issue();
        f32x4 acc[2][2];
        zero_rows(acc);
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            bf16x8 w[2];
#pragma unroll
            for (int ni = 0; ni < 2; ++ni)
                w[ni] = as_bf16x8(*reinterpret_cast<const uint4*>(
                    &ws[(s * 32 + w_row(ni, r16)) * 32 + (w_slot(w_row(ni, r16), g) << 3)]));
            const int tap = s * 2 + (g >> 1), dy = tap / 3, dx = tap - dy * 3;   // two taps per K step
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                const int p = (wave * 2 + r + dy) * HX + r16 + dx;
                uint4 v = make_uint4(0u, 0u, 0u, 0u);
                if (tap < 9) v = *reinterpret_cast<const uint4*>(&xb[p * CC + (halo_slot<CC>(p, g & 1) << 3)]);
#pragma unroll
                for (int ni = 0; ni < 2; ++ni)
                    acc[r][ni] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[ni], as_bf16x8(v), acc[r][ni], 0, 0, 0);
            }
        }
        uint4 q;
#pragma unroll
        for (int r = 0; r < 2; ++r)
            store_row(a, ct.b, ct.y * 16 + wave * 2 + r, ct.x * 16 + r16, 0, g, acc[r], bias, q);
        advance(a, ct);
        if (j + 1 < nsteps) stage((j + 1) & 1);
    }
}

// ------------------------------------------------- weight gradient (split-K)
struct WgradArgs {
    const uint16_t* in0;
    const uint16_t* in1;
    int c0, c1;
    const uint16_t* g;     // masked output gradient, NHWC with np channels
    int np;
    float* part;           // [nsplit][cin/CC][tap][np][CC]
    float* bpart;          // [nsplit][np]
    int B, H, W, nsplit, per_split, tiles_x, tiles_y;
};

typedef short s16x4 __attribute__((ext_vector_type(4)));

// Transposing LDS read (ds_read_b64_tr_b16): within each group of 16 lanes, lane
// i receives element i & 3 of the 8 bytes addressed by lanes i / 4, 4 + i / 4,
// 8 + i / 4 and 12 + i / 4. Lane l addressing channels 4 (l & 3).. of pixel
// (l & 15) / 4 thus yields channel l & 15 of four consecutive pixels.
__device__ inline uint2 lds_read_tr(const uint16_t* p) {
    return __builtin_bit_cast(
        uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)p));
}

// dW[tap][ci][co] = sum over pixels of X[pixel + tap][ci] G[pixel][co]: K is the
// pixels, 32 (two rows of 16) per MFMA step. A block of four waves owns 32 output
// channels x CC input channels x nine taps over a range of 16x16 tiles and each
// wave takes two of a tile's eight K steps, so every wave accumulates all nine
// taps and a fragment of G serves nine taps, a fragment of X all output channels.
// X's halo and G lie in LDS as in memory (pixel rows of CC / 32 channels) and are
// read transposed; three reads of a row give its eight pixels at dx = 0, 1 and 2
// (the middle one by 16-bit alignment in registers), 22 reads for 36 MFMAs.
// Tiles are staged by global->LDS loads into the other of two buffers while the
// MFMAs of this one run; 79 KB, two blocks per CU. Vectors of the right half of
// a row are swapped in pairs so that the two 8-pixel runs a read touches fall on
// different banks. The four waves' sums are added in wave order through LDS, the
// splits' in split order by k_wgrad_reduce: bit-reproducible.
// Bounded by HBM at full resolution (both tensors read once: 134 MB for 32 -> 32
// channels at 16 x 256^2), by staging and the MFMAs' LDS reads below. The 19 layers
// of a 16 x 256^2 step: 1.72 ms with 16-bit gathers from LDS (eight reads per MFMA and
// one 16x16 tile per wave) -> 0.69 ms, 427 TFLOP/s.
template <int CC>
__global__ __launch_bounds__(256, 2) void k_wgrad(WgradArgs a) {
    constexpr int CI = CC / 16;              // 16-channel tiles of X
    constexpr int VPP = CC / 8;              // 16-byte vectors per halo pixel
    constexpr int HXP = 20, HY = 18;         // halo row pitch (18 used) and rows
    constexpr int XSLOT = HXP * HY * VPP, GSLOT = 256 * 4;
    __shared__ __align__(16) uint16_t xa[XSLOT * 8];
    __shared__ __align__(16) uint16_t xb[XSLOT * 8];
    __shared__ __align__(16) uint16_t ga[GSLOT * 8];
    __shared__ __align__(16) uint16_t gb[GSLOT * 8];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int g = lane >> 4, r16 = lane & 15;
    const int nchunk = (a.c0 + a.c1) / CC, combos = nchunk * (a.np / 32);
    // the blocks that share a split's tiles run on one XCD (workgroups are dealt
    // round-robin to the 8 XCDs) and find them in its L2
    const int slot = blockIdx.x >> 3;
    const int split = (blockIdx.x & 7) + 8 * (slot / combos), combo = slot % combos;
    if (split >= a.nsplit) return;   // whole block
    const int c = combo % nchunk, nc = combo / nchunk;
    const int tpi = a.tiles_y * a.tiles_x;
    const int t0 = split * a.per_split, t1 = min(a.B * tpi, t0 + a.per_split);

    const int cb = c * CC;
    const uint16_t* src;
    int cs, co;
    if (cb < a.c0) { src = a.in0; cs = a.c0; co = cb; }
    else { src = a.in1; cs = a.c1; co = cb - a.c0; }

    // LDS-direct loads of tile t: lane l of load i fills 16-byte slot 64 i + l
    auto issue = [&](int t, uint16_t* xd, uint16_t* gd) {
        const int b = t / tpi, r = t - b * tpi;
        const int ty = r / a.tiles_x, x0 = (r - ty * a.tiles_x) * 16, y0 = ty * 16;
        const uint16_t* img = src + (size_t)b * a.H * a.W * cs + co;
#pragma unroll
        for (int i = wave; i < (XSLOT + 63) / 64; i += 4) {
            const int s = i * 64 + lane;
            if (s < XSLOT) {
                const int p = s / VPP, hy = p / HXP, hx = p - hy * HXP;
                const int v = (s % VPP) ^ (CC == 32 ? ((hx >> 3) & 1) << 1 : 0);
                const int gy = y0 - 1 + hy, gx = x0 - 1 + hx;
                const void* gp = g_zero_vec;
                if (hx < 18 && gy >= 0 && gy < a.H && gx >= 0 && gx < a.W)
                    gp = img + ((size_t)gy * a.W + gx) * cs + v * 8;
                __builtin_amdgcn_global_load_lds(gp, xd + i * 64 * 8, 16, 0, 0);
            }
        }
        const uint16_t* gimg = a.g + (size_t)b * a.H * a.W * a.np + nc * 32;
#pragma unroll
        for (int i = wave; i < GSLOT / 64; i += 4) {
            const int s = i * 64 + lane, p = s >> 2;
            const int v = (s & 3) ^ (((p >> 3) & 1) << 1);
            const int gy = y0 + (p >> 4), gx = x0 + (p & 15);
            const void* gp = g_zero_vec;
            if (gy < a.H && gx < a.W) gp = gimg + ((size_t)gy * a.W + gx) * a.np + v * 8;
            __builtin_amdgcn_global_load_lds(gp, gd + i * 64 * 8, 16, 0, 0);
        }
    };

    f32x4 acc[9][CI][2], bacc[2];
#pragma unroll
    for (int t = 0; t < 9; ++t)
#pragma unroll
        for (int m = 0; m < CI; ++m)
#pragma unroll
            for (int n = 0; n < 2; ++n) acc[t][m][n] = f32x4{0.f, 0.f, 0.f, 0.f};
    bacc[0] = bacc[1] = f32x4{0.f, 0.f, 0.f, 0.f};
    const bf16x8 ones = as_bf16x8(make_uint4(0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u));

    // this lane's part of a transposing read: pixel (r16 / 4) of a run, channels
    // 4 (r16 & 3).. of the first 16; bf16 offsets from the run's first pixel, for a
    // run in the row's left (parity g & 1 = 0) or right half, of tile m
    const int px = 8 * (g & 1) + (r16 >> 2);
    const int half = (r16 & 3) >> 1, sub = (r16 & 1) * 4;
    int xo[CI], go[2];
#pragma unroll
    for (int m = 0; m < CI; ++m)
        xo[m] = ((g >> 1) * HXP + px) * CC + (((2 * m + half) ^ (CC == 32 ? (g & 1) << 1 : 0)) << 3) + sub;
#pragma unroll
    for (int n = 0; n < 2; ++n) go[n] = ((g >> 1) * 16 + px) * 32 + (((2 * n + half) ^ ((g & 1) << 1)) << 3) + sub;

    auto compute = [&](const uint16_t* xs, const uint16_t* gs) {
#pragma unroll 1
        for (int k = 0; k < 2; ++k) {
            const int row = 2 * (wave * 2 + k);   // K step: rows row, row + 1
            bf16x8 bf[2];
#pragma unroll
            for (int n = 0; n < 2; ++n) {
                const uint16_t* p = gs + row * 16 * 32 + go[n];
                const uint2 lo = lds_read_tr(p), hi = lds_read_tr(p + 4 * 32);
                bf[n] = as_bf16x8(make_uint4(lo.x, lo.y, hi.x, hi.y));
            }
            if (c == 0) {
#pragma unroll
                for (int n = 0; n < 2; ++n) bacc[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, bf[n], bacc[n], 0, 0, 0);
            }
#pragma unroll
            for (int dy = 0; dy < 3; ++dy) {
#pragma unroll
                for (int m = 0; m < CI; ++m) {
                    const uint16_t* p = xs + (row + dy) * HXP * CC;
                    // pixels 8.. of the run lie in the other half: the pair's other order
                    const uint2 q0 = lds_read_tr(p + xo[m]), q1 = lds_read_tr(p + xo[m] + 4 * CC),
                                q2 = lds_read_tr(p + xo[CC == 32 ? m ^ 1 : m] + 8 * CC);
                    const bf16x8 f0 = as_bf16x8(make_uint4(q0.x, q0.y, q1.x, q1.y));
                    const bf16x8 f1 = as_bf16x8(make_uint4(
                        __builtin_amdgcn_alignbit(q0.y, q0.x, 16), __builtin_amdgcn_alignbit(q1.x, q0.y, 16),
                        __builtin_amdgcn_alignbit(q1.y, q1.x, 16), __builtin_amdgcn_alignbit(q2.x, q1.y, 16)));
                    const bf16x8 f2 = as_bf16x8(make_uint4(q0.y, q1.x, q1.y, q2.x));
#pragma unroll
                    for (int n = 0; n < 2; ++n) {
                        acc[dy * 3 + 0][m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f0, bf[n], acc[dy * 3 + 0][m][n], 0, 0, 0);
                        acc[dy * 3 + 1][m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f1, bf[n], acc[dy * 3 + 1][m][n], 0, 0, 0);
                        acc[dy * 3 + 2][m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f2, bf[n], acc[dy * 3 + 2][m][n], 0, 0, 0);
                    }
                }
            }
        }
    };
    auto loads_then_barrier = [&]() {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    };

    issue(t0, xa, ga);
    int t = t0;
    for (; t + 1 < t1; t += 2) {
        loads_then_barrier();          // tile t in (xa, ga); (xb, gb) no longer read
        issue(t + 1, xb, gb);
        compute(xa, ga);
        loads_then_barrier();          // tile t + 1 in (xb, gb); (xa, ga) no longer read
        if (t + 2 < t1) issue(t + 2, xa, ga);
        compute(xb, gb);
    }
    if (t < t1) {
        loads_then_barrier();
        compute(xa, ga);
    }

    // tile (tap, m, n): lane (g, r16), register i -> input channel 16 m + 4 g + i, output
    // channel 16 n + r16. Per tap, the waves' tiles go to LDS ([wave][n][ci]) and are added
    // in wave order; taps alternate between two buffers, one barrier each.
    __syncthreads();
    float* const out = a.part + ((size_t)(split * nchunk + c) * 9 * a.np + nc * 32) * CC;
    if (c == 0 && g == 0) {   // row 0 of the ones product: the sum over this wave's pixels
        float* red = reinterpret_cast<float*>(xa);
#pragma unroll
        for (int n = 0; n < 2; ++n) red[wave * 32 + n * 16 + r16] = bacc[n][0];
    }
#pragma unroll
    for (int tap = 0; tap < 9; ++tap) {
        float* red = reinterpret_cast<float*>((tap & 1) ? gb : ga);
#pragma unroll
        for (int m = 0; m < CI; ++m)
#pragma unroll
            for (int n = 0; n < 2; ++n)
                *reinterpret_cast<f32x4*>(&red[(wave * 32 + n * 16 + r16) * CC + m * 16 + g * 4]) = acc[tap][m][n];
        __syncthreads();
        if (tid < 8 * CC) {
            f32x4 v = *reinterpret_cast<const f32x4*>(&red[tid * 4]);
#pragma unroll
            for (int w = 1; w < 4; ++w) v += *reinterpret_cast<const f32x4*>(&red[w * 32 * CC + tid * 4]);
            *reinterpret_cast<f32x4*>(&out[(size_t)tap * a.np * CC + tid * 4]) = v;
        }
    }
    if (c == 0 && tid < 32) {
        const float* red = reinterpret_cast<const float*>(xa);
        a.bpart[(size_t)split * a.np + nc * 32 + tid] = ((red[tid] + red[32 + tid]) + red[64 + tid]) + red[96 + tid];
    }
}

// Sums the split partials into the logical layout W[tap][cin][cout] followed by
// bias[cout]. A block takes 64 float4 columns of the partials with 16 threads per
// column, each adding every 16th split in order; their sums are added in order
// (bit-reproducible). One thread per weight walking all splits with a stride of a
// whole partial took 4.35 ms of a 16 x 256^2 step (2048 splits on 36 blocks at full
// resolution); this form with the splits cut to two blocks per CU takes 0.12 ms.
__global__ __launch_bounds__(1024) void k_wgrad_reduce(const float* __restrict__ part, const float* __restrict__ bpart,
                                                       float* __restrict__ gw, int nsplit, int nchunk, int CC, int np,
                                                       int cin, int cout) {
    __shared__ float4 red[16][64];
    const int col = threadIdx.x & 63, grp = threadIdx.x >> 6;
    const int ncol = nchunk * 9 * np * CC / 4;   // float4 columns of the weights
    const int e = blockIdx.x * 64 + col;
    float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
    if (e < ncol) {
        const float4* p = reinterpret_cast<const float4*>(part) + e;
#pragma unroll 4
        for (int k = grp; k < nsplit; k += 16) {
            const float4 v = p[(size_t)k * ncol];
            s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
        }
    } else if (e < ncol + np / 4) {
        const float4* p = reinterpret_cast<const float4*>(bpart) + (e - ncol);
        for (int k = grp; k < nsplit; k += 16) {
            const float4 v = p[(size_t)k * (np / 4)];
            s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
        }
    }
    red[grp][col] = s;
    __syncthreads();
    if (grp != 0) return;
    for (int k = 1; k < 16; ++k) {
        const float4 v = red[k][col];
        s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
    }
    const float o[4] = {s.x, s.y, s.z, s.w};
    if (e < ncol) {
        const int q = e * 4, ci = q % CC, n = (q / CC) % np, tap = (q / (CC * np)) % 9, c = q / (CC * np * 9);
        if (n < cout)
            for (int k = 0; k < 4; ++k) gw[((size_t)tap * cin + c * CC + ci + k) * cout + n] = o[k];
    } else if (e < ncol + np / 4) {
        for (int k = 0; k < 4; ++k) {
            const int n = (e - ncol) * 4 + k;
            if (n < cout) gw[(size_t)9 * cin * cout + n] = o[k];
        }
    }
}

// ------------------------------------------------------------- weight packing
// One layer's packed copy: forward, [c][s][n][j] = W[tap][ci][n], K index s*32+j =
// tap*CC + (ci mod CC); or the input gradient's, a forward convolution over the output
// gradient with W'[t][co][ci] = W[8-t][ci][co] in chunks of 32 over cout (padded).
struct PackJob {
    const float* w;
    uint16_t* out;
    int cin, cout, np, cc, ks, dgrad, total, block0;   // np: outputs (forward) or cin; first block
};
constexpr int kMaxPackJobs = 40;
struct PackJobs {
    int n;
    PackJob job[kMaxPackJobs];
};

// All layers' copies in one launch, 34 us; 37 launches of 2 to 3 us each took 114 us of a step.
__global__ __launch_bounds__(256) void k_pack(PackJobs jobs) {
    int k = 0;
    while (k + 1 < jobs.n && (int)blockIdx.x >= jobs.job[k + 1].block0) ++k;   // uniform
    const PackJob& J = jobs.job[k];
    const int idx = ((int)blockIdx.x - J.block0) * 256 + threadIdx.x;
    if (idx >= J.total) return;
    const int j = idx & 31, n = (idx >> 5) % J.np, s = (idx / (32 * J.np)) % J.ks, c = idx / (32 * J.np * J.ks);
    float v = 0.0f;
    if (J.dgrad) {
        const int co = c * 32 + j;
        if (co < J.cout) v = J.w[((size_t)(8 - s) * J.cin + n) * J.cout + co];
    } else {
        const int kf = s * 32 + j, tap = kf / J.cc, ci = c * J.cc + (kf - tap * J.cc);
        if (tap < 9 && n < J.cout && ci < J.cin) v = J.w[((size_t)tap * J.cin + ci) * J.cout + n];
    }
    J.out[idx] = f2bf(v);
}

// ------------------------------------------------------- elementwise kernels
// 2x2 max-pool, H and W even.
__global__ __launch_bounds__(256) void k_pool_fwd(const uint16_t* __restrict__ in, uint16_t* __restrict__ out, int B,
                                                  int H, int W, int C) {
    const int h = H >> 1, w = W >> 1, cv = C >> 3;
    // 32-bit index arithmetic: check_shape bounds B*Hp*Wp by 2^28, so B*h*w*cv < 2^32
    const uint32_t total = (uint32_t)B * h * w * cv;
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= total) return;
    const int v = (int)(i % (uint32_t)cv);
    uint32_t r = i / (uint32_t)cv;
    const int x = (int)(r % (uint32_t)w);
    r /= (uint32_t)w;
    const int y = (int)(r % (uint32_t)h);
    const int b = (int)(r / (uint32_t)h);
    uint4 q[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
        q[k] = *reinterpret_cast<const uint4*>(in + ((size_t)(b * H + 2 * y + (k >> 1)) * W + 2 * x + (k & 1)) * C + v * 8);
    *reinterpret_cast<uint4*>(out + ((size_t)(b * h + y) * w + x) * C + v * 8) = max4_bf16(q);
}

// Routes the pooled gradient to the first maximum of each 2x2 window (scan
// order (0,0),(0,1),(1,0),(1,1)), adds it to gin (the skip's gradient) and zeroes the
// sum where the ReLU output `in` is not positive.
__global__ __launch_bounds__(256) void k_pool_bwd(const uint16_t* __restrict__ in, const uint16_t* __restrict__ gout,
                                                  uint16_t* __restrict__ gin, int B, int H, int W, int C) {
    const int h = H >> 1, w = W >> 1, cv = C >> 3;
    // 32-bit index arithmetic: check_shape bounds B*Hp*Wp by 2^28, so B*h*w*cv < 2^32
    const uint32_t total = (uint32_t)B * h * w * cv;
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= total) return;
    const int v = (int)(i % (uint32_t)cv);
    uint32_t r = i / (uint32_t)cv;
    const int x = (int)(r % (uint32_t)w);
    r /= (uint32_t)w;
    const int y = (int)(r % (uint32_t)h);
    const int b = (int)(r / (uint32_t)h);
    uint4 q[4], gi[4];
    size_t off[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        off[k] = ((size_t)(b * H + 2 * y + (k >> 1)) * W + 2 * x + (k & 1)) * C + v * 8;
        q[k] = *reinterpret_cast<const uint4*>(in + off[k]);
        gi[k] = *reinterpret_cast<const uint4*>(gin + off[k]);
    }
    const uint4 go = *reinterpret_cast<const uint4*>(gout + ((size_t)(b * h + y) * w + x) * C + v * 8);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        int arg = 0;
        float bv = bf2f(reinterpret_cast<const uint16_t*>(&q[0])[e]);
#pragma unroll
        for (int k = 1; k < 4; ++k) {
            const float cv2 = bf2f(reinterpret_cast<const uint16_t*>(&q[k])[e]);
            if (cv2 > bv) { bv = cv2; arg = k; }
        }
        uint16_t* t = reinterpret_cast<uint16_t*>(&gi[arg]);
        t[e] = f2bf(bf2f(t[e]) + bf2f(reinterpret_cast<const uint16_t*>(&go)[e]));
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) *reinterpret_cast<uint4*>(gin + off[k]) = relu_masked(gi[k], q[k]);
}

__global__ __launch_bounds__(256) void k_up_fwd(const uint16_t* __restrict__ in, uint16_t* __restrict__ out, int B,
                                                int h, int w, int C) {
    const int H = 2 * h, W = 2 * w, cv = C >> 3;
    // 32-bit index arithmetic: check_shape bounds B*Hp*Wp by 2^28, so B*H*W*cv < 2^32
    const uint32_t total = (uint32_t)B * H * W * cv;
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= total) return;
    const int v = (int)(i % (uint32_t)cv);
    uint32_t r = i / (uint32_t)cv;
    const int X = (int)(r % (uint32_t)W);
    r /= (uint32_t)W;
    const int Y = (int)(r % (uint32_t)H);
    const int b = (int)(r / (uint32_t)H);
    *reinterpret_cast<uint4*>(out + ((size_t)(b * H + Y) * W + X) * C + v * 8) =
        up8(in + (size_t)b * h * w * C + v * 8, Y, X, h, w, C);
}

// Weight with which input sample i contributes to output coordinate X.
__device__ inline float up_weight(int X, int n, int i) {
    int i0, i1;
    float l1;
    up_taps(X, n, i0, i1, l1);
    return (i0 == i ? 1.0f - l1 : 0.0f) + (i1 == i ? l1 : 0.0f);
}

// Transpose of k_up_fwd in gather form (each input sample sums the output
// samples that read it, fixed order), zeroed where the ReLU output `in` is not positive.
__global__ __launch_bounds__(256) void k_up_bwd(const uint16_t* __restrict__ gout, const uint16_t* __restrict__ in,
                                                uint16_t* __restrict__ gin, int B, int h, int w, int C) {
    const int H = 2 * h, W = 2 * w, cv = C >> 3;
    // 32-bit index arithmetic: check_shape bounds B*Hp*Wp by 2^28, so B*h*w*cv < 2^32
    const uint32_t total = (uint32_t)B * h * w * cv;
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= total) return;
    const int v = (int)(i % (uint32_t)cv);
    uint32_t r = i / (uint32_t)cv;
    const int x = (int)(r % (uint32_t)w);
    r /= (uint32_t)w;
    const int y = (int)(r % (uint32_t)h);
    const int b = (int)(r / (uint32_t)h);
    float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int Y = max(0, 2 * y - 2); Y <= min(H - 1, 2 * y + 2); ++Y) {
        const float wy = up_weight(Y, h, y);
        if (wy == 0.0f) continue;
        for (int X = max(0, 2 * x - 2); X <= min(W - 1, 2 * x + 2); ++X) {
            const float wx = up_weight(X, w, x);
            if (wx == 0.0f) continue;
            const uint4 q = *reinterpret_cast<const uint4*>(gout + ((size_t)(b * H + Y) * W + X) * C + v * 8);
            const float wgt = wy * wx;
#pragma unroll
            for (int e = 0; e < 8; ++e) acc[e] += wgt * bf2f(reinterpret_cast<const uint16_t*>(&q)[e]);
        }
    }
    uint4 o;
    uint16_t* oe = reinterpret_cast<uint16_t*>(&o);
#pragma unroll
    for (int e = 0; e < 8; ++e) oe[e] = f2bf(acc[e]);
    const size_t at = ((size_t)(b * h + y) * w + x) * C + v * 8;
    *reinterpret_cast<uint4*>(gin + at) = relu_masked(o, *reinterpret_cast<const uint4*>(in + at));
}

// Guide images -> 16-channel bf16 input at padded size (edge replication):
// log1p radiance (3), albedo (3), normal (3), log1p depth (1), zeros (6).
__global__ __launch_bounds__(256) void k_features(const float4* __restrict__ rad, const float4* __restrict__ alb,
                                                  const float4* __restrict__ nrm, const float* __restrict__ dep,
                                                  uint16_t* __restrict__ x0, int B, int H, int W, int Hp, int Wp) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;   // B*Hp*Wp <= 2^28 (check_shape)
    const uint32_t total = (uint32_t)B * Hp * Wp;
    if (i >= total) return;
    const int x = (int)(i % (uint32_t)Wp);
    const int y = (int)((i / (uint32_t)Wp) % (uint32_t)Hp);
    const int b = (int)(i / ((uint32_t)Wp * Hp));
    const FeatureSrc f{rad, alb, nrm, dep, H, W};
    reinterpret_cast<uint4*>(x0)[(size_t)i * 2] = features8(f, b, y, x, 0);
    reinterpret_cast<uint4*>(x0)[(size_t)i * 2 + 1] = features8(f, b, y, x, 1);
}

// Tonemap of the training loss: T(x) = (ACES(0.5 x) + 1e-3)^(1/2.2), ACES
// clamped to [0, 1]; returns T and dT/dx.
__device__ inline float tonemap_loss(float x, float& dT) {
    const float u = 0.5f * fmaxf(x, 0.0f);
    const float num = u * (2.51f * u + 0.03f);
    const float den = u * (2.43f * u + 0.59f) + 0.14f;
    float f = num / den;
    float df = 0.0f;
    if (x > 0.0f && f < 1.0f) {
        const float dnum = 5.02f * u + 0.03f, dden = 4.86f * u + 0.59f;
        df = 0.5f * (dnum * den - num * dden) / (den * den);
    }
    f = fminf(fmaxf(f, 0.0f), 1.0f);
    const float p = powf(f + 1e-3f, 1.0f / 2.2f);
    dT = df * (1.0f / 2.2f) * p / (f + 1e-3f);
    return p;
}

struct KpnArgs {
    const float* logits;   // [B][Hp][Wp][32]
    const float4* rad;     // [B][H][W]
    const float4* target;  // [B][H][W] or null
    float4* out;           // [B][H][W] or null
    uint16_t* dlogits;     // [B][Hp][Wp][32] or null
    float* loss_part;      // [gridDim.x] or null
    int B, H, W, Hp, Wp;
    float inv_count;       // 1 / (B*H*W*3)
};

// Softmax over the 25 logits, filter of the noisy radiance (edge-clamped
// 5x5 window), and for training the L1 tonemapped loss with its gradient.
__global__ __launch_bounds__(256) void k_kpn(KpnArgs a) {
    __shared__ float red[256];
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;   // B*Hp*Wp <= 2^28 (check_shape)
    const uint32_t total = (uint32_t)a.B * a.Hp * a.Wp;
    float lsum = 0.0f;
    if (i < total) {
        const int x = (int)(i % (uint32_t)a.Wp);
        const int y = (int)((i / (uint32_t)a.Wp) % (uint32_t)a.Hp);
        const int b = (int)(i / ((uint32_t)a.Wp * a.Hp));
        if (y < a.H && x < a.W) {
            float s[25];
            float3 rk[25];
            const float3 o = kpn_apply(a.logits + (size_t)i * 32, a.rad, b, y, x, a.H, a.W, s, rk);
            const size_t pix = ((size_t)b * a.H + y) * a.W + x;
            if (a.out) a.out[pix] = make_float4(o.x, o.y, o.z, 1.0f);
            if (a.target) {
                const float4 t = a.target[pix];
                float d0, d1, d2, dd;
                const float e0 = tonemap_loss(o.x, d0) - tonemap_loss(t.x, dd);
                const float e1 = tonemap_loss(o.y, d1) - tonemap_loss(t.y, dd);
                const float e2 = tonemap_loss(o.z, d2) - tonemap_loss(t.z, dd);
                lsum = fabsf(e0) + fabsf(e1) + fabsf(e2);
                const float g0 = (e0 > 0.0f ? 1.0f : (e0 < 0.0f ? -1.0f : 0.0f)) * d0 * a.inv_count;
                const float g1 = (e1 > 0.0f ? 1.0f : (e1 < 0.0f ? -1.0f : 0.0f)) * d1 * a.inv_count;
                const float g2 = (e2 > 0.0f ? 1.0f : (e2 < 0.0f ? -1.0f : 0.0f)) * d2 * a.inv_count;
                if (a.dlogits) {
                    uint16_t dl[32];
#pragma unroll
                    for (int k = 0; k < 25; ++k)
                        dl[k] = f2bf(s[k] * (g0 * (rk[k].x - o.x) + g1 * (rk[k].y - o.y) + g2 * (rk[k].z - o.z)));
#pragma unroll
                    for (int k = 25; k < 32; ++k) dl[k] = 0;
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        reinterpret_cast<uint4*>(a.dlogits + (size_t)i * 32)[v] = reinterpret_cast<const uint4*>(dl)[v];
                }
            }
        } else if (a.dlogits) {
#pragma unroll
            for (int v = 0; v < 4; ++v) reinterpret_cast<uint4*>(a.dlogits + (size_t)i * 32)[v] = make_uint4(0u, 0u, 0u, 0u);
        }
    }
    if (a.loss_part) {
        red[threadIdx.x] = lsum;
        __syncthreads();
        for (int o = 128; o > 0; o >>= 1) {
            if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
            __syncthreads();
        }
        if (threadIdx.x == 0) a.loss_part[blockIdx.x] = red[0];
    }
}

__global__ __launch_bounds__(256) void k_sum_serial(const float* __restrict__ in, int n, float scale,
                                                    float* __restrict__ out) {
    __shared__ float red[256];
    float s = 0.0f;
    for (int i = threadIdx.x; i < n; i += 256) s += in[i];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[0] = red[0] * scale;
}

__global__ __launch_bounds__(256) void k_adam(float* __restrict__ p, const float* __restrict__ g,
                                              float* __restrict__ m, float* __restrict__ v, size_t n, float lr,
                                              float b1, float b2, float eps, float bc1, float bc2) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= (lr / bc1) * mi / (sqrtf(vi) / sqrtf(bc2) + eps);
}

__global__ __launch_bounds__(256) void k_bf16_to_f32(const uint16_t* __restrict__ in, float* __restrict__ out,
                                                     size_t n) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) out[i] = bf2f(in[i]);
}

// ------------------------------------------------------------- network tables
enum : int { X0, A0, E0, P1, A1, E1, P2, A2, E2, P3, A3, E3, P4, A4, E4,
             U3, B3, D3, U2, B2, D2, U1, B1, D1, U0, B0, D0, kNumAct };
constexpr int kLogits = kNumAct;   // tensor index of the head logits
constexpr int kActLevel[kNumAct] = {0, 0, 0, 1, 1, 1, 2, 2, 2, 3, 3, 3, 4, 4, 4,
                                    3, 3, 3, 2, 2, 2, 1, 1, 1, 0, 0, 0};
constexpr int kActChan[kNumAct] = {16, 32, 32, 32, 64, 64, 64, 96, 96, 96, 128, 128, 128, 160, 160,
                                   160, 128, 128, 128, 96, 96, 96, 64, 64, 64, 32, 32};
struct LayerSpec { int in0, in1, out, cout, relu; };
constexpr int kNumLayers = 19;
constexpr LayerSpec kLayers[kNumLayers] = {
    {X0, -1, A0, 32, 1},  {A0, -1, E0, 32, 1},   {P1, -1, A1, 64, 1},   {A1, -1, E1, 64, 1},
    {P2, -1, A2, 96, 1},  {A2, -1, E2, 96, 1},   {P3, -1, A3, 128, 1},  {A3, -1, E3, 128, 1},
    {P4, -1, A4, 160, 1}, {A4, -1, E4, 160, 1},  {U3, E3, B3, 128, 1},  {B3, -1, D3, 128, 1},
    {U2, E2, B2, 96, 1},  {B2, -1, D2, 96, 1},   {U1, E1, B1, 64, 1},   {B1, -1, D1, 64, 1},
    {U0, E0, B0, 32, 1},  {B0, -1, D0, 32, 1},   {D0, -1, kLogits, 25, 0}};
constexpr int kInputChannels = 10;   // real channels of X0 (the rest are zero padding)

struct Layer {
    LayerSpec sp;
    int cin0, cin1, cin, cout, np, cc, ks, nchunk;
    size_t w_off, b_off;   // offsets into the FP32 parameter vector
    DevBuf wf, wd;         // packed bf16 weights: forward, input gradient
};

}  // namespace

struct ohpt_denoiser {
    int device = 0;
    int num_cus = 256;     // compute units (persistent convolution grids)
    hipStream_t stream = nullptr;
    std::vector<Layer> layers;
    size_t nparam = 0;
    DevBuf params, grads, adam_m, adam_v;
    int adam_t = 0;
    bool have_grads = false;
    bool profile = false;

    size_t cap_px = 0;     // level-0 pixel capacity (batch * Hp * Wp)
    int B = 0, H = 0, W = 0, Hp = 0, Wp = 0;   // shape of the last call
    DevBuf act[kNumAct], gact[kNumAct];
    DevBuf logits, dlogits;
    DevBuf wpart, bpart, loss_part, loss_dev;
    DevBuf in_rad, in_alb, in_nrm, in_dep, in_tgt, out_stage;

    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    std::vector<hipEvent_t> conv_ev;
    int conv_ev_used = 0;
    ohpt_denoiser_stats stats{};
};

namespace {

int pad16(int v) { return (v + 15) & ~15; }

hipError_t ensure_capacity(ohpt_denoiser* d, int B, int Hp, int Wp) {
    const size_t px = (size_t)B * Hp * Wp;
    if (px <= d->cap_px) return hipSuccess;
    for (int t = 0; t < kNumAct; ++t) {
        const size_t n = (px >> (2 * kActLevel[t])) * kActChan[t] * 2;
        hipError_t e = d->act[t].ensure(n);
        if (e != hipSuccess) return e;
        if (t != X0) {
            e = d->gact[t].ensure(n);
            if (e != hipSuccess) return e;
        }
    }
    hipError_t e = d->logits.ensure(px * 32 * 4);
    if (e == hipSuccess) e = d->dlogits.ensure(px * 32 * 2);
    if (e == hipSuccess) e = d->loss_part.ensure((px / 256 + 1) * 4);
    if (e == hipSuccess) d->cap_px = px;
    return e;
}

// 16-pixel tiles per block row: 1 keeps LDS at 37 KB (4 blocks per CU); wider
// tiles reuse each weight fragment more but fit fewer blocks and measured slower.
constexpr int kConvMX = 1;
constexpr int kConvRows = 16;

// Persistent streaming launch over the 16x16 tiles: as many blocks per compute
// unit as its registers and LDS allow (measured once per kernel), rounded up to
// a multiple of the 8 XCDs.
template <class K>
void launch_stream(ohpt_denoiser* d, ConvArgs a, K kernel, int& per_cu) {
    if (per_cu <= 0 &&
        (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, kStreamNT, 0) != hipSuccess || per_cu <= 0))
        per_cu = 1;
    const int n_tiles = a.B * a.tiles_x * a.tiles_y;
    const int max_blocks = std::max(8, per_cu * d->num_cus);
    a.per_block = (int)cdiv(n_tiles, max_blocks);
    const int nb = ((int)cdiv(n_tiles, a.per_block) + 7) & ~7;
    kernel<<<nb, kStreamNT, 0, d->stream>>>(a);
}

void launch_conv(ohpt_denoiser* d, const Layer& L, const ConvArgs& a, int cc) {
    // 16 output rows per block for 32-channel chunks (measured best of 8/16/24/32 at
    // 1080p); the 16-channel input layer keeps 8, where the output staging would not fit.
    // Upsampling layers with a multiple of 64 output channels cover 64 per block (one
    // halo stage feeds twice the MFMA work; measured 2 % faster per inference than 32).
    const int rows = cc == 16 ? 8 : kConvRows;
    const int no = cc == 16 ? 32 : (a.np % 64 == 0 && !a.outf ? 64 : 32);
    dim3 grid(cdiv(a.W, 16 * kConvMX), cdiv(a.H, rows), (uint32_t)(a.B * (a.np / no)));
    hipEvent_t e0 = nullptr, e1 = nullptr;
    if (d->profile) {
        if ((int)d->conv_ev.size() < d->conv_ev_used + 2) {
            hipEvent_t x, y;
            (void)hipEventCreate(&x);
            (void)hipEventCreate(&y);
            d->conv_ev.push_back(x);
            d->conv_ev.push_back(y);
        }
        e0 = d->conv_ev[d->conv_ev_used];
        e1 = d->conv_ev[d->conv_ev_used + 1];
        d->conv_ev_used += 2;
        (void)hipEventRecord(e0, d->stream);
    }
    if (a.tiles_x > 0) {
        static int per_cu[4] = {};
        if (cc == 16) launch_stream(d, a, k_conv_features, per_cu[3]);
        else if (a.kpn_out) launch_stream(d, a, k_conv_stream<2>, per_cu[2]);
        else if (a.pool_out) launch_stream(d, a, k_conv_stream<1>, per_cu[1]);
        else launch_stream(d, a, k_conv_stream<0>, per_cu[0]);
    } else if (cc == 16) k_conv3x3<16, kConvMX, 8, 1, false><<<grid, 256, 0, d->stream>>>(a);
    else if (!a.up0) {
        // 32 output channels per block: two blocks per CU (78 KB of LDS each); more than two
        // tiles and channel groups for each: the persistent form with the resident blocks over
        // equal ranges. Kernel times (us) tile per block (k_conv_dma) / persistent, 64 -> 96 and
        // 96 -> 96 channels: 1.1 times the resident blocks 13.0 / 14.0 and 17.5 / 19.7, 1.5 times
        // 14.9 / 15.2 and 19.7 / 20.6, 2.0 times (342 tiles) 20.8 / 19.5 and 28.8 / 28.8, 3.0
        // times (510) 26.2 / 20.0 and 36.3 / 28.3, 5.6 times (960) 44.3 / 36.4 and 61.1 / 49.4.
        // Persistent with a tile per block lies between them (24.2 and 32.3 at 510), also where
        // equal ranges leave blocks idle (512 tiles: four each on 384 of 512 blocks, 23.0 and
        // 33.9; a tile per block 24.7 and 33.2).
        ConvArgs p = a;
        p.tiles_x = (int)cdiv(a.W, 16);
        p.tiles_y = (int)cdiv(a.H, 16);
        const int ncout = a.np / 32, n_tiles = a.B * p.tiles_x * p.tiles_y;
        const int64_t slots = 2ll * d->num_cus, work = (int64_t)n_tiles * ncout;
        if (work <= 2 * slots) {
            grid.z = (uint32_t)(a.B * ncout);
            if (a.mask0) k_conv_dma<true><<<grid, 512, 0, d->stream>>>(a);
            else k_conv_dma<false><<<grid, 512, 0, d->stream>>>(a);
        } else {
            p.per_block = (int)cdiv(n_tiles, (uint64_t)std::max<int64_t>(1, slots / ncout));
            k_conv_ring<<<(cdiv(n_tiles, p.per_block) * ncout + 7u) & ~7u, 512, 0, d->stream>>>(p);
        }
    }
    else if (no == 64 && a.up0) k_conv3x3<32, kConvMX, kConvRows, 2, true><<<grid, 32 * kConvRows, 0, d->stream>>>(a);
    else k_conv3x3<32, kConvMX, kConvRows, 1, true><<<grid, 32 * kConvRows, 0, d->stream>>>(a);
    if (d->profile) (void)hipEventRecord(e1, d->stream);
    (void)L;
}

// Forward of layer L at level lvl. up_src >= 0: the first input is the x2
// upsample of that (half-resolution) tensor, computed in the halo load.
// pool_dst >= 0: the epilogue also writes the 2x2 max-pool of the output there.
struct KpnTarget { const float4* rad; float4* out; int H, W; };

// stream: inference may use k_conv_stream (full-resolution layers with 32 outputs).
void conv_forward(ohpt_denoiser* d, const Layer& L, int lvl, int up_src = -1, int pool_dst = -1,
                  const FeatureSrc* feat = nullptr, const KpnTarget* kpn = nullptr, bool stream = false) {
    const int H = d->Hp >> lvl, W = d->Wp >> lvl;
    ConvArgs a{};
    if (feat) a.feat = *feat;
    if (kpn) {
        a.kpn_rad = kpn->rad;
        a.kpn_out = kpn->out;
        a.img_H = kpn->H;
        a.img_W = kpn->W;
    }
    a.in0 = d->act[up_src >= 0 ? up_src : L.sp.in0].as<uint16_t>();
    a.up0 = up_src >= 0;
    a.pool_out = pool_dst >= 0 ? d->act[pool_dst].as<uint16_t>() : nullptr;
    a.in1 = L.sp.in1 >= 0 ? d->act[L.sp.in1].as<uint16_t>() : nullptr;
    a.c0 = L.cin0;
    a.c1 = L.cin1;
    a.wp = L.wf.as<uint16_t>();
    a.np = L.np;
    a.bias = d->params.as<float>() + L.b_off;
    a.nb = L.cout;
    if (L.sp.out == kLogits) {
        a.outf = d->logits.as<float>();
    } else {
        a.out0 = d->act[L.sp.out].as<uint16_t>();
        a.oc0 = L.np;
    }
    a.relu = L.sp.relu;
    a.B = d->B;
    a.H = H;
    a.W = W;
    // level 0 is padded to multiples of 16, so the inference head (kpn) always streams
    if ((stream || kpn) && lvl == 0 && L.np == 32 && H % 16 == 0 && W % 16 == 0 && up_src < 0 &&
        ((L.cc == 16 && feat) || (L.cc == 32 && !feat && L.nchunk == 1))) {
        a.tiles_x = W / 16;
        a.tiles_y = H / 16;
    }
    launch_conv(d, L, a, L.cc);
}

// Input gradient of layer L from G (its masked output gradient).
void conv_dgrad(ohpt_denoiser* d, const Layer& L, const uint16_t* G, int lvl) {
    const int H = d->Hp >> lvl, W = d->Wp >> lvl;
    ConvArgs a{};
    a.in0 = G;
    a.c0 = L.np;
    a.c1 = 0;
    a.wp = L.wd.as<uint16_t>();
    a.np = L.cin;
    a.out0 = d->gact[L.sp.in0].as<uint16_t>();
    a.oc0 = L.cin0;
    // pooled and upsampled inputs are no ReLU outputs: what they lead to is masked there
    static constexpr bool kRelu[kNumAct] = {0, 1, 1, 0, 1, 1, 0, 1, 1, 0, 1, 1, 0, 1, 1, 0, 1, 1, 0, 1, 1, 0, 1, 1, 0, 1, 1};
    a.mask0 = kRelu[L.sp.in0] ? d->act[L.sp.in0].as<uint16_t>() : nullptr;
    a.out1 = L.sp.in1 >= 0 ? d->gact[L.sp.in1].as<uint16_t>() : nullptr;
    a.oc1 = L.cin1;
    a.B = d->B;
    a.H = H;
    a.W = W;
    launch_conv(d, L, a, 32);
}

hipError_t conv_wgrad(ohpt_denoiser* d, const Layer& L, const uint16_t* G, int lvl) {
    const int H = d->Hp >> lvl, W = d->Wp >> lvl;
    const int tx = (int)cdiv(W, 16), ty = (int)cdiv(H, 16);
    const int ntiles = d->B * tx * ty;
    // as many splits as give every CU its two blocks; each split's tiles are read once
    // per combination of 32 output and CC input channels
    const int combos = (L.np / 32) * L.nchunk;
    const int per = (int)cdiv(ntiles, std::max(1, 2 * d->num_cus / combos));
    const int nsplit = (int)cdiv(ntiles, per);
    const size_t part_n = (size_t)nsplit * L.nchunk * 9 * L.np * L.cc;
    hipError_t e = d->wpart.ensure(part_n * 4);
    if (e == hipSuccess) e = d->bpart.ensure((size_t)nsplit * L.np * 4);
    if (e != hipSuccess) return e;
    WgradArgs a{};
    a.in0 = d->act[L.sp.in0].as<uint16_t>();
    a.in1 = L.sp.in1 >= 0 ? d->act[L.sp.in1].as<uint16_t>() : nullptr;
    a.c0 = L.cin0;
    a.c1 = L.cin1;
    a.g = G;
    a.np = L.np;
    a.part = d->wpart.as<float>();
    a.bpart = d->bpart.as<float>();
    a.B = d->B;
    a.H = H;
    a.W = W;
    a.nsplit = nsplit;
    a.per_split = per;
    a.tiles_x = tx;
    a.tiles_y = ty;
    const uint32_t grid = 8 * cdiv(nsplit, 8) * combos;
    if (L.cc == 16) k_wgrad<16><<<grid, 256, 0, d->stream>>>(a);
    else k_wgrad<32><<<grid, 256, 0, d->stream>>>(a);
    const int ncol = L.nchunk * 9 * L.np * L.cc / 4 + L.np / 4;
    k_wgrad_reduce<<<cdiv(ncol, 64), 1024, 0, d->stream>>>(a.part, a.bpart, d->grads.as<float>() + L.w_off, nsplit,
                                                           L.nchunk, L.cc, L.np, L.cin, L.cout);
    return hipSuccess;
}

void pool_forward(ohpt_denoiser* d, int src, int dst) {
    const int lvl = kActLevel[src], C = kActChan[src];
    const int H = d->Hp >> lvl, W = d->Wp >> lvl;
    const size_t n = (size_t)d->B * (H / 2) * (W / 2) * (C / 8);
    k_pool_fwd<<<cdiv(n, 256), 256, 0, d->stream>>>(d->act[src].as<uint16_t>(), d->act[dst].as<uint16_t>(), d->B, H,
                                                    W, C);
}

void pool_backward(ohpt_denoiser* d, int src, int dst) {   // dst = pooled tensor, gradient flows into src
    const int lvl = kActLevel[src], C = kActChan[src];
    const int H = d->Hp >> lvl, W = d->Wp >> lvl;
    const size_t n = (size_t)d->B * (H / 2) * (W / 2) * (C / 8);
    k_pool_bwd<<<cdiv(n, 256), 256, 0, d->stream>>>(d->act[src].as<uint16_t>(), d->gact[dst].as<uint16_t>(),
                                                    d->gact[src].as<uint16_t>(), d->B, H, W, C);
}

void up_forward(ohpt_denoiser* d, int src, int dst) {
    const int lvl = kActLevel[src], C = kActChan[src];
    const int h = d->Hp >> lvl, w = d->Wp >> lvl;
    const size_t n = (size_t)d->B * (2 * h) * (2 * w) * (C / 8);
    k_up_fwd<<<cdiv(n, 256), 256, 0, d->stream>>>(d->act[src].as<uint16_t>(), d->act[dst].as<uint16_t>(), d->B, h, w,
                                                  C);
}

void up_backward(ohpt_denoiser* d, int src, int dst) {   // gradient of dst (upsampled) -> src
    const int lvl = kActLevel[src], C = kActChan[src];
    const int h = d->Hp >> lvl, w = d->Wp >> lvl;
    const size_t n = (size_t)d->B * h * w * (C / 8);
    k_up_bwd<<<cdiv(n, 256), 256, 0, d->stream>>>(d->gact[dst].as<uint16_t>(), d->act[src].as<uint16_t>(),
                                                  d->gact[src].as<uint16_t>(), d->B, h, w, C);
}

double conv_flops(const ohpt_denoiser* d, int H, int W, bool training) {
    double f = 0.0;
    for (const Layer& L : d->layers) {
        const int lvl = kActLevel[L.sp.in0];
        const double px = (double)d->B * (double)(H >> lvl) * (double)(W >> lvl);
        const double cin = (L.sp.in0 == X0) ? kInputChannels : (double)L.cin;
        const double fwd = 2.0 * 9.0 * cin * L.cout * px;
        f += fwd;
        if (training) f += fwd + (L.sp.in0 == X0 ? 0.0 : fwd);   // weight gradient + input gradient
    }
    return f;
}

// The encoder's max-pools run in the epilogues of the convolutions that feed
// them. Training stores the upsampled decoder inputs (the weight gradient reads
// them); inference computes them in the decoder convolutions' halo loads.
void network_forward(ohpt_denoiser* d, bool training, const FeatureSrc& feat, float4* kpn_out) {
    const auto& Ls = d->layers;
    // training stores the input features (its weight gradient reads them); inference builds
    // them in the first convolution's halo load
    if (training) {
        const size_t ppx = (size_t)d->B * d->Hp * d->Wp;
        k_features<<<cdiv(ppx, 256), 256, 0, d->stream>>>(feat.rad, feat.alb, feat.nrm, feat.dep,
                                                          d->act[X0].as<uint16_t>(), d->B, feat.H, feat.W, d->Hp,
                                                          d->Wp);
        conv_forward(d, Ls[0], 0);
    } else {
        conv_forward(d, Ls[0], 0, -1, -1, &feat, nullptr, true);
    }
    conv_forward(d, Ls[1], 0, -1, P1, nullptr, nullptr, !training);
    conv_forward(d, Ls[2], 1);
    conv_forward(d, Ls[3], 1, -1, P2);
    conv_forward(d, Ls[4], 2);
    conv_forward(d, Ls[5], 2, -1, P3);
    conv_forward(d, Ls[6], 3);
    conv_forward(d, Ls[7], 3, -1, P4);
    conv_forward(d, Ls[8], 4);
    conv_forward(d, Ls[9], 4);
    static constexpr int kUp[4][4] = {{E4, U3, 10, 3}, {D3, U2, 12, 2}, {D2, U1, 14, 1}, {D1, U0, 16, 0}};
    for (const auto& u : kUp) {
        if (training) {
            up_forward(d, u[0], u[1]);
            conv_forward(d, Ls[u[2]], u[3]);
        } else {
            conv_forward(d, Ls[u[2]], u[3], u[0], -1, nullptr, nullptr, true);
        }
        conv_forward(d, Ls[u[2] + 1], u[3], -1, -1, nullptr, nullptr, !training);
    }
    if (training || !kpn_out) {
        conv_forward(d, Ls[18], 0);   // logits stored; k_kpn applies them
    } else {
        KpnTarget kt{feat.rad, kpn_out, feat.H, feat.W};
        conv_forward(d, Ls[18], 0, -1, -1, nullptr, &kt, true);
    }
}

// Backward of one convolution given the gradient of its output tensor, which the
// kernel that wrote it last has masked by the ReLU (k_up_bwd, k_pool_bwd, conv_dgrad).
hipError_t layer_backward(ohpt_denoiser* d, int li, bool need_input_grad) {
    const Layer& L = d->layers[li];
    const int lvl = kActLevel[L.sp.in0];
    const uint16_t* G;
    if (L.sp.out == kLogits) {
        G = d->dlogits.as<uint16_t>();
    } else {
        G = d->gact[L.sp.out].as<uint16_t>();
    }
    hipError_t e = conv_wgrad(d, L, G, lvl);
    if (e != hipSuccess) return e;
    if (need_input_grad) conv_dgrad(d, L, G, lvl);
    return hipSuccess;
}

hipError_t network_backward(ohpt_denoiser* d) {
    hipError_t e;
#define BW(i) do { e = layer_backward(d, (i), true); if (e != hipSuccess) return e; } while (0)
    BW(18);
    BW(17);
    BW(16);
    up_backward(d, D1, U0);
    BW(15);
    BW(14);
    up_backward(d, D2, U1);
    BW(13);
    BW(12);
    up_backward(d, D3, U2);
    BW(11);
    BW(10);
    up_backward(d, E4, U3);
    BW(9);
    BW(8);
    pool_backward(d, E3, P4);
    BW(7);
    BW(6);
    pool_backward(d, E2, P3);
    BW(5);
    BW(4);
    pool_backward(d, E1, P2);
    BW(3);
    BW(2);
    pool_backward(d, E0, P1);
    BW(1);
#undef BW
    return layer_backward(d, 0, false);
}

hipError_t pack_weights(ohpt_denoiser* d) {
    PackJobs P{};
    static_assert(2 * kNumLayers <= kMaxPackJobs, "a forward and an input-gradient copy per layer");
    int blocks = 0;
    auto add = [&](const Layer& L, uint16_t* out, int np, int cc, int ks, int dgrad, int total) {
        P.job[P.n++] = PackJob{d->params.as<float>() + L.w_off, out, L.cin, L.cout, np, cc, ks, dgrad, total, blocks};
        blocks += (int)cdiv(total, 256);
    };
    for (const Layer& L : d->layers) {
        add(L, L.wf.as<uint16_t>(), L.np, L.cc, L.ks, 0, L.nchunk * L.ks * L.np * 32);
        if (L.sp.in0 != X0) add(L, L.wd.as<uint16_t>(), L.cin, 32, 9, 1, (L.np / 32) * 9 * L.cin * 32);
    }
    k_pack<<<blocks, 256, 0, d->stream>>>(P);
    return hipGetLastError();
}

// Stages the guide images (and target) on the device when given host pointers.
struct Inputs { const float4* rad; const float4* alb; const float4* nrm; const float* dep; const float4* tgt; };

int stage_inputs(ohpt_denoiser* d, const ohpt_denoise_inputs* in, const float* target, size_t npx, int on_device,
                 Inputs& out) {
    if (on_device) {
        out = {reinterpret_cast<const float4*>(in->radiance), reinterpret_cast<const float4*>(in->albedo),
               reinterpret_cast<const float4*>(in->normal), in->depth, reinterpret_cast<const float4*>(target)};
        return OHPT_OK;
    }
    auto up = [&](DevBuf& buf, const void* src, size_t bytes) -> hipError_t {
        hipError_t e = buf.ensure(bytes);
        if (e == hipSuccess) e = hipMemcpyAsync(buf.p, src, bytes, hipMemcpyHostToDevice, d->stream);
        return e;
    };
    out = {};
    DNCHK(up(d->in_rad, in->radiance, npx * 16));
    out.rad = d->in_rad.as<float4>();
    if (in->albedo) { DNCHK(up(d->in_alb, in->albedo, npx * 16)); out.alb = d->in_alb.as<float4>(); }
    if (in->normal) { DNCHK(up(d->in_nrm, in->normal, npx * 16)); out.nrm = d->in_nrm.as<float4>(); }
    if (in->depth) { DNCHK(up(d->in_dep, in->depth, npx * 4)); out.dep = d->in_dep.as<float>(); }
    if (target) { DNCHK(up(d->in_tgt, target, npx * 16)); out.tgt = d->in_tgt.as<float4>(); }
    return OHPT_OK;
}

int check_shape(ohpt_denoiser* d, const ohpt_denoise_inputs* in, uint32_t batch, uint32_t width, uint32_t height) {
    if (!d || !in || !in->radiance) return set_error(OHPT_ERR_INVALID_ARG, "denoiser: null argument");
    if (batch == 0 || width == 0 || height == 0 || batch > 1024 || width > 16384 || height > 16384)
        return set_error(OHPT_ERR_INVALID_ARG, "denoiser: bad image size");
    if ((uint64_t)batch * pad16((int)width) * pad16((int)height) > (1ull << 28))
        return set_error(OHPT_ERR_INVALID_ARG, "denoiser: batch too large");
    return OHPT_OK;
}

// Forward of the network; in inference (kpn_out != null) the head convolution
// also applies the kernel prediction and writes the denoised radiance.
int run_forward(ohpt_denoiser* d, const Inputs& x, uint32_t batch, uint32_t width, uint32_t height,
                bool training, float4* kpn_out = nullptr) {
    d->B = (int)batch;
    d->H = (int)height;
    d->W = (int)width;
    d->Hp = pad16((int)height);
    d->Wp = pad16((int)width);
    DNCHK(ensure_capacity(d, d->B, d->Hp, d->Wp));
    network_forward(d, training, FeatureSrc{x.rad, x.alb, x.nrm, x.dep, d->H, d->W}, kpn_out);
    DNCHK(hipGetLastError());
    return OHPT_OK;
}

void begin_timing(ohpt_denoiser* d) {
    d->conv_ev_used = 0;
    (void)hipEventRecord(d->ev0, d->stream);
}

int end_timing(ohpt_denoiser* d, bool training) {
    DNCHK(hipEventRecord(d->ev1, d->stream));
    DNCHK(hipEventSynchronize(d->ev1));
    float ms = 0.0f;
    DNCHK(hipEventElapsedTime(&ms, d->ev0, d->ev1));
    d->stats.ms_total = ms;
    float conv = 0.0f;
    for (int i = 0; i + 1 < d->conv_ev_used; i += 2) {
        float m = 0.0f;
        if (hipEventElapsedTime(&m, d->conv_ev[i], d->conv_ev[i + 1]) == hipSuccess) conv += m;
    }
    d->stats.ms_conv = conv;
    d->stats.conv_flops = conv_flops(d, d->H, d->W, training);
    d->stats.padded_width = (uint32_t)d->Wp;
    d->stats.padded_height = (uint32_t)d->Hp;
    d->stats.batch = (uint32_t)d->B;
    return OHPT_OK;
}

// Seeded normal variates (splitmix64 + Box-Muller) for the initial weights.
struct InitRng {
    uint64_t s;
    uint64_t next() {
        uint64_t z = (s += 0x9E3779B97F4A7C15ull);
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        return z ^ (z >> 31);
    }
    double uniform() { return ((next() >> 11) + 0.5) * (1.0 / 9007199254740992.0); }
    double normal() {
        const double u1 = uniform(), u2 = uniform();
        return std::sqrt(-2.0 * std::log(u1)) * std::cos(6.283185307179586 * u2);
    }
};

}  // namespace

extern "C" {

int ohpt_denoiser_create(ohpt_denoiser** out, int device, uint64_t seed) {
    if (!out) return set_error(OHPT_ERR_INVALID_ARG, "ohpt_denoiser_create: null output");
    *out = nullptr;
    int ndev = 0;
    DNCHK(hipGetDeviceCount(&ndev));
    if (device < 0 || device >= ndev) return set_error(OHPT_ERR_INVALID_ARG, "ohpt_denoiser_create: no such device");
    DNCHK(hipSetDevice(device));
    auto* d = new ohpt_denoiser();
    d->device = device;
    if (hipDeviceGetAttribute(&d->num_cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess ||
        d->num_cus <= 0)
        d->num_cus = 256;
    size_t off = 0;
    for (int i = 0; i < kNumLayers; ++i) {
        Layer L{};
        L.sp = kLayers[i];
        L.cin0 = kActChan[L.sp.in0];
        L.cin1 = L.sp.in1 >= 0 ? kActChan[L.sp.in1] : 0;
        L.cin = L.cin0 + L.cin1;
        L.cout = L.sp.cout;
        L.np = (L.cout + 31) & ~31;
        L.cc = (L.cin % 32 == 0) ? 32 : 16;
        L.ks = (9 * L.cc + 31) / 32;
        L.nchunk = L.cin / L.cc;
        L.w_off = off;
        off += (size_t)9 * L.cin * L.cout;
        L.b_off = off;
        off += L.cout;
        d->layers.push_back(std::move(L));
    }
    d->nparam = off;
    // initial parameters on the host
    std::vector<float> p(d->nparam, 0.0f);
    InitRng rng{seed ^ 0x6F68707464656E6Full};
    for (const Layer& L : d->layers) {
        const double fan_in = 9.0 * (L.sp.in0 == X0 ? kInputChannels : L.cin);
        double std_ = std::sqrt(2.0 / fan_in);
        if (L.sp.out == kLogits) std_ = 0.1 * std::sqrt(1.0 / fan_in);
        for (int t = 0; t < 9; ++t)
            for (int ci = 0; ci < L.cin; ++ci)
                for (int co = 0; co < L.cout; ++co) {
                    const bool pad_channel = (L.sp.in0 == X0 && ci >= kInputChannels);
                    const double v = rng.normal() * std_;
                    p[L.w_off + ((size_t)t * L.cin + ci) * L.cout + co] = pad_channel ? 0.0f : (float)v;
                }
    }
    auto fail_out = [&](int rc) { ohpt_denoiser_destroy(d); return rc; };
    hipError_t e = hipStreamCreateWithFlags(&d->stream, hipStreamNonBlocking);
    if (e == hipSuccess) e = hipEventCreate(&d->ev0);
    if (e == hipSuccess) e = hipEventCreate(&d->ev1);
    if (e == hipSuccess) e = d->params.ensure(d->nparam * 4);
    if (e == hipSuccess) e = d->grads.ensure(d->nparam * 4);
    if (e == hipSuccess) e = d->adam_m.ensure(d->nparam * 4);
    if (e == hipSuccess) e = d->adam_v.ensure(d->nparam * 4);
    if (e == hipSuccess) e = d->loss_dev.ensure(16);
    for (Layer& L : d->layers) {
        if (e == hipSuccess) e = L.wf.ensure((size_t)L.nchunk * L.ks * L.np * 32 * 2);
        if (e == hipSuccess && L.sp.in0 != X0) e = L.wd.ensure((size_t)(L.np / 32) * 9 * L.cin * 32 * 2);
    }
    if (e != hipSuccess) return fail_out(set_hip_error("ohpt_denoiser_create", e));
    *out = d;
    const int rc = ohpt_denoiser_set_params(d, p.data(), d->nparam);
    if (rc != OHPT_OK) {
        *out = nullptr;
        return fail_out(rc);
    }
    return OHPT_OK;
}

int ohpt_denoiser_destroy(ohpt_denoiser* d) {
    if (!d) return OHPT_OK;
    (void)hipSetDevice(d->device);
    if (d->stream) (void)hipStreamSynchronize(d->stream);
    for (hipEvent_t e : d->conv_ev) (void)hipEventDestroy(e);
    if (d->ev0) (void)hipEventDestroy(d->ev0);
    if (d->ev1) (void)hipEventDestroy(d->ev1);
    hipStream_t s = d->stream;
    delete d;
    if (s) (void)hipStreamDestroy(s);
    return OHPT_OK;
}

int ohpt_denoiser_param_count(ohpt_denoiser* d, uint64_t* n) {
    if (!d || !n) return set_error(OHPT_ERR_INVALID_ARG, "ohpt_denoiser_param_count: null argument");
    *n = d->nparam;
    return OHPT_OK;
}

int ohpt_denoiser_get_params(ohpt_denoiser* d, float* out, uint64_t n) {
    if (!d || !out) return set_error(OHPT_ERR_INVALID_ARG, "ohpt_denoiser_get_params: null argument");
    if (n != d->nparam) return set_error(OHPT_ERR_INVALID_ARG, "ohpt_denoiser_get_params: wrong count");
    DNCHK(hipSetDevice(d->device));
    DNCHK(hipMemcpyAsync(out, d->params.p, n * 4, hipMemcpyDeviceToHost, d->stream));
    DNCHK(hipStreamSynchronize(d->stream));
    return OHPT_OK;
}

int ohpt_denoiser_set_params(ohpt_denoiser* d, const float* in, uint64_t n) {
    if (!d || !in) return set_error(OHPT_ERR_INVALID_ARG, "ohpt_denoiser_set_params: null argument");
    if (n != d->nparam) return set_error(OHPT_ERR_INVALID_ARG, "ohpt_denoiser_set_params: wrong count");
    DNCHK(hipSetDevice(d->device));
    DNCHK(hipMemcpyAsync(d->params.p, in, n * 4, hipMemcpyHostToDevice, d->stream));
    DNCHK(hipMemsetAsync(d->adam_m.p, 0, n * 4, d->stream));
    DNCHK(hipMemsetAsync(d->adam_v.p, 0, n * 4, d->stream));
    DNCHK(hipMemsetAsync(d->grads.p, 0, n * 4, d->stream));
    d->adam_t = 0;
    d->have_grads = false;
    DNCHK(pack_weights(d));
    DNCHK(hipStreamSynchronize(d->stream));
    return OHPT_OK;
}

int ohpt_denoiser_get_grads(ohpt_denoiser* d, float* out, uint64_t n) {
    if (!d || !out) return set_error(OHPT_ERR_INVALID_ARG, "ohpt_denoiser_get_grads: null argument");
    if (n != d->nparam) return set_error(OHPT_ERR_INVALID_ARG, "ohpt_denoiser_get_grads: wrong count");
    DNCHK(hipSetDevice(d->device));
    DNCHK(hipMemcpyAsync(out, d->grads.p, n * 4, hipMemcpyDeviceToHost, d->stream));
    DNCHK(hipStreamSynchronize(d->stream));
    return OHPT_OK;
}

int ohpt_denoiser_forward_backward(ohpt_denoiser* d, const ohpt_denoise_inputs* in, const float* target,
                                   uint32_t batch, uint32_t width, uint32_t height, float* loss, int on_device) {
    int rc = check_shape(d, in, batch, width, height);
    if (rc != OHPT_OK) return rc;
    if (!target) return set_error(OHPT_ERR_INVALID_ARG, "ohpt_denoiser_forward_backward: null target");
    DNCHK(hipSetDevice(d->device));
    Inputs x{};
    rc = stage_inputs(d, in, target, (size_t)batch * width * height, on_device, x);
    if (rc != OHPT_OK) return rc;
    begin_timing(d);
    rc = run_forward(d, x, batch, width, height, true);
    if (rc != OHPT_OK) return rc;
    const size_t ppx = (size_t)d->B * d->Hp * d->Wp;
    KpnArgs k{};
    k.logits = d->logits.as<float>();
    k.rad = x.rad;
    k.target = x.tgt;
    k.dlogits = d->dlogits.as<uint16_t>();
    k.loss_part = d->loss_part.as<float>();
    k.B = d->B;
    k.H = d->H;
    k.W = d->W;
    k.Hp = d->Hp;
    k.Wp = d->Wp;
    k.inv_count = (float)(1.0 / (3.0 * (double)batch * width * height));
    const uint32_t nblk = cdiv(ppx, 256);
    k_kpn<<<nblk, 256, 0, d->stream>>>(k);
    k_sum_serial<<<1, 256, 0, d->stream>>>(d->loss_part.as<float>(), (int)nblk, k.inv_count, d->loss_dev.as<float>());
    DNCHK(network_backward(d));
    DNCHK(hipGetLastError());
    rc = end_timing(d, true);
    if (rc != OHPT_OK) return rc;
    d->have_grads = true;
    if (loss) {
        DNCHK(hipMemcpyAsync(loss, d->loss_dev.p, 4, hipMemcpyDeviceToHost, d->stream));
        DNCHK(hipStreamSynchronize(d->stream));
    }
    return OHPT_OK;
}

int ohpt_denoiser_adam_step(ohpt_denoiser* d, float lr) {
    if (!d) return set_error(OHPT_ERR_INVALID_ARG, "ohpt_denoiser_adam_step: null denoiser");
    if (!d->have_grads) return set_error(OHPT_ERR_STATE, "ohpt_denoiser_adam_step: no gradient computed yet");
    if (!(lr >= 0.0f)) return set_error(OHPT_ERR_INVALID_ARG, "ohpt_denoiser_adam_step: bad learning rate");
    DNCHK(hipSetDevice(d->device));
    d->adam_t += 1;
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    const float bc1 = (float)(1.0 - std::pow(0.9, d->adam_t));
    const float bc2 = (float)(1.0 - std::pow(0.999, d->adam_t));
    k_adam<<<cdiv(d->nparam, 256), 256, 0, d->stream>>>(d->params.as<float>(), d->grads.as<float>(),
                                                         d->adam_m.as<float>(), d->adam_v.as<float>(), d->nparam, lr,
                                                         b1, b2, eps, bc1, bc2);
    DNCHK(pack_weights(d));
    return OHPT_OK;
}

int ohpt_denoiser_train_step(ohpt_denoiser* d, const ohpt_denoise_inputs* in, const float* target, uint32_t batch,
                             uint32_t width, uint32_t height, float lr, float* loss, int on_device) {
    const int rc = ohpt_denoiser_forward_backward(d, in, target, batch, width, height, loss, on_device);
    if (rc != OHPT_OK) return rc;
    return ohpt_denoiser_adam_step(d, lr);
}

int ohpt_denoiser_infer(ohpt_denoiser* d, const ohpt_denoise_inputs* in, float* out, uint32_t batch, uint32_t width,
                        uint32_t height, int on_device) {
    int rc = check_shape(d, in, batch, width, height);
    if (rc != OHPT_OK) return rc;
    if (!out) return set_error(OHPT_ERR_INVALID_ARG, "ohpt_denoiser_infer: null output");
    DNCHK(hipSetDevice(d->device));
    const size_t npx = (size_t)batch * width * height;
    Inputs x{};
    rc = stage_inputs(d, in, nullptr, npx, on_device, x);
    if (rc != OHPT_OK) return rc;
    float4* dst = reinterpret_cast<float4*>(out);
    if (!on_device) {
        DNCHK(d->out_stage.ensure(npx * 16));
        dst = d->out_stage.as<float4>();
    }
    begin_timing(d);
    rc = run_forward(d, x, batch, width, height, false, dst);   // the head convolution writes dst
    if (rc != OHPT_OK) return rc;
    DNCHK(hipGetLastError());
    rc = end_timing(d, false);
    if (rc != OHPT_OK) return rc;
    if (!on_device) {
        DNCHK(hipMemcpyAsync(out, dst, npx * 16, hipMemcpyDeviceToHost, d->stream));
        DNCHK(hipStreamSynchronize(d->stream));
    }
    return OHPT_OK;
}

int ohpt_denoiser_read_tensor(ohpt_denoiser* d, uint32_t index, float* out, uint64_t n) {
    if (!d || !out) return set_error(OHPT_ERR_INVALID_ARG, "ohpt_denoiser_read_tensor: null argument");
    if (d->B == 0) return set_error(OHPT_ERR_STATE, "ohpt_denoiser_read_tensor: nothing computed yet");
    DNCHK(hipSetDevice(d->device));
    const size_t px = (size_t)d->B * d->Hp * d->Wp;
    const bool grad = index >= 100;
    const uint32_t t = grad ? index - 100 : index;
    if (t == (uint32_t)kLogits) {
        const size_t cnt = px * 32;
        if (n != cnt) return set_error(OHPT_ERR_INVALID_ARG, "ohpt_denoiser_read_tensor: wrong count");
        if (!grad) {
            DNCHK(hipMemcpyAsync(out, d->logits.p, cnt * 4, hipMemcpyDeviceToHost, d->stream));
            DNCHK(hipStreamSynchronize(d->stream));
            return OHPT_OK;
        }
        DevBuf tmp;
        DNCHK(tmp.ensure(cnt * 4));
        k_bf16_to_f32<<<cdiv(cnt, 256), 256, 0, d->stream>>>(d->dlogits.as<uint16_t>(), tmp.as<float>(), cnt);
        DNCHK(hipMemcpyAsync(out, tmp.p, cnt * 4, hipMemcpyDeviceToHost, d->stream));
        DNCHK(hipStreamSynchronize(d->stream));
        return OHPT_OK;
    }
    if (t >= (uint32_t)kNumAct || (grad && t == (uint32_t)X0))
        return set_error(OHPT_ERR_INVALID_ARG, "ohpt_denoiser_read_tensor: no such tensor");
    const size_t cnt = (px >> (2 * kActLevel[t])) * kActChan[t];
    if (n != cnt) return set_error(OHPT_ERR_INVALID_ARG, "ohpt_denoiser_read_tensor: wrong count");
    DevBuf tmp;
    DNCHK(tmp.ensure(cnt * 4));
    const DevBuf& src = grad ? d->gact[t] : d->act[t];
    k_bf16_to_f32<<<cdiv(cnt, 256), 256, 0, d->stream>>>(src.as<uint16_t>(), tmp.as<float>(), cnt);
    DNCHK(hipMemcpyAsync(out, tmp.p, cnt * 4, hipMemcpyDeviceToHost, d->stream));
    DNCHK(hipStreamSynchronize(d->stream));
    return OHPT_OK;
}

int ohpt_denoiser_set_profiling(ohpt_denoiser* d, int on) {
    if (!d) return set_error(OHPT_ERR_INVALID_ARG, "ohpt_denoiser_set_profiling: null denoiser");
    d->profile = on != 0;
    return OHPT_OK;
}

int ohpt_denoiser_get_stats(ohpt_denoiser* d, ohpt_denoiser_stats* out) {
    if (!d || !out) return set_error(OHPT_ERR_INVALID_ARG, "ohpt_denoiser_get_stats: null argument");
    *out = d->stats;
    return OHPT_OK;
}

}  // extern "C"

namespace ohpt {
// Device-side entry used by ohpt_denoise: inputs already resolved on the device.
int denoiser_infer_device(ohpt_denoiser* d, const float* rad, const float* alb, const float* nrm, const float* dep,
                          float* out, uint32_t width, uint32_t height) {
    ohpt_denoise_inputs in{rad, alb, nrm, dep};
    return ohpt_denoiser_infer(d, &in, out, 1, width, height, 1);
}
}  // namespace ohpt
