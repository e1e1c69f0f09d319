// Environment importance-sampling tables on the GPU (EnvCDF::build,
// ohao/render/rt/env_cdf.cpp:13-61): per-row prefix sums of
// luminance * sin(theta_row_centre), normalised, plus the marginal CDF over
// rows and the integral. Each row is summed sequentially in column order, as
// the reference does, so the tables differ from it only through sinf.
#pragma clang fp contract(off)

#include "ohpt_internal.h"

namespace ohpt {
namespace {

constexpr uint32_t kScanChunk = 2048;   // values per LDS pass, a multiple of the block

// Prefix sums of n values in their order, on from `acc`: one thread, from LDS, so
// an addition waits for the last one and not for memory.
__device__ __forceinline__ float scan_in_order(float* v, uint32_t n, float acc) {
    uint32_t i = 0;
    for (; i + 4 <= n; i += 4) {
        float4 q = *reinterpret_cast<const float4*>(v + i);
        acc += q.x; q.x = acc;
        acc += q.y; q.y = acc;
        acc += q.z; q.z = acc;
        acc += q.w; q.w = acc;
        *reinterpret_cast<float4*>(v + i) = q;
    }
    for (; i < n; ++i) { acc += v[i]; v[i] = acc; }
    return acc;
}

// A block per row: the texels are read and weighted by all threads, summed in column
// order by one, and divided by all. With a thread per row every step of the sum waited
// for its texel: 512x256 260 us, 2048x1024 1054 us; now 13 and 59 us.
__global__ __launch_bounds__(256) void k_env_rows(const float4* __restrict__ env, uint32_t W, uint32_t H,
                                                  float* __restrict__ cond, float* __restrict__ row_sum) {
    __shared__ __align__(16) float v[kScanChunk];
    __shared__ float total;
    const uint32_t y = blockIdx.x;
    const float kPiF = 3.14159265358979323846f;
    const float theta = kPiF * ((float)y + 0.5f) / (float)H;
    const float s = sinf(theta);
    const float4* row = env + (size_t)y * W;
    float* c = cond + (size_t)y * W;
    if (threadIdx.x == 0) total = 0.0f;
    for (uint32_t x0 = 0; x0 < W; x0 += kScanChunk) {
        const uint32_t n = min(kScanChunk, W - x0);
        for (uint32_t i = threadIdx.x; i < n; i += 256) {
            const float4 p = row[x0 + i];
            const float l = 0.2126f * p.x + 0.7152f * p.y + 0.0722f * p.z;
            v[i] = l * s;
        }
        __syncthreads();
        if (threadIdx.x == 0) total = scan_in_order(v, n, total);
        __syncthreads();
        for (uint32_t i = threadIdx.x; i < n; i += 256) c[x0 + i] = v[i];
        __syncthreads();
    }
    const float acc = total;
    for (uint32_t x = threadIdx.x; x < W; x += 256)   // each thread's own sums again
        c[x] = acc > 0.0f ? c[x] / acc : (float)(x + 1) / (float)W;
    if (threadIdx.x == 0) row_sum[y] = acc;
}

// The same for the rows' sums, one block.
__global__ __launch_bounds__(256) void k_env_marginal(const float* __restrict__ row_sum, uint32_t H,
                                                      float* __restrict__ marg, float* __restrict__ integral) {
    __shared__ __align__(16) float v[kScanChunk];
    __shared__ float total;
    if (threadIdx.x == 0) total = 0.0f;
    for (uint32_t y0 = 0; y0 < H; y0 += kScanChunk) {
        const uint32_t n = min(kScanChunk, H - y0);
        for (uint32_t i = threadIdx.x; i < n; i += 256) v[i] = row_sum[y0 + i];
        __syncthreads();
        if (threadIdx.x == 0) total = scan_in_order(v, n, total);
        __syncthreads();
        for (uint32_t i = threadIdx.x; i < n; i += 256) marg[y0 + i] = v[i];
        __syncthreads();
    }
    const float acc = total;
    if (threadIdx.x == 0) *integral = acc;
    for (uint32_t y = threadIdx.x; y < H; y += 256) marg[y] = acc > 0.0f ? marg[y] / acc : (float)(y + 1) / (float)H;
}

// Guide tables for CDF inversion (the cutpoint method): for a CDF of n
// entries and M = 2^log2m cells, guide[k] = first index i with cdf[i] >= k/M
// (k/M is exact), guide[M] likewise for 1. A lookup of u in cell
// k = floor(u*M) (exact: M is a power of two) then searches only
// [guide[k], guide[k+1]], which holds the answer of the full search, so the
// sampled texel is the same as with the full binary search.
__global__ __launch_bounds__(256) void k_env_guide(const float* __restrict__ cdf, uint32_t n, uint32_t rows,
                                                   uint32_t log2m, uint32_t* __restrict__ guide) {
    const uint32_t m = 1u << log2m;
    const uint64_t t = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= (uint64_t)rows * (m + 1)) return;
    const uint32_t row = (uint32_t)(t / (m + 1)), k = (uint32_t)(t % (m + 1));
    guide[t] = cdf_lower_bound(cdf + (size_t)row * n, n, ldexpf((float)k, -(int)log2m));
}

__global__ __launch_bounds__(256) void k_env_sample(DevScene S, const float* __restrict__ u, float4* __restrict__ out,
                                                    uint32_t n) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    f3 d = mk(0.0f, 0.0f, 0.0f);
    float pdf = 0.0f;
    if (!env_sample(S, u[2 * i], u[2 * i + 1], d, pdf)) pdf = 0.0f;
    out[i] = make_float4(d.x, d.y, d.z, pdf);
}

}  // namespace

void launch_env_sample(const DevScene& S, const float* u, float4* out, uint32_t n, hipStream_t s) {
    if (n == 0 || S.env_w == 0) return;
    k_env_sample<<<(n + 255) / 256, 256, 0, s>>>(S, u, out, n);
}

uint32_t env_guide_log2(uint32_t n) {
    uint32_t l = 0;
    while ((2u << l) <= n && l < 16) ++l;   // largest power of two <= n, at most 2^16 cells
    return l;
}

hipError_t env_cdf_build(const float4* env, uint32_t W, uint32_t H, float* marg, float* cond, float* row_sum,
                         float* integral_dev, uint32_t* marg_guide, uint32_t* cond_guide, hipStream_t s) {
    if (W == 0 || H == 0) return hipSuccess;
    k_env_rows<<<H, 256, 0, s>>>(env, W, H, cond, row_sum);
    k_env_marginal<<<1, 256, 0, s>>>(row_sum, H, marg, integral_dev);
    const uint32_t lm = env_guide_log2(H), lc = env_guide_log2(W);
    const uint64_t nm = (1ull << lm) + 1, nc = ((1ull << lc) + 1) * H;
    k_env_guide<<<(uint32_t)((nm + 255) / 256), 256, 0, s>>>(marg, H, 1u, lm, marg_guide);
    k_env_guide<<<(uint32_t)((nc + 255) / 256), 256, 0, s>>>(cond, W, H, lc, cond_guide);
    return hipGetLastError();
}

}  // namespace ohpt
