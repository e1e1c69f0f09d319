// Texel layout conversion on the device: callers hold w*h*channels floats, the
// kernels read and differentiate a packed copy of four floats per texel (one
// float for one channel).
//
// Bounded by HBM (28 B per three-channel texel, 29 MB or about 7 us for 1024^2);
// what these kernels replaced was a host loop between two copies over the bus:
// update 4.94 -> 0.052 ms, gradient read 2.61 -> 0.040 ms (both of device memory) and
// upload 3.07 -> 0.56 ms (the copy over the bus) for a 1024^2 RGB texture.
#include "ohpt_internal.h"

namespace ohpt {
namespace {

constexpr uint32_t kMeanBlocks = 512;   // two blocks per CU; the partial sums of one fit one block

// Packs texels and sums each channel in double: a thread takes every
// (gridDim * 256)-th texel, the block's threads are added as a tree, the blocks
// by k_texel_mean, so the mean depends on nothing but the texels.
template <int C>
__global__ __launch_bounds__(256) void k_texel_pack(const float* __restrict__ src, size_t n, float* __restrict__ dst,
                                                    double* __restrict__ partial) {
    __shared__ double red[3][256];
    double s[3] = {0.0, 0.0, 0.0};
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
        float v[4] = {0.0f, 0.0f, 0.0f, C == 3 ? 1.0f : 0.0f};
#pragma unroll
        for (int k = 0; k < C; ++k) v[k] = src[i * C + k];
        if constexpr (C == 1) dst[i] = v[0];
        else reinterpret_cast<float4*>(dst)[i] = make_float4(v[0], v[1], v[2], v[3]);
#pragma unroll
        for (int k = 0; k < (C < 3 ? C : 3); ++k) s[k] += (double)v[k];
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) red[k][threadIdx.x] = s[k];
    __syncthreads();
    for (uint32_t o = 128; o > 0; o >>= 1) {
        if (threadIdx.x < o)
            for (int k = 0; k < 3; ++k) red[k][threadIdx.x] += red[k][threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x < 3) partial[blockIdx.x * 3 + threadIdx.x] = red[threadIdx.x][0];
}

// One block: partial sums of nb <= kMeanBlocks blocks -> per-channel means (one
// channel reads as grey).
__global__ __launch_bounds__(256) void k_texel_mean(const double* __restrict__ partial, uint32_t nb, size_t n,
                                                    int grey, double* __restrict__ mean) {
    __shared__ double red[3][256];
    for (int k = 0; k < 3; ++k) {
        double s = 0.0;
        for (uint32_t b = threadIdx.x; b < nb; b += 256) s += partial[b * 3 + k];
        red[k][threadIdx.x] = s;
    }
    __syncthreads();
    for (uint32_t o = 128; o > 0; o >>= 1) {
        if (threadIdx.x < o)
            for (int k = 0; k < 3; ++k) red[k][threadIdx.x] += red[k][threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x < 3) mean[threadIdx.x] = red[grey ? 0 : threadIdx.x][0] / (double)n;
}

// Packed texels (four floats each) -> C floats each.
template <int C>
__global__ __launch_bounds__(256) void k_texel_unpack(const float* __restrict__ src, size_t n, float* __restrict__ dst) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;   // one float of the output
    if (i < n * C) dst[i] = src[(i / C) * 4 + i % C];
}

inline uint32_t div_up(uint64_t a, uint64_t b) { return (uint32_t)((a + b - 1) / b); }

}  // namespace

size_t texel_mean_scratch_bytes() { return (kMeanBlocks + 1) * 3 * sizeof(double); }

void launch_texel_pack(const float* src, size_t n, uint32_t channels, float* packed, void* scratch, hipStream_t s) {
    if (n == 0) return;
    double* mean = reinterpret_cast<double*>(scratch);
    double* partial = mean + 3;
    const uint32_t nb = n < (size_t)kMeanBlocks * 256 ? div_up(n, 256) : kMeanBlocks;
    if (channels == 1) k_texel_pack<1><<<nb, 256, 0, s>>>(src, n, packed, partial);
    else if (channels == 2) k_texel_pack<2><<<nb, 256, 0, s>>>(src, n, packed, partial);
    else if (channels == 3) k_texel_pack<3><<<nb, 256, 0, s>>>(src, n, packed, partial);
    else k_texel_pack<4><<<nb, 256, 0, s>>>(src, n, packed, partial);
    k_texel_mean<<<1, 256, 0, s>>>(partial, nb, n, channels == 1, mean);
}

void launch_texel_unpack(const float* packed, size_t n, uint32_t channels, float* dst, hipStream_t s) {
    if (n == 0) return;
    const uint32_t nb = div_up(n * channels, 256);
    if (channels == 2) k_texel_unpack<2><<<nb, 256, 0, s>>>(packed, n, dst);
    else k_texel_unpack<3><<<nb, 256, 0, s>>>(packed, n, dst);
}

}  // namespace ohpt
