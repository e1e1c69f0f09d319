// Ray/box and ray/triangle tests and the child ordering of the LBVH traversal
// (traverse.hip's persistent kernels).
//
// Ray/box: robust slab test with tmax scaled by 1+2*gamma(3) (Ize 2013).
// Ray/triangle: watertight test of Woop, Benthin & Wald (JCGT 2013); an edge
// function that rounds to zero is re-evaluated with an exact-sign difference
// of products (fused multiply-adds) instead of the paper's double precision.
#pragma once
// Every floating-point operation as written (no contraction), here and in the
// rest of each file that includes this header: hits match the oracle bit for bit.
#pragma clang fp contract(off)

#include "ohpt_internal.h"

namespace ohpt {
namespace trace {

constexpr float kGamma3Scale = 1.0f + 2.0f * (3.0f * 5.9604645e-08f) / (1.0f - 3.0f * 5.9604645e-08f);
struct RayPre {
    float ox, oy, oz;
    float ix, iy, iz;
    int kx, ky, kz;
    float Sx, Sy, Sz;
};

__device__ __forceinline__ float sel(float a, float b, float c, int k) { return k == 0 ? a : (k == 1 ? b : c); }

__device__ __forceinline__ RayPre ray_setup(float3 o, float3 d) {
    RayPre r;
    float dx = d.x, dy = d.y, dz = d.z;
    if (fabsf(dx) < 1e-20f) dx = copysignf(1e-20f, dx);
    if (fabsf(dy) < 1e-20f) dy = copysignf(1e-20f, dy);
    if (fabsf(dz) < 1e-20f) dz = copysignf(1e-20f, dz);
    r.ox = o.x; r.oy = o.y; r.oz = o.z;
    r.ix = 1.0f / dx; r.iy = 1.0f / dy; r.iz = 1.0f / dz;
    const float ax = fabsf(dx), ay = fabsf(dy), az = fabsf(dz);
    const int kz = (ax > ay) ? ((ax > az) ? 0 : 2) : ((ay > az) ? 1 : 2);
    int kx = kz + 1; if (kx == 3) kx = 0;
    int ky = kx + 1; if (ky == 3) ky = 0;
    const float dkz = sel(dx, dy, dz, kz);
    if (dkz < 0.0f) { const int t = kx; kx = ky; ky = t; }
    r.kx = kx; r.ky = ky; r.kz = kz;
    r.Sx = sel(dx, dy, dz, kx) / dkz;
    r.Sy = sel(dx, dy, dz, ky) / dkz;
    r.Sz = 1.0f / dkz;
    return r;
}

// entry distance, or +inf when the box is missed
__device__ __forceinline__ float box_hit(const RayPre& r, float lx, float ly, float lz, float hx, float hy,
                                         float hz, float tmin, float tmax) {
    const float ax = (lx - r.ox) * r.ix, bx = (hx - r.ox) * r.ix;
    const float ay = (ly - r.oy) * r.iy, by = (hy - r.oy) * r.iy;
    const float az = (lz - r.oz) * r.iz, bz = (hz - r.oz) * r.iz;
    float t0 = tmin;
    t0 = fmaxf(t0, fminf(ax, bx));
    t0 = fmaxf(t0, fminf(ay, by));
    t0 = fmaxf(t0, fminf(az, bz));
    // the exit distance scaled once: rounding x * s is monotonic for s > 0, so
    // min_i(x_i * s) == min_i(x_i) * s up to the sign of a zero, which the
    // comparison below ignores (and fminf skips NaNs either way)
    const float t1 = fminf(tmax, fminf(fminf(fmaxf(ax, bx), fmaxf(ay, by)), fmaxf(az, bz)) * kGamma3Scale);
    return (t0 <= t1) ? t0 : INFINITY;
}

// a*b - c*d by Kahan's algorithm with fused multiply-adds (error-free
// product residual; relative error below 2 ulp, Jeannerod, Louvet & Muller
// 2013): exactly zero only when the exact value is, otherwise of the exact
// sign -- what the watertight test needs when a float edge function rounds
// to zero.
__device__ __forceinline__ float diff_of_products(float a, float b, float c, float d) {
    const float w = c * d;
    const float e = fmaf(-c, d, w);
    const float f = fmaf(a, b, -w);
    return f + e;
}

__device__ __forceinline__ bool tri_hit(const RayPre& r, float4 a, float4 b, float4 c, float tmin, float tmax,
                                        float& tout, float& uout, float& vout) {
    const float Ax0 = a.x - r.ox, Ay0 = a.y - r.oy, Az0 = a.z - r.oz;
    const float Bx0 = b.x - r.ox, By0 = b.y - r.oy, Bz0 = b.z - r.oz;
    const float Cx0 = c.x - r.ox, Cy0 = c.y - r.oy, Cz0 = c.z - r.oz;
    const float Akz = sel(Ax0, Ay0, Az0, r.kz), Bkz = sel(Bx0, By0, Bz0, r.kz), Ckz = sel(Cx0, Cy0, Cz0, r.kz);
    const float Ax = sel(Ax0, Ay0, Az0, r.kx) - r.Sx * Akz;
    const float Ay = sel(Ax0, Ay0, Az0, r.ky) - r.Sy * Akz;
    const float Bx = sel(Bx0, By0, Bz0, r.kx) - r.Sx * Bkz;
    const float By = sel(Bx0, By0, Bz0, r.ky) - r.Sy * Bkz;
    const float Cx = sel(Cx0, Cy0, Cz0, r.kx) - r.Sx * Ckz;
    const float Cy = sel(Cx0, Cy0, Cz0, r.ky) - r.Sy * Ckz;
    float U = Cx * By - Cy * Bx;
    float V = Ax * Cy - Ay * Cx;
    float W = Bx * Ay - By * Ax;
    if (U == 0.0f || V == 0.0f || W == 0.0f) {
        U = diff_of_products(Cx, By, Cy, Bx);
        V = diff_of_products(Ax, Cy, Ay, Cx);
        W = diff_of_products(Bx, Ay, By, Ax);
    }
    if ((U < 0.0f || V < 0.0f || W < 0.0f) && (U > 0.0f || V > 0.0f || W > 0.0f)) return false;
    float det = U + V + W;
    if (det == 0.0f) return false;
    const float Az = r.Sz * Akz, Bz = r.Sz * Bkz, Cz = r.Sz * Ckz;
    float T = U * Az + V * Bz + W * Cz;
    if (det < 0.0f) { T = -T; det = -det; U = -U; V = -V; W = -W; }
    if (!(T > tmin * det) || !(T < tmax * det)) return false;
    const float rcp = 1.0f / det;
    tout = T * rcp;
    uout = V * rcp;
    vout = W * rcp;
    return true;
}

// Child order key: the entry distance's bits mapped to an unsigned total
// order, the two low bits replaced by the slot (keys of one node are distinct;
// entries within four ulps order by slot).
__device__ __forceinline__ uint32_t order_key(float e, uint32_t slot) {
    const uint32_t b = __float_as_uint(e);
    const uint32_t m = (b & 0x80000000u) ? 0xFFFFFFFFu : 0x80000000u;
    return ((b ^ m) & ~3u) | slot;
}
// The same order where no entry distance is negative (tmin >= +0: the maximum with
// +0 is never -0).
__device__ __forceinline__ uint32_t order_key_pos(float e, uint32_t slot) { return (__float_as_uint(e) & ~3u) | slot; }

}  // namespace trace
}  // namespace ohpt
