// LBVH builder for gfx950: 30-bit Morton codes of triangle centroids, a stable
// LSD radix sort with LDS-local ranking (8-bit digits, wave64 ballot match),
// Karras 2012 hierarchy over (morton << 32 | prim) keys, and a bottom-up AABB
// refit level by level, then a collapse to 4-wide nodes (two binary levels per
// node) for traversal. Replaces the driver-built BLAS/TLAS of
// ohao/render/rt/rt_acceleration_structure.cpp:205-309, :419-535.
//
// Every floating-point step is IEEE add/mul/div/min/max without contraction,
// so the tree (topology and boxes) is bit-identical to a sequential build.
#pragma clang fp contract(off)

#include "ohpt_internal.h"

namespace ohpt {
namespace {

constexpr uint32_t kRadixBlock = 256;
constexpr uint32_t kRadixItems = 16;
constexpr uint32_t kRadixTile = kRadixBlock * kRadixItems;
constexpr uint32_t kRadixDigits = 256;

__device__ __forceinline__ uint32_t expand_bits10(uint32_t v) {
    v = (v * 0x00010001u) & 0xFF0000FFu;
    v = (v * 0x00000101u) & 0x0F00F00Fu;
    v = (v * 0x00000011u) & 0xC30C30C3u;
    v = (v * 0x00000005u) & 0x49249249u;
    return v;
}

__device__ __forceinline__ uint32_t quantize10(float c, float lo, float hi) {
    const float ext = hi - lo;
    float x = 0.5f;
    if (ext > 0.0f) x = (c - lo) / ext;
    const float f = x * 1024.0f;
    if (!(f > 0.0f)) return 0u;
    if (f >= 1023.0f) return 1023u;
    return (uint32_t)f;
}

__device__ __forceinline__ void tri_bounds(const float* t, float lo[3], float hi[3]) {
    for (int a = 0; a < 3; ++a) {
        lo[a] = fminf(fminf(t[a], t[3 + a]), t[6 + a]);
        hi[a] = fmaxf(fmaxf(t[a], t[3 + a]), t[6 + a]);
    }
}

// --- centroid bounds: per-block partial min/max, then one block folds them
__global__ __launch_bounds__(256) void k_centroid_bounds(const float* __restrict__ tp, uint32_t n,
                                                         float* __restrict__ partial) {
    __shared__ float smin[3][256], smax[3][256];
    float mn[3] = {INFINITY, INFINITY, INFINITY}, mx[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
        float lo[3], hi[3];
        tri_bounds(tp + (size_t)i * 9, lo, hi);
        for (int a = 0; a < 3; ++a) {
            const float c = (lo[a] + hi[a]) * 0.5f;
            mn[a] = fminf(mn[a], c);
            mx[a] = fmaxf(mx[a], c);
        }
    }
    for (int a = 0; a < 3; ++a) { smin[a][threadIdx.x] = mn[a]; smax[a][threadIdx.x] = mx[a]; }
    __syncthreads();
    for (uint32_t s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s)
            for (int a = 0; a < 3; ++a) {
                smin[a][threadIdx.x] = fminf(smin[a][threadIdx.x], smin[a][threadIdx.x + s]);
                smax[a][threadIdx.x] = fmaxf(smax[a][threadIdx.x], smax[a][threadIdx.x + s]);
            }
        __syncthreads();
    }
    if (threadIdx.x == 0)
        for (int a = 0; a < 3; ++a) {
            partial[blockIdx.x * 6 + a] = smin[a][0];
            partial[blockIdx.x * 6 + 3 + a] = smax[a][0];
        }
}

__global__ __launch_bounds__(256) void k_fold_bounds(float* __restrict__ partial, uint32_t nparts) {
    __shared__ float s[6][256];
    float v[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
    for (uint32_t i = threadIdx.x; i < nparts; i += 256)
        for (int a = 0; a < 3; ++a) {
            v[a] = fminf(v[a], partial[i * 6 + a]);
            v[3 + a] = fmaxf(v[3 + a], partial[i * 6 + 3 + a]);
        }
    for (int a = 0; a < 6; ++a) s[a][threadIdx.x] = v[a];
    __syncthreads();
    for (uint32_t st = 128; st > 0; st >>= 1) {
        if (threadIdx.x < st)
            for (int a = 0; a < 3; ++a) {
                s[a][threadIdx.x] = fminf(s[a][threadIdx.x], s[a][threadIdx.x + st]);
                s[3 + a][threadIdx.x] = fmaxf(s[3 + a][threadIdx.x], s[3 + a][threadIdx.x + st]);
            }
        __syncthreads();
    }
    // result stored after the partials region at index nparts
    if (threadIdx.x < 6) partial[(size_t)nparts * 6 + threadIdx.x] = s[threadIdx.x][0];
}

__global__ __launch_bounds__(256) void k_morton(const float* __restrict__ tp, uint32_t n,
                                                const float* __restrict__ bounds, uint32_t* __restrict__ keys,
                                                uint32_t* __restrict__ vals) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    float lo[3], hi[3];
    tri_bounds(tp + (size_t)i * 9, lo, hi);
    uint32_t q[3];
    for (int a = 0; a < 3; ++a) q[a] = quantize10((lo[a] + hi[a]) * 0.5f, bounds[a], bounds[3 + a]);
    keys[i] = (expand_bits10(q[0]) << 2) | (expand_bits10(q[1]) << 1) | expand_bits10(q[2]);
    vals[i] = i;
}

// --- stable LSD radix sort -------------------------------------------------
__global__ __launch_bounds__(kRadixBlock) void k_radix_hist(const uint32_t* __restrict__ keys, uint32_t n,
                                                            uint32_t shift, uint32_t nblocks,
                                                            uint32_t* __restrict__ hist) {
    __shared__ uint32_t h[kRadixDigits];
    h[threadIdx.x] = 0;
    __syncthreads();
    const uint32_t base = blockIdx.x * kRadixTile;
    for (uint32_t r = 0; r < kRadixItems; ++r) {
        const uint32_t idx = base + r * kRadixBlock + threadIdx.x;
        if (idx < n) atomicAdd(&h[(keys[idx] >> shift) & 0xFFu], 1u);
    }
    __syncthreads();
    hist[threadIdx.x * nblocks + blockIdx.x] = h[threadIdx.x];
}

__global__ __launch_bounds__(kRadixBlock) void k_radix_scatter(const uint32_t* __restrict__ kin,
                                                               const uint32_t* __restrict__ vin,
                                                               uint32_t* __restrict__ kout,
                                                               uint32_t* __restrict__ vout,
                                                               const uint32_t* __restrict__ offsets,
                                                               const uint32_t* __restrict__ digit_base, uint32_t n,
                                                               uint32_t shift, uint32_t nblocks) {
    __shared__ uint32_t s_base[kRadixDigits];
    __shared__ uint32_t s_wave[kRadixBlock / 64][kRadixDigits];
    const uint32_t t = threadIdx.x, wave = t >> 6, lane = t & 63u;
    s_base[t] = offsets[t * nblocks + blockIdx.x] + digit_base[t];
    const uint32_t base = blockIdx.x * kRadixTile;
    for (uint32_t r = 0; r < kRadixItems; ++r) {
        for (uint32_t w = 0; w < kRadixBlock / 64; ++w) s_wave[w][t] = 0u;
        __syncthreads();
        const uint32_t idx = base + r * kRadixBlock + t;
        const bool valid = idx < n;
        const uint32_t key = valid ? kin[idx] : 0u;
        const uint32_t digit = (key >> shift) & 0xFFu;
        uint64_t peers = __ballot(valid);
        for (uint32_t bit = 0; bit < 8; ++bit) {
            const bool set = (digit >> bit) & 1u;
            const uint64_t bm = __ballot(valid && set);
            peers &= set ? bm : ~bm;
        }
        const uint32_t rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(peers >> 32),
                                                        __builtin_amdgcn_mbcnt_lo((uint32_t)peers, 0u));
        const int leader = __ffsll((unsigned long long)peers) - 1;
        if (valid && (int)lane == leader) s_wave[wave][digit] = (uint32_t)__popcll(peers);
        __syncthreads();
        {
            uint32_t run = s_base[t];
            for (uint32_t w = 0; w < kRadixBlock / 64; ++w) {
                const uint32_t c = s_wave[w][t];
                s_wave[w][t] = run;
                run += c;
            }
            s_base[t] = run;
        }
        __syncthreads();
        if (valid) {
            const uint32_t pos = s_wave[wave][digit] + rank;
            kout[pos] = key;
            vout[pos] = vin[idx];
        }
        __syncthreads();
    }
}

// --- sorted geometry ----------------------------------------------------------
__global__ __launch_bounds__(256) void k_gather(const float* __restrict__ tp, const float* __restrict__ tn,
                                                const float* __restrict__ tuv, const uint32_t* __restrict__ tm,
                                                const uint32_t* __restrict__ sorted_prim, uint32_t n,
                                                float4* __restrict__ tris, float4* __restrict__ attrs,
                                                uint32_t* __restrict__ prim_out, uint32_t* __restrict__ slot_of) {
    const uint32_t s = blockIdx.x * 256 + threadIdx.x;
    if (s >= n) return;
    const uint32_t p = sorted_prim[s];
    const float* t = tp + (size_t)p * 9;
    tris[(size_t)s * 3 + 0] = make_float4(t[0], t[1], t[2], __uint_as_float(p));
    tris[(size_t)s * 3 + 1] = make_float4(t[3], t[4], t[5], 0.0f);
    tris[(size_t)s * 3 + 2] = make_float4(t[6], t[7], t[8], 0.0f);
    float nn[9];
    if (tn) {
        for (int k = 0; k < 9; ++k) nn[k] = tn[(size_t)p * 9 + k];
    } else {
        const float e1x = t[3] - t[0], e1y = t[4] - t[1], e1z = t[5] - t[2];
        const float e2x = t[6] - t[0], e2y = t[7] - t[1], e2z = t[8] - t[2];
        const float cx = e1y * e2z - e1z * e2y, cy = e1z * e2x - e1x * e2z, cz = e1x * e2y - e1y * e2x;
        for (int k = 0; k < 3; ++k) { nn[k * 3] = cx; nn[k * 3 + 1] = cy; nn[k * 3 + 2] = cz; }
    }
    float uv[6] = {0, 0, 0, 0, 0, 0};
    if (tuv)
        for (int k = 0; k < 6; ++k) uv[k] = tuv[(size_t)p * 6 + k];
    const uint32_t m = tm ? tm[p] : 0u;
    attrs[(size_t)s * 4 + 0] = make_float4(nn[0], nn[1], nn[2], nn[3]);
    attrs[(size_t)s * 4 + 1] = make_float4(nn[4], nn[5], nn[6], nn[7]);
    attrs[(size_t)s * 4 + 2] = make_float4(nn[8], uv[0], uv[1], uv[2]);
    attrs[(size_t)s * 4 + 3] = make_float4(uv[3], uv[4], uv[5], __uint_as_float(m));
    prim_out[s] = p;
    slot_of[p] = s;
}

// --- Karras 2012 hierarchy ------------------------------------------------------
__device__ __forceinline__ int kdelta(const uint32_t* __restrict__ mk, const uint32_t* __restrict__ pk,
                                      int64_t n, int64_t i, int64_t j) {
    if (j < 0 || j >= n) return -1;
    const uint64_t a = ((uint64_t)mk[i] << 32) | pk[i];
    const uint64_t b = ((uint64_t)mk[j] << 32) | pk[j];
    return __clzll((long long)(a ^ b));
}

__global__ __launch_bounds__(256) void k_karras(const uint32_t* __restrict__ mk, const uint32_t* __restrict__ pk,
                                                uint32_t n, uint32_t* __restrict__ nodes_u,
                                                uint32_t* __restrict__ node_parent,
                                                uint32_t* __restrict__ leaf_parent) {
    const int64_t i = blockIdx.x * 256 + threadIdx.x;
    const int64_t N = n;
    if (i >= N - 1) return;
    const int d = (kdelta(mk, pk, N, i, i + 1) - kdelta(mk, pk, N, i, i - 1)) >= 0 ? 1 : -1;
    const int dmin = kdelta(mk, pk, N, i, i - d);
    int64_t lmax = 2;
    while (kdelta(mk, pk, N, i, i + lmax * d) > dmin) lmax *= 2;
    int64_t l = 0;
    for (int64_t t = lmax / 2; t >= 1; t /= 2)
        if (kdelta(mk, pk, N, i, i + (l + t) * d) > dmin) l += t;
    const int64_t j = i + l * d;
    const int dnode = kdelta(mk, pk, N, i, j);
    int64_t s = 0, div = 2, t;
    do {
        t = (l + div - 1) / div;
        if (kdelta(mk, pk, N, i, i + (s + t) * d) > dnode) s += t;
        div *= 2;
    } while (t > 1);
    const int64_t gamma = i + s * d + min(d, 0);
    const int64_t lo = min(i, j), hi = max(i, j);
    const uint32_t c0 = (lo == gamma) ? (kLeafBit | (uint32_t)gamma) : (uint32_t)gamma;
    const uint32_t c1 = (hi == gamma + 1) ? (kLeafBit | (uint32_t)(gamma + 1)) : (uint32_t)(gamma + 1);
    nodes_u[(size_t)i * 16 + 12] = c0;
    nodes_u[(size_t)i * 16 + 13] = c1;
    nodes_u[(size_t)i * 16 + 15] = 0u;
    if (c0 & kLeafBit) leaf_parent[c0 & ~kLeafBit] = (uint32_t)i; else node_parent[c0] = (uint32_t)i;
    if (c1 & kLeafBit) leaf_parent[c1 & ~kLeafBit] = (uint32_t)i; else node_parent[c1] = (uint32_t)i;
    if (i == 0) node_parent[0] = kMiss;
}

__global__ void k_single_leaf(uint32_t* nodes_u, uint32_t* node_parent, uint32_t* leaf_parent) {
    nodes_u[12] = kLeafBit;
    nodes_u[13] = kLeafBit;
    nodes_u[15] = 0u;
    node_parent[0] = kMiss;
    leaf_parent[0] = 0u;
}

// --- level-synchronous refit -----------------------------------------------
// Cross-CU communication inside one kernel would need device-scope release/
// acquire (L2 write-back/invalidate on every XCD); instead nodes are bucketed
// by depth and refitted one level per launch, deepest first, so every child
// box was written by an earlier launch.
constexpr uint32_t kMaxLevels = 64;

__global__ __launch_bounds__(256) void k_node_depth(const uint32_t* __restrict__ node_parent, uint32_t ni,
                                                    uint32_t* __restrict__ depth, uint32_t* __restrict__ level_count) {
    __shared__ uint32_t h[kMaxLevels];
    if (threadIdx.x < kMaxLevels) h[threadIdx.x] = 0u;
    __syncthreads();
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i < ni) {
        uint32_t d = 0, p = i;
        while (node_parent[p] != kMiss && d < kMaxLevels - 1) { p = node_parent[p]; ++d; }
        depth[i] = d;
        atomicAdd(&h[d], 1u);
    }
    __syncthreads();
    if (threadIdx.x < kMaxLevels && h[threadIdx.x]) atomicAdd(&level_count[threadIdx.x], h[threadIdx.x]);
}

// level_cursor[d] starts at the level's offset; nodes are appended per level
__global__ __launch_bounds__(256) void k_level_scatter(const uint32_t* __restrict__ depth, uint32_t ni,
                                                       uint32_t* __restrict__ level_cursor,
                                                       uint32_t* __restrict__ level_nodes) {
    __shared__ uint32_t cnt[kMaxLevels], base[kMaxLevels];
    if (threadIdx.x < kMaxLevels) cnt[threadIdx.x] = 0u;
    __syncthreads();
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    uint32_t d = 0, r = 0;
    if (i < ni) {
        d = depth[i];
        r = atomicAdd(&cnt[d], 1u);
    }
    __syncthreads();
    if (threadIdx.x < kMaxLevels && cnt[threadIdx.x]) base[threadIdx.x] = atomicAdd(&level_cursor[threadIdx.x], cnt[threadIdx.x]);
    __syncthreads();
    if (i < ni) level_nodes[base[d] + r] = i;
}

__device__ __forceinline__ void child_box(uint32_t c, const float4* __restrict__ tris, const float* __restrict__ nodes_f,
                                          float lo[3], float hi[3]) {
    if (c & kLeafBit) {
        const size_t s = c & ~kLeafBit;
        const float4 a = tris[s * 3], b = tris[s * 3 + 1], e = tris[s * 3 + 2];
        const float v[9] = {a.x, a.y, a.z, b.x, b.y, b.z, e.x, e.y, e.z};
        tri_bounds(v, lo, hi);
    } else {
        const float* cb = nodes_f + (size_t)c * 16;
        for (int k = 0; k < 3; ++k) {
            lo[k] = fminf(cb[k], cb[6 + k]);
            hi[k] = fmaxf(cb[3 + k], cb[9 + k]);
        }
    }
}

__global__ __launch_bounds__(256) void k_refit_level(const float4* __restrict__ tris, float* __restrict__ nodes_f,
                                                     const uint32_t* __restrict__ node_parent,
                                                     const uint32_t* __restrict__ level_nodes, uint32_t count) {
    const uint32_t t = blockIdx.x * 256 + threadIdx.x;
    if (t >= count) return;
    const uint32_t node = level_nodes[t];
    const uint32_t* nodes_u = reinterpret_cast<const uint32_t*>(nodes_f);
    const uint32_t c0 = nodes_u[(size_t)node * 16 + 12], c1 = nodes_u[(size_t)node * 16 + 13];
    float lo0[3], hi0[3], lo1[3], hi1[3];
    child_box(c0, tris, nodes_f, lo0, hi0);
    child_box(c1, tris, nodes_f, lo1, hi1);
    float* nd = nodes_f + (size_t)node * 16;
    for (int k = 0; k < 3; ++k) { nd[k] = lo0[k]; nd[3 + k] = hi0[k]; nd[6 + k] = lo1[k]; nd[9 + k] = hi1[k]; }
    reinterpret_cast<uint32_t*>(nd)[14] = node_parent[node];
}

// --- 4-wide collapse ----------------------------------------------------------
// Every internal node at even depth becomes a 4-wide node; they are numbered in
// binary-node order by an exclusive scan of the even-depth flags (tiles of
// kCollapseTile nodes: per-tile counts, a scan of the counts, per-tile ranks),
// so the numbering does not depend on scheduling.
constexpr uint32_t kCollapseItems = 16;
constexpr uint32_t kCollapseTile = 256 * kCollapseItems;

__global__ __launch_bounds__(256) void k_even_count(const uint32_t* __restrict__ depth, uint32_t ni,
                                                    uint32_t* __restrict__ tile_count) {
    __shared__ uint32_t red[256];
    const uint32_t b0 = blockIdx.x * kCollapseTile + threadIdx.x * kCollapseItems;
    uint32_t c = 0;
    for (uint32_t k = 0; k < kCollapseItems; ++k) {
        const uint32_t i = b0 + k;
        if (i < ni && (depth[i] & 1u) == 0) ++c;
    }
    red[threadIdx.x] = c;
    __syncthreads();
    for (uint32_t off = 128; off > 0; off >>= 1) {
        if (threadIdx.x < off) red[threadIdx.x] += red[threadIdx.x + off];
        __syncthreads();
    }
    if (threadIdx.x == 0) tile_count[blockIdx.x] = red[0];
}

// tile_base: exclusive scan of the tile counts
__global__ __launch_bounds__(256) void k_even_map(const uint32_t* __restrict__ depth, uint32_t ni,
                                                  const uint32_t* __restrict__ tile_base, uint32_t* __restrict__ map) {
    __shared__ uint32_t part[256];
    const uint32_t b0 = blockIdx.x * kCollapseTile + threadIdx.x * kCollapseItems;
    uint32_t c = 0;
    for (uint32_t k = 0; k < kCollapseItems; ++k) {
        const uint32_t i = b0 + k;
        if (i < ni && (depth[i] & 1u) == 0) ++c;
    }
    part[threadIdx.x] = c;
    __syncthreads();
    for (uint32_t off = 1; off < 256; off <<= 1) {
        const uint32_t v = threadIdx.x >= off ? part[threadIdx.x - off] : 0u;
        __syncthreads();
        part[threadIdx.x] += v;
        __syncthreads();
    }
    uint32_t run = tile_base[blockIdx.x] + part[threadIdx.x] - c;
    for (uint32_t k = 0; k < kCollapseItems; ++k) {
        const uint32_t i = b0 + k;
        if (i >= ni) break;
        map[i] = ((depth[i] & 1u) == 0) ? run++ : kMiss;
    }
}

// One thread per even-depth binary node: its 4-wide node holds its children,
// an internal child replaced by that child's two children (boxes as refitted).
__global__ __launch_bounds__(256) void k_collapse(const float* __restrict__ nodes_f, const uint32_t* __restrict__ depth,
                                                  const uint32_t* __restrict__ map, uint32_t ni,
                                                  float4* __restrict__ nodes4) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= ni || (depth[i] & 1u)) return;
    const uint32_t* nodes_u = reinterpret_cast<const uint32_t*>(nodes_f);
    float b[6][4];
    uint32_t ref[4] = {kMiss, kMiss, kMiss, kMiss};
#pragma unroll
    for (int a = 0; a < 6; ++a) b[a][0] = b[a][1] = b[a][2] = b[a][3] = 0.0f;
    uint32_t m = 0;
    for (int c = 0; c < 2; ++c) {
        const uint32_t ch = nodes_u[(size_t)i * 16 + 12 + c];
        if (ch & kLeafBit) {
            for (int a = 0; a < 6; ++a) b[a][m] = nodes_f[(size_t)i * 16 + 6 * c + a];
            ref[m++] = ch;
        } else {
            for (int cc = 0; cc < 2; ++cc) {
                const uint32_t g = nodes_u[(size_t)ch * 16 + 12 + cc];
                for (int a = 0; a < 6; ++a) b[a][m] = nodes_f[(size_t)ch * 16 + 6 * cc + a];
                ref[m++] = (g & kLeafBit) ? g : map[g];
            }
        }
    }
    float4* q = nodes4 + (size_t)map[i] * 8;
#pragma unroll
    for (int a = 0; a < 6; ++a) q[a] = make_float4(b[a][0], b[a][1], b[a][2], b[a][3]);
    q[6] = make_float4(__uint_as_float(ref[0]), __uint_as_float(ref[1]), __uint_as_float(ref[2]),
                       __uint_as_float(ref[3]));
    q[7] = make_float4(__uint_as_float(i), __uint_as_float(m), 0.0f, 0.0f);
}

inline uint32_t div_up(uint64_t a, uint64_t b) { return (uint32_t)((a + b - 1) / b); }

struct ScratchLayout {
    size_t keys0, vals0, keys1, vals1, hist, digit, partial, node_parent, leaf_parent, node_depth, levels,
        level_nodes, map4, tiles4, total;
};
ScratchLayout layout(uint32_t n) {
    auto al = [](size_t x) { return (x + 255) & ~size_t(255); };
    const uint32_t nb = div_up(n, kRadixTile);
    ScratchLayout L{};
    size_t o = 0;
    L.keys0 = o; o += al((size_t)n * 4);
    L.vals0 = o; o += al((size_t)n * 4);
    L.keys1 = o; o += al((size_t)n * 4);
    L.vals1 = o; o += al((size_t)n * 4);
    L.hist = o; o += al((size_t)kRadixDigits * nb * 4 + 4);
    L.digit = o; o += al((size_t)kRadixDigits * 4 * 2);
    L.partial = o; o += al((size_t)(1024 + 1) * 6 * 4);
    L.node_parent = o; o += al((size_t)n * 4 + 4);
    L.leaf_parent = o; o += al((size_t)n * 4 + 4);
    L.node_depth = o; o += al((size_t)n * 4 + 4);
    L.levels = o; o += al((size_t)kMaxLevels * 4 * 2);
    L.level_nodes = o; o += al((size_t)n * 4 + 4);
    L.map4 = o; o += al((size_t)n * 4 + 4);
    L.tiles4 = o; o += al((size_t)div_up(n, kCollapseTile) * 4 + 8);
    L.total = o;
    return L;
}

__global__ void k_fill(uint32_t* p, uint32_t v, uint32_t n) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) p[i] = v;
}

// Exclusive scan of one digit's per-block counts (one block per digit);
// writes the digit's total.
__global__ __launch_bounds__(256) void k_scan_digit(uint32_t* __restrict__ hist, uint32_t nb,
                                                    uint32_t* __restrict__ totals) {
    __shared__ uint32_t part[256];
    uint32_t* row = hist + (size_t)blockIdx.x * nb;
    const uint32_t per = (nb + 255) / 256;
    const uint32_t b0 = threadIdx.x * per, e = min(b0 + per, nb);
    uint32_t s = 0;
    for (uint32_t i = b0; i < e; ++i) s += row[i];
    part[threadIdx.x] = s;
    __syncthreads();
    for (uint32_t off = 1; off < 256; off <<= 1) {
        const uint32_t v = threadIdx.x >= off ? part[threadIdx.x - off] : 0u;
        __syncthreads();
        part[threadIdx.x] += v;
        __syncthreads();
    }
    uint32_t run = part[threadIdx.x] - s;
    for (uint32_t i = b0; i < e; ++i) {
        const uint32_t v = row[i];
        row[i] = run;
        run += v;
    }
    if (threadIdx.x == 255) totals[blockIdx.x] = part[255];
}

// Exclusive scan of the 256 digit totals -> digit base offsets.
__global__ __launch_bounds__(256) void k_scan_totals(const uint32_t* __restrict__ totals, uint32_t* __restrict__ base) {
    __shared__ uint32_t part[256];
    const uint32_t v0 = totals[threadIdx.x];
    part[threadIdx.x] = v0;
    __syncthreads();
    for (uint32_t off = 1; off < 256; off <<= 1) {
        const uint32_t v = threadIdx.x >= off ? part[threadIdx.x - off] : 0u;
        __syncthreads();
        part[threadIdx.x] += v;
        __syncthreads();
    }
    base[threadIdx.x] = part[threadIdx.x] - v0;
}

void radix_pass(const uint32_t* kin, const uint32_t* vin, uint32_t* kout, uint32_t* vout, uint32_t n, uint32_t shift,
                uint32_t nb, uint32_t* hist, uint32_t* digit, hipStream_t s) {
    k_radix_hist<<<nb, kRadixBlock, 0, s>>>(kin, n, shift, nb, hist);
    k_scan_digit<<<kRadixDigits, 256, 0, s>>>(hist, nb, digit);
    k_scan_totals<<<1, 256, 0, s>>>(digit, digit + kRadixDigits);
    k_radix_scatter<<<nb, kRadixBlock, 0, s>>>(kin, vin, kout, vout, hist, digit + kRadixDigits, n, shift, nb);
}

}  // namespace

size_t radix_sort_scratch_bytes(uint32_t n) {
    const uint32_t nb = div_up(n, kRadixTile);
    return ((size_t)n * 8 + 256) + ((size_t)kRadixDigits * nb * 4 + 256) + kRadixDigits * 8;
}

hipError_t radix_sort_pairs(uint32_t* keys, uint32_t* vals, uint32_t n, uint32_t key_bits, void* scratch,
                            hipStream_t s) {
    if (n == 0) return hipSuccess;
    const uint32_t nb = div_up(n, kRadixTile);
    uint32_t* k1 = reinterpret_cast<uint32_t*>(scratch);
    uint32_t* v1 = k1 + n;
    const size_t hist_off = ((size_t)n * 8 + 255) & ~size_t(255);
    uint32_t* hist = reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(scratch) + hist_off);
    uint32_t* digit = reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(scratch) + hist_off +
                                                  (((size_t)kRadixDigits * nb * 4 + 255) & ~size_t(255)));
    uint32_t *ka = keys, *va = vals, *kb = k1, *vb = v1;
    const uint32_t passes = (key_bits + 7) / 8;
    for (uint32_t p = 0; p < passes; ++p) {
        radix_pass(ka, va, kb, vb, n, p * 8, nb, hist, digit, s);
        std::swap(ka, kb);
        std::swap(va, vb);
    }
    if (ka != keys) {
        hipError_t e = hipMemcpyAsync(keys, ka, (size_t)n * 4, hipMemcpyDeviceToDevice, s);
        if (e == hipSuccess) e = hipMemcpyAsync(vals, va, (size_t)n * 4, hipMemcpyDeviceToDevice, s);
        if (e != hipSuccess) return e;
    }
    return hipGetLastError();
}

hipError_t exclusive_scan_u32(uint32_t* data, uint32_t n, uint32_t* total, hipStream_t s) {
    if (n == 0) return hipSuccess;
    k_scan_digit<<<1, 256, 0, s>>>(data, n, total);
    return hipGetLastError();
}

size_t lbvh_scratch_bytes(uint32_t n) { return layout(n).total; }

namespace {
// World-space corners (and normals) of one mesh's triangles from its
// object-space vertices, in double without contraction (off in this file) as
// world_triangle computes the emitters' on the host; commits and refits share it.
__global__ __launch_bounds__(256) void k_transform_mesh(const float* __restrict__ vpos, const float* __restrict__ vnrm,
                                                        const uint32_t* __restrict__ idx, uint32_t nt,
                                                        MeshTransform x, float* __restrict__ tpos,
                                                        float* __restrict__ tnrm) {
    const uint32_t t = blockIdx.x * 256 + threadIdx.x;
    if (t >= nt) return;
    const double* M = x.m;
    const double* N = x.n;
    float P[9];
    for (int k = 0; k < 3; ++k) {
        const uint32_t vi = idx[(size_t)t * 3 + k];
        const double px = vpos[(size_t)vi * 3], py = vpos[(size_t)vi * 3 + 1], pz = vpos[(size_t)vi * 3 + 2];
        if (x.has_world) {
            P[k * 3 + 0] = (float)(M[0] * px + M[4] * py + M[8] * pz + M[12]);
            P[k * 3 + 1] = (float)(M[1] * px + M[5] * py + M[9] * pz + M[13]);
            P[k * 3 + 2] = (float)(M[2] * px + M[6] * py + M[10] * pz + M[14]);
        } else {
            P[k * 3 + 0] = (float)px; P[k * 3 + 1] = (float)py; P[k * 3 + 2] = (float)pz;
        }
        if (tnrm && vnrm) {
            const double nx = vnrm[(size_t)vi * 3], ny = vnrm[(size_t)vi * 3 + 1], nz = vnrm[(size_t)vi * 3 + 2];
            double o0 = nx, o1 = ny, o2 = nz;
            if (x.has_world) {
                o0 = N[0] * nx + N[1] * ny + N[2] * nz;
                o1 = N[3] * nx + N[4] * ny + N[5] * nz;
                o2 = N[6] * nx + N[7] * ny + N[8] * nz;
            }
            float* Nn = tnrm + (size_t)t * 9 + k * 3;
            Nn[0] = (float)o0; Nn[1] = (float)o1; Nn[2] = (float)o2;
        }
    }
    for (int k = 0; k < 9; ++k) tpos[(size_t)t * 9 + k] = P[k];
    if (tnrm && !vnrm) {   // a mesh without normals in a scene with normals: its geometric normal
        const float e1[3] = {P[3] - P[0], P[4] - P[1], P[5] - P[2]}, e2[3] = {P[6] - P[0], P[7] - P[1], P[8] - P[2]};
        const float n[3] = {e1[1] * e2[2] - e1[2] * e2[1], e1[2] * e2[0] - e1[0] * e2[2], e1[0] * e2[1] - e1[1] * e2[0]};
        for (int k = 0; k < 3; ++k)
            for (int q = 0; q < 3; ++q) tnrm[(size_t)t * 9 + k * 3 + q] = n[q];
    }
}

__global__ __launch_bounds__(256) void k_gather_uv(const float* __restrict__ vuv, const uint32_t* __restrict__ idx,
                                                   uint32_t nc, float* __restrict__ tuv) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;   // corner
    if (i >= nc) return;
    const float2 v = vuv ? reinterpret_cast<const float2*>(vuv)[idx[i]] : make_float2(0.0f, 0.0f);
    reinterpret_cast<float2*>(tuv)[i] = v;
}
}  // namespace

void launch_gather_uv(const float* vuv, const uint32_t* idx, uint32_t nt, float* tuv, hipStream_t s) {
    if (nt) k_gather_uv<<<(uint32_t)(((uint64_t)nt * 3 + 255) / 256), 256, 0, s>>>(vuv, idx, nt * 3, tuv);
}

void launch_transform_mesh(const float* vpos, const float* vnrm, const uint32_t* idx, uint32_t nt,
                           const MeshTransform& x, float* tpos, float* tnrm, hipStream_t s) {
    if (nt) k_transform_mesh<<<(nt + 255) / 256, 256, 0, s>>>(vpos, vnrm, idx, nt, x, tpos, tnrm);
}

__global__ __launch_bounds__(256) void k_parent_from_nodes(const uint32_t* __restrict__ nodes_u, uint32_t ni,
                                                          uint32_t* __restrict__ node_parent) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i < ni) node_parent[i] = nodes_u[(size_t)i * 16 + 14];
}

// Depth buckets, level-by-level refit and the 4-wide numbering, shared by the
// build and the refit (node_parent filled, topology in b.nodes).
hipError_t refit_levels(const LbvhBuffers& b, const ScratchLayout& L, hipStream_t s, uint32_t* depth_out,
                        uint32_t* n4_out) {
    const uint32_t n = b.n;
    char* sc = reinterpret_cast<char*>(b.scratch);
    uint32_t* node_parent = reinterpret_cast<uint32_t*>(sc + L.node_parent);
    uint32_t* node_depth = reinterpret_cast<uint32_t*>(sc + L.node_depth);
    uint32_t* level_count = reinterpret_cast<uint32_t*>(sc + L.levels);
    uint32_t* level_cursor = level_count + kMaxLevels;
    uint32_t* level_nodes = reinterpret_cast<uint32_t*>(sc + L.level_nodes);
    const uint32_t ni = n > 1 ? n - 1 : 1;
    k_fill<<<1, 256, 0, s>>>(level_count, 0u, 2 * kMaxLevels);
    k_node_depth<<<div_up(ni, 256), 256, 0, s>>>(node_parent, ni, node_depth, level_count);
    uint32_t counts[kMaxLevels];
    hipError_t e = hipMemcpyAsync(counts, level_count, sizeof(counts), hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) return e;
    uint32_t offs[kMaxLevels], maxd = 0, acc = 0, n4 = 0;
    for (uint32_t d = 0; d < kMaxLevels; ++d) {
        offs[d] = acc;
        acc += counts[d];
        if (counts[d]) maxd = d;
        if ((d & 1u) == 0) n4 += counts[d];
    }
    e = hipMemcpyAsync(level_cursor, offs, sizeof(offs), hipMemcpyHostToDevice, s);
    if (e != hipSuccess) return e;
    k_level_scatter<<<div_up(ni, 256), 256, 0, s>>>(node_depth, ni, level_cursor, level_nodes);
    for (int d = (int)maxd; d >= 0; --d) {
        if (counts[d] == 0) continue;
        k_refit_level<<<div_up(counts[d], 256), 256, 0, s>>>(b.tris, reinterpret_cast<float*>(b.nodes), node_parent,
                                                              level_nodes + offs[d], counts[d]);
    }
    // 4-wide numbering: even-depth flags -> per-tile counts -> scan -> ranks
    const uint32_t nt4 = div_up(ni, kCollapseTile);
    uint32_t* tiles4 = reinterpret_cast<uint32_t*>(sc + L.tiles4);
    uint32_t* map4 = reinterpret_cast<uint32_t*>(sc + L.map4);
    k_even_count<<<nt4, 256, 0, s>>>(node_depth, ni, tiles4);
    k_scan_digit<<<1, 256, 0, s>>>(tiles4, nt4, tiles4 + nt4);
    k_even_map<<<nt4, 256, 0, s>>>(node_depth, ni, tiles4, map4);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    // deepest leaf = two levels below the deepest internal node (root at 0, leaves counted)
    if (depth_out) *depth_out = maxd + 2;
    if (n4_out) *n4_out = n4;
    return hipStreamSynchronize(s);
}

hipError_t lbvh_refit(const LbvhBuffers& b, hipStream_t s) {
    const uint32_t n = b.n;
    if (n == 0) return hipSuccess;
    const ScratchLayout L = layout(n);
    char* sc = reinterpret_cast<char*>(b.scratch);
    uint32_t* node_parent = reinterpret_cast<uint32_t*>(sc + L.node_parent);
    const uint32_t ni = n > 1 ? n - 1 : 1;
    // new vertex data into the committed leaf order (b.prim: slot -> triangle id)
    k_gather<<<div_up(n, 256), 256, 0, s>>>(b.tri_pos, b.tri_nrm, b.tri_uv, b.tri_mat, b.prim, n, b.tris, b.attrs,
                                             reinterpret_cast<uint32_t*>(sc + L.vals0), b.slot_of);
    k_parent_from_nodes<<<div_up(ni, 256), 256, 0, s>>>(reinterpret_cast<const uint32_t*>(b.nodes), ni, node_parent);
    return refit_levels(b, L, s, nullptr, nullptr);
}

hipError_t lbvh_build(const LbvhBuffers& b, hipStream_t s, uint32_t* depth_out, uint32_t* n4_out) {
    const uint32_t n = b.n;
    if (n == 0) return hipSuccess;
    const ScratchLayout L = layout(n);
    char* sc = reinterpret_cast<char*>(b.scratch);
    uint32_t* keys0 = reinterpret_cast<uint32_t*>(sc + L.keys0);
    uint32_t* vals0 = reinterpret_cast<uint32_t*>(sc + L.vals0);
    uint32_t* keys1 = reinterpret_cast<uint32_t*>(sc + L.keys1);
    uint32_t* vals1 = reinterpret_cast<uint32_t*>(sc + L.vals1);
    uint32_t* hist = reinterpret_cast<uint32_t*>(sc + L.hist);
    float* partial = reinterpret_cast<float*>(sc + L.partial);
    uint32_t* digit = reinterpret_cast<uint32_t*>(sc + L.digit);
    uint32_t* node_parent = reinterpret_cast<uint32_t*>(sc + L.node_parent);
    uint32_t* leaf_parent = reinterpret_cast<uint32_t*>(sc + L.leaf_parent);

    const uint32_t nparts = std::min<uint32_t>(1024u, div_up(n, 256));
    k_centroid_bounds<<<nparts, 256, 0, s>>>(b.tri_pos, n, partial);
    k_fold_bounds<<<1, 256, 0, s>>>(partial, nparts);
    const float* bounds = partial + (size_t)nparts * 6;
    k_morton<<<div_up(n, 256), 256, 0, s>>>(b.tri_pos, n, bounds, keys0, vals0);

    // 30-bit keys: four 8-bit passes (the last covers bits 24..29)
    const uint32_t nb = div_up(n, kRadixTile);
    uint32_t *ka = keys0, *va = vals0, *kb = keys1, *vb = vals1;
    for (uint32_t p = 0; p < 4; ++p) {
        radix_pass(ka, va, kb, vb, n, p * 8, nb, hist, digit, s);
        std::swap(ka, kb);
        std::swap(va, vb);
    }
    k_gather<<<div_up(n, 256), 256, 0, s>>>(b.tri_pos, b.tri_nrm, b.tri_uv, b.tri_mat, va, n, b.tris, b.attrs,
                                             b.prim, b.slot_of);
    uint32_t* nodes_u = reinterpret_cast<uint32_t*>(b.nodes);
    if (n == 1) {
        k_single_leaf<<<1, 1, 0, s>>>(nodes_u, node_parent, leaf_parent);
    } else {
        k_karras<<<div_up(n - 1, 256), 256, 0, s>>>(ka, va, n, nodes_u, node_parent, leaf_parent);
    }
    // bucket internal nodes by depth, then refit level by level, deepest first
    return refit_levels(b, L, s, depth_out, n4_out);
}

hipError_t bvh4_collapse(const LbvhBuffers& b, float4* nodes4, hipStream_t s) {
    const uint32_t n = b.n;
    if (n == 0) return hipSuccess;
    const ScratchLayout L = layout(n);
    const char* sc = reinterpret_cast<const char*>(b.scratch);
    const uint32_t ni = n > 1 ? n - 1 : 1;
    k_collapse<<<div_up(ni, 256), 256, 0, s>>>(reinterpret_cast<const float*>(b.nodes),
                                                reinterpret_cast<const uint32_t*>(sc + L.node_depth),
                                                reinterpret_cast<const uint32_t*>(sc + L.map4), ni, nodes4);
    return hipGetLastError();
}

}  // namespace ohpt
