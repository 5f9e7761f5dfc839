// Grid construction (bounding cube, normalization, cell key, stable sort into sorted space), the
// Morton-ordered search structure with per-level cell hash tables, and the output gathers.
//
// Reference: GridKNNCuda.cu:1023-1133 (InitStructure), :74-88 (cell key), :898-936 (getBuckets),
// getOutputPoints.cu:9-63, GridKNNCuda.cu:1941-1968 (GetKNNIndexes).
#include <algorithm>
#include <cmath>
#include <cstring>
#include "egt_device.h"
#include "egt_internal.h"

namespace egt {
namespace {

constexpr int BLK = 256;
constexpr int MM_WORDS = 7;  // six extremes and the count of non-finite points
// Cells, over all levels, up to which the level tables are sized by their bound (every point a cell of its own, or
// every cell of the level's grid): 2 million points at the default grid, 0.5 GB of tables. Saves the trip to the host,
// and coarse levels, whose bound is far above their count on a surface, get short probe chains. Whole build / search,
// k=16, by count -> by bound, us: sphere 1,500 points 187 / 49 -> 165 / 49, 100,000 379 / 211 -> 357 / 208, 700,000
// 873 / 805 -> 859 / 771, 1.9M 1678 / 2068 -> 1806 / 2023; mixture 700,000 799 / 2153 -> 797 / 1904, 1.9M 1500 / 4457
// -> 1524 / 4085. Beyond, emptying and caching the larger tables costs more than it gives.
constexpr size_t TABLE_BOUND = (size_t)1 << 23;

// Per-block min/max of x, y, z (thrust reduce with minimum/maximum, GridKNNCuda.cu:1042-1059) plus a
// count of non-finite inputs.
__global__ void __launch_bounds__(BLK) k_minmax_partial(const float* __restrict__ x, const float* __restrict__ y,
                                                         const float* __restrict__ z, int64_t n,
                                                         float* __restrict__ part) {
    float v[6] = {1e8f, -1e8f, 1e8f, -1e8f, 1e8f, -1e8f};
    uint32_t nb = 0;
    for (int64_t i = (int64_t)blockIdx.x * BLK + threadIdx.x; i < n; i += (int64_t)gridDim.x * BLK) {
        const float a = x[i], b = y[i], c = z[i];
        nb += !(__builtin_isfinite(a) && __builtin_isfinite(b) && __builtin_isfinite(c));
        v[0] = fminf(v[0], a); v[1] = fmaxf(v[1], a);
        v[2] = fminf(v[2], b); v[3] = fmaxf(v[3], b);
        v[4] = fminf(v[4], c); v[5] = fmaxf(v[5], c);
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
#pragma unroll
        for (int c = 0; c < 6; c += 2) {
            v[c] = fminf(v[c], __shfl_xor(v[c], d, 64));
            v[c + 1] = fmaxf(v[c + 1], __shfl_xor(v[c + 1], d, 64));
        }
        nb += __shfl_xor(nb, d, 64);
    }
    __shared__ float s[BLK / 64][6];
    __shared__ uint32_t sb[BLK / 64];
    const int wid = threadIdx.x / 64;
    if (__lane_id() == 0) {
        for (int c = 0; c < 6; ++c) s[wid][c] = v[c];
        sb[wid] = nb;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < BLK / 64; ++w)
            for (int c = 0; c < 6; c += 2) {
                s[0][c] = fminf(s[0][c], s[w][c]);
                s[0][c + 1] = fmaxf(s[0][c + 1], s[w][c + 1]);
            }
        uint32_t t = 0;
        for (int w = 0; w < BLK / 64; ++w) t += sb[w];
        for (int c = 0; c < 6; ++c) part[blockIdx.x * MM_WORDS + c] = s[0][c];
        part[blockIdx.x * MM_WORDS + 6] = __uint_as_float(t);
    }
}

// Bounding cube of one cloud from the per-axis min/max, GridKNNCuda.cu:1042-1077.
__device__ inline void cube_from_minmax(const float (&v)[6], float& mn, float& mx) {
    const float minx = v[0] - 1e-6f, maxx = v[1] + 1e-6f, miny = v[2] - 1e-6f, maxy = v[3] + 1e-6f;
    const float minz = v[4] - 1e-6f, maxz = v[5] + 1e-6f;
    mn = fminf(fminf(minx, miny), minz);
    mx = fmaxf(fmaxf(maxx, maxy), maxz);
}

// The cube goes to the cloud's table entry, where the next kernels read it, and to the report, which the host
// reads once at the end of the build.
__device__ inline void write_cloud(CloudDev* __restrict__ cloud, uint32_t* __restrict__ cube, int64_t base, int64_t n,
                                   const float (&v)[6]) {
    float mn, mx;
    cube_from_minmax(v, mn, mx);
    CloudDev c{};
    c.base = base;
    c.n = n;
    c.min_extent = mn;
    c.extent = mx - mn;
    c.max_extent = mx;
    *cloud = c;
    cube[0] = __float_as_uint(mn);
    cube[1] = __float_as_uint(mx);
}

// One cloud: the blocks' partials to its entry and the count of non-finite points.
__global__ void __launch_bounds__(64) k_cloud_cube(const float* __restrict__ part, int nb, int64_t n,
                                                    CloudDev* __restrict__ cloud, uint32_t* __restrict__ bad,
                                                    uint32_t* __restrict__ cube) {
    float v[6] = {1e8f, -1e8f, 1e8f, -1e8f, 1e8f, -1e8f};
    uint32_t t = 0;
    for (int b = (int)threadIdx.x; b < nb; b += 64) {
        const float* p = part + (size_t)b * MM_WORDS;
#pragma unroll
        for (int c = 0; c < 6; c += 2) {
            v[c] = fminf(v[c], p[c]);
            v[c + 1] = fmaxf(v[c + 1], p[c + 1]);
        }
        t += __float_as_uint(p[6]);
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
#pragma unroll
        for (int c = 0; c < 6; c += 2) {
            v[c] = fminf(v[c], __shfl_xor(v[c], d, 64));
            v[c + 1] = fmaxf(v[c + 1], __shfl_xor(v[c + 1], d, 64));
        }
        t += __shfl_xor(t, d, 64);
    }
    if (threadIdx.x == 0) {
        write_cloud(cloud, cube, 0, n, v);
        *bad = t;
    }
}

// normalize_points GridKNNCuda.cu:840-849 fused with get_buckets_no_binary :74-88. With icloud (batch) each
// point uses its own cloud's cube. The normalized point and its key go out as one 16-byte record in input
// order (the gather into sorted order then reads one record per point), the key and index also as the sort's
// key and value arrays. Where a point is not finite the build goes on with every point at one place, and the host,
// which reads the count at its end, throws: no value reaches a cell index or a table.
__global__ void __launch_bounds__(BLK) k_normalize_key(const float* __restrict__ x, const float* __restrict__ y,
                                                        const float* __restrict__ z, int64_t n,
                                                        const int32_t* __restrict__ icloud,
                                                        const CloudDev* __restrict__ clouds,
                                                        const uint32_t* __restrict__ bad, float a, float ba, int B,
                                                        int log2B, float4* __restrict__ tp, uint32_t* __restrict__ key,
                                                        uint32_t* __restrict__ idx) {
    const int64_t i = (int64_t)blockIdx.x * BLK + threadIdx.x;
    if (i >= n) return;
    const CloudDev& c = clouds[icloud ? icloud[i] : 0];
    const float mn = c.min_extent, d = c.extent;
    float xn = (x[i] - mn) / d, yn = (y[i] - mn) / d, zn = (z[i] - mn) / d;
    if (*bad) xn = yn = zn = 0.5f;
    const uint32_t cx = (uint32_t)cell_of(xn, a, ba, B), cy = (uint32_t)cell_of(yn, a, ba, B),
                   cz = (uint32_t)cell_of(zn, a, ba, B);
    const uint32_t k = cx | (cy << log2B) | (cz << (2 * log2B));
    tp[i] = make_float4(xn, yn, zn, __uint_as_float(k));
    key[i] = k;
    idx[i] = (uint32_t)i;
}

// Cloud of every input point (binary search over the input offsets).
__global__ void __launch_bounds__(BLK) k_cloud_of(const int64_t* __restrict__ off, int nclouds, int64_t n,
                                                   int32_t* __restrict__ cloud) {
    const int64_t i = (int64_t)blockIdx.x * BLK + threadIdx.x;
    if (i >= n) return;
    int lo = 0, hi = nclouds - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (off[mid] <= i) lo = mid;
        else hi = mid - 1;
    }
    cloud[i] = lo;
}

// Order-preserving float <-> int map, so float min/max can use integer atomics.
__device__ inline int f2o(float f) {
    const int i = __float_as_int(f);
    return i >= 0 ? i : i ^ 0x7FFFFFFF;
}

// Per-cloud min/max of x, y, z (fold starting at +-1e8, as the reference's thrust reductions
// GridKNNCuda.cu:1042-1059) plus a count of non-finite inputs. A wave takes groups of 64 MM_ROUNDS consecutive points,
// the loads of a group in flight together. Rounds that lie in the running cloud fold into registers; where the cloud
// changes the wave reduces what it holds and one lane sends it, and a round that straddles clouds sends its points one
// by one. (With 16 points a thread, a stride of the block apart, a block of small clouds straddled in every thread:
// 110 us for 24 clouds of 38,000 points in all, the longest step of their build; now 17, and 140 for 20M points in
// 192 clouds, 560 with one group a wave.)
constexpr int MM_ROUNDS = 4;
__device__ inline void minmax_flush(int* __restrict__ mm, int c, const float (&v)[6]) {
    // atomics only where they change something: the waves of a large cloud would queue at its six words
    int seen[6];
#pragma unroll
    for (int j = 0; j < 6; ++j) seen[j] = __hip_atomic_load(&mm[c * 6 + j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
    for (int j = 0; j < 6; j += 2) {
        if (f2o(v[j]) < seen[j]) atomicMin(&mm[c * 6 + j], f2o(v[j]));
        if (f2o(v[j + 1]) > seen[j + 1]) atomicMax(&mm[c * 6 + j + 1], f2o(v[j + 1]));
    }
}
__global__ void __launch_bounds__(BLK) k_cloud_minmax(const float* __restrict__ x, const float* __restrict__ y,
                                                       const float* __restrict__ z, const int32_t* __restrict__ icloud,
                                                       int64_t n, int groups, int* __restrict__ mm,
                                                       uint32_t* __restrict__ bad) {
    const int lane = __lane_id();
    const int64_t w = (int64_t)blockIdx.x * (BLK / 64) + threadIdx.x / 64;
    float v[6] = {1e8f, -1e8f, 1e8f, -1e8f, 1e8f, -1e8f};
    uint32_t nb = 0;
    int run = -1;  // cloud of v
    auto flush = [&] {
        if (run < 0) return;
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) {
#pragma unroll
            for (int j = 0; j < 6; j += 2) {
                v[j] = fminf(v[j], __shfl_xor(v[j], d, 64));
                v[j + 1] = fmaxf(v[j + 1], __shfl_xor(v[j + 1], d, 64));
            }
        }
        if (lane == 0) minmax_flush(mm, run, v);
        run = -1;
#pragma unroll
        for (int j = 0; j < 6; j += 2) {
            v[j] = 1e8f;
            v[j + 1] = -1e8f;
        }
    };
    for (int g = 0; g < groups; ++g) {
        const int64_t first = (w * groups + g) * (64 * MM_ROUNDS);
        if (first >= n) break;  // wave-uniform
        float p[MM_ROUNDS][3];
        int ci[MM_ROUNDS];
#pragma unroll
        for (int r = 0; r < MM_ROUNDS; ++r) {
            const int64_t i = min(first + r * 64 + lane, n - 1);  // past the end: the last point again
            ci[r] = icloud[i];
            p[r][0] = x[i];
            p[r][1] = y[i];
            p[r][2] = z[i];
        }
#pragma unroll
        for (int r = 0; r < MM_ROUNDS; ++r) {
            nb += first + r * 64 + lane < n &&
                  !(__builtin_isfinite(p[r][0]) && __builtin_isfinite(p[r][1]) && __builtin_isfinite(p[r][2]));
            const int c0 = __builtin_amdgcn_readfirstlane(ci[r]);
            const bool uniform = __ballot(ci[r] == c0) == ~0ull;
            if (!uniform || c0 != run) flush();
            if (uniform) {
                run = c0;
#pragma unroll
                for (int ax = 0; ax < 3; ++ax) {
                    v[2 * ax] = fminf(v[2 * ax], p[r][ax]);
                    v[2 * ax + 1] = fmaxf(v[2 * ax + 1], p[r][ax]);
                }
            } else {
                float q[6];
#pragma unroll
                for (int ax = 0; ax < 3; ++ax) {
                    q[2 * ax] = fminf(1e8f, p[r][ax]);
                    q[2 * ax + 1] = fmaxf(-1e8f, p[r][ax]);
                }
                minmax_flush(mm, ci[r], q);
            }
        }
    }
    flush();
    if (nb) atomicAdd(bad, nb);
}

__global__ void __launch_bounds__(BLK) k_minmax_init(int* __restrict__ mm, int nclouds, uint32_t* __restrict__ bad) {
    const int i = blockIdx.x * BLK + threadIdx.x;
    if (i < nclouds * 6) mm[i] = f2o((i & 1) ? -1e8f : 1e8f);
    if (i == 0) *bad = 0;
}

// A batch: the entry of every cloud.
__global__ void __launch_bounds__(BLK) k_cloud_cubes(const int* __restrict__ mm, const int64_t* __restrict__ off,
                                                      int nclouds, CloudDev* __restrict__ clouds,
                                                      uint32_t* __restrict__ cubes) {
    const int c = blockIdx.x * BLK + threadIdx.x;
    if (c >= nclouds) return;
    float v[6];
#pragma unroll
    for (int j = 0; j < 6; ++j) {
        const int iv = mm[c * 6 + j];
        v[j] = __int_as_float(iv >= 0 ? iv : iv ^ 0x7FFFFFFF);
    }
    write_cloud(clouds + c, cubes + 2 * c, off[c], off[c + 1] - off[c], v);
}

// Cloud of each element of an index list (second, stable sort pass by cloud).
__global__ void __launch_bounds__(BLK) k_gather_cloud(const int32_t* __restrict__ cloud_of,
                                                       const uint32_t* __restrict__ idx, int64_t n,
                                                       uint32_t* __restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * BLK + threadIdx.x;
    if (i < n) out[i] = (uint32_t)cloud_of[idx[i]];
}

// Sort keys of the Morton order: the fine cell's Morton code and the Morton code of the point's position
// inside the cell (sorted first, stably, so that points of a cell end up in sub-code order); also the point as
// one 16-byte record (x, y, z, key) in sorted order for the gather into Morton order.
struct MortonKeys {
    float a, ba;
    int B, log2B;
    uint32_t *code, *sub, *idx;
    float4* spts;
};
__device__ inline void morton_keys(const MortonKeys& K, int64_t s, float px, float py, float pz, uint32_t k) {
    const uint32_t m = (1u << K.log2B) - 1u;
    const uint32_t cx = k & m, cy = (k >> K.log2B) & m, cz = k >> (2 * K.log2B);
    K.code[s] = morton_code(cx, cy, cz);
    K.sub[s] = vcell_sub(vcell_pack(vcoord(px, K.a, K.ba, K.B, (int)cx), vcoord(py, K.a, K.ba, K.B, (int)cy),
                                    vcoord(pz, K.a, K.ba, K.B, (int)cz)));
    K.idx[s] = (uint32_t)s;
    K.spts[s] = make_float4(px, py, pz, __int_as_float((int32_t)k));
}

// thrust::gather into sorted order, GridKNNCuda.cu:1114-1128: one 16-byte record per point; its Morton sort keys
// while it is at hand.
__global__ void __launch_bounds__(BLK) k_gather_sorted(const float4* __restrict__ tp, const int32_t* __restrict__ icloud,
                                                        const uint32_t* __restrict__ sidx, int64_t n,
                                                        float* __restrict__ x, float* __restrict__ y,
                                                        float* __restrict__ z, int32_t* __restrict__ perm,
                                                        int32_t* __restrict__ key, int32_t* __restrict__ scloud,
                                                        MortonKeys K) {
    const int64_t s = (int64_t)blockIdx.x * BLK + threadIdx.x;
    if (s >= n) return;
    const uint32_t o = sidx[s];
    const float4 v = tp[o];
    perm[s] = (int32_t)o;
    key[s] = __float_as_int(v.w);
    if (scloud) scloud[s] = icloud[o];
    x[s] = v.x;
    y[s] = v.y;
    z[s] = v.z;
    morton_keys(K, s, v.x, v.y, v.z, __float_as_uint(v.w));
}

__global__ void __launch_bounds__(BLK) k_gather_u32(const uint32_t* __restrict__ src,
                                                     const uint32_t* __restrict__ idx, int64_t n,
                                                     uint32_t* __restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * BLK + threadIdx.x;
    if (i < n) out[i] = src[idx[i]];
}

__global__ void __launch_bounds__(BLK) k_morton_points(const float4* __restrict__ spts,
                                                        const int32_t* __restrict__ scloud,
                                                        const uint32_t* __restrict__ order, int64_t n, float a,
                                                        float ba, int B, int log2B, float4* __restrict__ mpts,
                                                        uint32_t* __restrict__ mcell, unsigned long long* __restrict__ mvcell,
                                                        uint32_t* __restrict__ mcode, int32_t* __restrict__ mcloud,
                                                        int32_t* __restrict__ morder, int32_t* __restrict__ minv) {
    const int64_t m = (int64_t)blockIdx.x * BLK + threadIdx.x;
    if (m >= n) return;
    const uint32_t s = order[m];
    morder[m] = (int32_t)s;
    minv[s] = (int32_t)m;
    const float4 v = spts[s];
    const float px = v.x, py = v.y, pz = v.z;
    mpts[m] = make_float4(px, py, pz, __int_as_float((int)s));
    const uint32_t k = (uint32_t)__float_as_int(v.w), msk = (1u << log2B) - 1u;
    const uint32_t cx = k & msk, cy = (k >> log2B) & msk, cz = k >> (2 * log2B);
    mcell[m] = cx | (cy << 10) | (cz << 20);
    mvcell[m] = vcell_pack(vcoord(px, a, ba, B, (int)cx), vcoord(py, a, ba, B, (int)cy), vcoord(pz, a, ba, B, (int)cz));
    mcode[m] = morton_code(cx, cy, cz);
    if (mcloud) mcloud[m] = scloud[s];
}

// ---- Level tables ---------------------------------------------------------------------------------------
// Level l groups 2^l fine cells per axis (Morton code >> 3 l). Position m is the first of its level-l cell for
// every l below first_levels(m): the highest bit in which its code differs from the previous position's tells
// all levels at once, so one pass over the codes serves the whole pyramid. The counting and ranking kernels
// walk tiles of LV_TILE positions, position base + 256 r + thread, so a group of 64 positions is one wave's
// round r and a level's ranks come from ballots.
//
// Bound: launches on small clouds, the inserts' random lines on large ones. A flag pass, a scan (one to three
// launches), a starts pass and an insert pass per level were 45-80 launches per grid build, now 4-5. Whole calls:
// 1,500 points 2.45 -> 2.26 ms, 100,000 points (k=40, 150 iterations) 4.80 -> 4.58, 1M points (k=16, 50
// iterations, normals) 8.85 -> 8.31, 192 clouds of 20M points 145.8 -> 138.8.
constexpr int LV_ITEMS = 8;
constexpr int LV_TILE = BLK * LV_ITEMS;  // 2048
constexpr int LV_GROUPS = LV_TILE / 64;  // 32

__device__ inline int first_levels(const uint32_t* __restrict__ code, const int32_t* __restrict__ mcloud, int64_t m,
                                   int64_t n, int nl) {
    if (m >= n) return 0;
    if (m == 0 || (mcloud && mcloud[m] != mcloud[m - 1])) return nl;
    const uint32_t x = code[m] ^ code[m - 1];
    return x ? min(nl, (31 - __builtin_clz(x)) / 3 + 1) : 0;
}

// Cells that start in each tile: cnt[l * nb + tile].
__global__ void __launch_bounds__(BLK) k_level_count(const uint32_t* __restrict__ code,
                                                      const int32_t* __restrict__ mcloud, int64_t n, int nl, int nb,
                                                      uint32_t* __restrict__ cnt) {
    __shared__ uint32_t s[EGT_MAX_LEVELS];
    if (threadIdx.x < EGT_MAX_LEVELS) s[threadIdx.x] = 0;
    __syncthreads();
    const int64_t base = (int64_t)blockIdx.x * LV_TILE + threadIdx.x;
    int fl[LV_ITEMS];
#pragma unroll
    for (int r = 0; r < LV_ITEMS; ++r) fl[r] = first_levels(code, mcloud, base + r * BLK, n, nl);
    for (int l = 0; l < nl; ++l) {
        uint32_t c = 0;
#pragma unroll
        for (int r = 0; r < LV_ITEMS; ++r) c += (uint32_t)__popcll(__ballot(fl[r] > l));
        if (__lane_id() == 0) atomicAdd(&s[l], c);
    }
    __syncthreads();
    if ((int)threadIdx.x < nl) cnt[(int64_t)threadIdx.x * nb + blockIdx.x] = s[threadIdx.x];
}

// Exclusive prefix over the tiles of each level, in place (one block per level); the level's cell count goes
// to total[l * stride].
constexpr int LVS_BLK = 1024;
__global__ void __launch_bounds__(LVS_BLK) k_level_scan(uint32_t* __restrict__ cnt, int nb, uint32_t* __restrict__ total,
                                                         int stride) {
    __shared__ uint32_t ws[LVS_BLK / 64];
    uint32_t* c = cnt + (int64_t)blockIdx.x * nb;
    const int lane = __lane_id(), wid = threadIdx.x / 64;
    uint32_t run = 0;
    for (int b0 = 0; b0 < nb; b0 += LVS_BLK) {
        const int i = b0 + (int)threadIdx.x;
        const uint32_t v = i < nb ? c[i] : 0u;
        uint32_t x = v;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t o = __shfl_up(x, d, 64);
            if (lane >= d) x += o;
        }
        if (lane == 63) ws[wid] = x;
        __syncthreads();
        uint32_t off = 0, all = 0;
#pragma unroll
        for (int w = 0; w < LVS_BLK / 64; ++w) {
            if (w < wid) off += ws[w];
            all += ws[w];
        }
        if (i < nb) c[i] = run + off + x - v;
        run += all;
        __syncthreads();
    }
    if (threadIdx.x == 0) total[(int64_t)blockIdx.x * stride] = run;
}

// First position of every cell of every level: starts + soff[l], in Morton order. In a batch also the running cell
// count of every level at each cloud's first position, which is the rank of the cell that begins there:
// out[l * stride + 1 + c] (entry 0 of a level holds its total). A single tile needs no prefix (pre null): it writes the
// totals itself.
struct LevelStarts {
    uint64_t soff[EGT_MAX_LEVELS];
};
__global__ void __launch_bounds__(BLK) k_level_starts(const uint32_t* __restrict__ code,
                                                       const int32_t* __restrict__ mcloud, int64_t n, int nl, int nb,
                                                       const uint32_t* __restrict__ pre, LevelStarts S,
                                                       uint32_t* __restrict__ starts, uint32_t* __restrict__ out,
                                                       int stride) {
    __shared__ uint32_t g[EGT_MAX_LEVELS][LV_GROUPS];
    const int lane = __lane_id(), wid = threadIdx.x / 64;
    const int64_t base = (int64_t)blockIdx.x * LV_TILE + threadIdx.x;
    int fl[LV_ITEMS];
#pragma unroll
    for (int r = 0; r < LV_ITEMS; ++r) fl[r] = first_levels(code, mcloud, base + r * BLK, n, nl);
    for (int l = 0; l < nl; ++l) {
#pragma unroll
        for (int r = 0; r < LV_ITEMS; ++r) {
            const uint32_t c = (uint32_t)__popcll(__ballot(fl[r] > l));
            if (lane == 0) g[l][r * (BLK / 64) + wid] = c;
        }
    }
    __syncthreads();
    if ((int)threadIdx.x < nl) {
        uint32_t run = pre ? pre[(int64_t)threadIdx.x * nb + blockIdx.x] : 0u;
        for (int i = 0; i < LV_GROUPS; ++i) {
            const uint32_t c = g[threadIdx.x][i];
            g[threadIdx.x][i] = run;
            run += c;
        }
        if (!pre) out[(int64_t)threadIdx.x * stride] = run;
    }
    __syncthreads();
    const uint64_t lt = (1ull << lane) - 1ull;
    int first_of[LV_ITEMS];  // the cloud whose first position it is, or -1
    if (mcloud) {
#pragma unroll
        for (int r = 0; r < LV_ITEMS; ++r) {
            const int64_t m = base + r * BLK;
            first_of[r] = fl[r] == nl && (m == 0 || mcloud[m] != mcloud[m - 1]) ? mcloud[m] : -1;
        }
    }
    for (int l = 0; l < nl; ++l) {
#pragma unroll
        for (int r = 0; r < LV_ITEMS; ++r) {
            const uint64_t b = __ballot(fl[r] > l);
            if (fl[r] > l) {
                const uint32_t rank = g[l][r * (BLK / 64) + wid] + (uint32_t)__popcll(b & lt);
                starts[S.soff[l] + rank] = (uint32_t)(base + r * BLK);
                if (mcloud && first_of[r] >= 0) out[(int64_t)l * stride + 1 + first_of[r]] = rank;
            }
        }
    }
}

// Inserts the cells of every level (thread i: cell i - first[l] of the level l whose range holds i; ranges may be
// longer than the level's cell count count[l * stride]), one CAS per cell into a random slot. The level's largest cell
// is kept by one atomic per wave, and only by a wave that exceeds the value read first: with one unconditional atomic
// per wave, every wave of a level queued at one address (1M points: 411 us for the 11 levels, 158 us now; 4M points:
// 905 -> 347).
struct LevelInsert {
    int64_t first[EGT_MAX_LEVELS + 1];  // first thread of each level; first[nl] = all
    uint64_t soff[EGT_MAX_LEVELS];      // the level's cell starts
    uint64_t offset[EGT_MAX_LEVELS];    // the level's table
    uint32_t log2cap[EGT_MAX_LEVELS];
    uint64_t slots;                     // of all tables
    int nl;
};
__device__ inline void max_if_larger(int* p, int v) {
    if (v > __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(p, v);
}
__global__ void __launch_bounds__(BLK) k_level_insert(LevelInsert P, const uint32_t* __restrict__ starts, int64_t n,
                                                       const uint32_t* __restrict__ code,
                                                       const int32_t* __restrict__ mcloud,
                                                       const uint32_t* __restrict__ count, int stride,
                                                       uint4* __restrict__ tab, LevelDev* __restrict__ lev,
                                                       int64_t first_group) {
    const int64_t i = (first_group + blockIdx.x) * BLK + threadIdx.x;
    int l = 0;
    for (int j = 1; j < P.nl; ++j) l += i >= P.first[j] ? 1 : 0;
    int cnt = 0;
    const int64_t c = i - P.first[l], cells = count[(int64_t)l * stride];
    if (c < cells) {
        const uint32_t* st_l = starts + P.soff[l];
        const uint32_t st = st_l[c];
        const uint32_t en = c + 1 < cells ? st_l[c + 1] : (uint32_t)n;
        const unsigned long long cc = cell_key(mcloud ? (uint32_t)mcloud[st] : 0u, code[st] >> (3 * l));
        const uint32_t log2cap = P.log2cap[l], mask = (1u << log2cap) - 1u;
        uint32_t s = hash_slot(cc, log2cap);
        // a table has at least twice as many slots as cells, so an empty slot is always found
        for (;;) {
            uint4* e = &tab[P.offset[l] + s];
            const unsigned long long prev =
                atomicCAS(reinterpret_cast<unsigned long long*>(e), (unsigned long long)HASH_EMPTY, cc);
            if (prev == HASH_EMPTY) {
                reinterpret_cast<uint2*>(e)[1] = make_uint2(st, en - st);
                break;
            }
            s = (s + 1u) & mask;
        }
        cnt = (int)(en - st);
    }
    // levels ascend with the thread, so a wave that starts and ends in one level lies in it
    const int l0 = __shfl(l, 0, 64);
    if (__shfl(l, 63, 64) == l0) {
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) cnt = max(cnt, __shfl_xor(cnt, d, 64));
        if (__lane_id() == 0) max_if_larger(&lev[l0].max_count, cnt);
    } else {
        max_if_larger(&lev[l].max_count, cnt);
    }
}

// Empties the tables and writes their descriptors.
__global__ void __launch_bounds__(BLK) k_level_init(LevelInsert P, uint64_t* __restrict__ tab, LevelDev* __restrict__ lev) {
    for (uint64_t i = (uint64_t)blockIdx.x * BLK + threadIdx.x; i < 2 * P.slots; i += (uint64_t)gridDim.x * BLK)
        tab[i] = HASH_EMPTY;
    if (blockIdx.x == 0 && (int)threadIdx.x < P.nl)
        lev[threadIdx.x] = LevelDev{P.offset[threadIdx.x], P.log2cap[threadIdx.x], 0};
}

// produce_output_GKNN + rearrange_output, getOutputPoints.cu:9-30, into separate output buffers.
__global__ void __launch_bounds__(BLK) k_output(const float* __restrict__ x, const float* __restrict__ y,
                                                 const float* __restrict__ z, const int32_t* __restrict__ perm,
                                                 const int32_t* __restrict__ scloud,
                                                 const CloudDev* __restrict__ clouds, int64_t n, float mn, float d,
                                                 float* __restrict__ ox, float* __restrict__ oy,
                                                 float* __restrict__ oz) {
    const int64_t s = (int64_t)blockIdx.x * BLK + threadIdx.x;
    if (s >= n) return;
    if (scloud) {
        const CloudDev& c = clouds[scloud[s]];
        mn = c.min_extent;
        d = c.extent;
    }
    const int32_t o = perm[s];
    ox[o] = x[s] * d + mn;
    oy[o] = y[s] * d + mn;
    oz[o] = z[s] * d + mn;
}

// rearrangeReferenceNeighbors GridKNNCuda.cu:862-872 plus the host scatter :1959-1966, on the device.
__global__ void __launch_bounds__(BLK) k_knn_original(const int32_t* __restrict__ knn,
                                                       const int32_t* __restrict__ perm, int64_t n, int k,
                                                       int32_t* __restrict__ out) {
    const int64_t t = (int64_t)blockIdx.x * BLK + threadIdx.x;
    if (t >= n * k) return;
    const int64_t s = t / k;
    const int j = (int)(t - s * k);
    const int32_t v = knn[t];
    out[(int64_t)perm[s] * k + j] = v >= 0 ? perm[v] : -1;
}

// Rows of one cloud of a batch, in that cloud's own original order and index space.
__global__ void __launch_bounds__(BLK) k_knn_original_cloud(const int32_t* __restrict__ knn,
                                                             const int32_t* __restrict__ perm, CloudDev c,
                                                             int64_t in_base, int32_t* __restrict__ out) {
    const int64_t t = (int64_t)blockIdx.x * BLK + threadIdx.x;
    if (t >= c.n * c.k) return;
    const int64_t r = t / c.k;
    const int j = (int)(t - r * c.k);
    const int32_t v = knn[c.row_off + t];
    const int64_t s = c.base + r;
    out[(perm[s] - in_base) * c.k + j] = v >= 0 ? (int32_t)(perm[c.base + v] - in_base) : -1;
}

int ilog2(int v) {
    int l = 0;
    while ((1 << l) < v) ++l;
    return l;
}

}  // namespace

namespace {

int ceil_log2(int64_t v) {
    int l = 0;
    while ((1ll << l) < v) ++l;
    return l;
}

// What a build tells the host, behind the level descriptors in one buffer, so that one copy brings it over: the count
// of non-finite input points, the cubes of the clouds, and per level the cell count and the running counts at each
// cloud's first position.
struct Report {
    int nc, nl;
    size_t bad() const { return EGT_MAX_LEVELS * sizeof(LevelDev) / sizeof(uint32_t); }
    size_t cubes() const { return bad() + 2; }
    size_t counts() const { return cubes() + 2 * (size_t)nc; }
    size_t words() const { return counts() + (size_t)nl * (nc + 1); }
    uint32_t* dev(egt_ctx* h) const {
        h->dlev.alloc((words() * sizeof(uint32_t) + sizeof(LevelDev) - 1) / sizeof(LevelDev));
        return reinterpret_cast<uint32_t*>(h->dlev.p);
    }
};
Report report_of(const egt_ctx* h) { return Report{h->nclouds, ilog2(h->B) + 1}; }

// Points of the largest cloud: where they fit a workgroup's sort, each cloud is sorted by one, in one launch (24 clouds
// of 38,000 points in all: 22 launches of passes over all points before).
int64_t max_cloud(const egt_ctx* h) {
    int64_t m = 0;
    for (const CloudDev& c : h->clouds) m = std::max(m, c.n);
    return m;
}

// Sort keys and values of the Morton order (buffers apart from those of the first sort).
MortonKeys morton_buffers(egt_ctx* h) {
    const int64_t n = h->n;
    Scratch& sc = h->scratch;
    const float a = -h->eps;
    return MortonKeys{a, (1.0f + h->eps) - a, h->B, ilog2(h->B), sc.get<uint32_t>(8, n), sc.get<uint32_t>(22, n),
                      sc.get<uint32_t>(10, n), sc.get<float4>(11, n)};
}

// Normalize, key, stable sort (by cloud, then key) and gather into sorted space. icloud is null for one
// cloud.
MortonKeys sort_into_sorted_space(egt_ctx* h, const float* dx, const float* dy, const float* dz, const int32_t* icloud) {
    const int64_t n = h->n;
    hipStream_t s = h->stream;
    Scratch& sc = h->scratch;
    const int log2B = ilog2(h->B);
    const float a = -h->eps, b = 1.0f + h->eps, ba = b - a;
    float4* tp = sc.get<float4>(9, n);
    uint32_t* skey = sc.get<uint32_t>(12, n);
    uint32_t* sidx = sc.get<uint32_t>(13, n);
    const Report R = report_of(h);
    k_normalize_key<<<ceil_div(n, BLK), BLK, 0, s>>>(dx, dy, dz, n, icloud, h->dclouds.p, R.dev(h) + R.bad(), a, ba,
                                                      h->B, log2B, tp, skey, sidx);
    LAUNCH_CHECK();
    const bool by_cloud = sort_segments(skey, sidx, max_cloud(h), 3 * log2B, icloud ? h->in_off.p : nullptr, h->nclouds,
                                        nullptr, 0, s);
    if (!by_cloud) radix_sort_pairs(skey, sidx, n, 3 * log2B, s, sc);
    if (icloud) h->scloud.alloc(n);
    if (icloud && !by_cloud) {
        // second stable pass by cloud: sorted by (cloud, key), ties in input order
        uint32_t* cl = sc.get<uint32_t>(22, n);
        k_gather_cloud<<<ceil_div(n, BLK), BLK, 0, s>>>(icloud, sidx, n, cl);
        LAUNCH_CHECK();
        radix_sort_pairs(cl, sidx, n, std::max(1, ceil_log2(h->nclouds)), s, sc, false);
    }
    h->x.alloc(n);
    h->y.alloc(n);
    h->z.alloc(n);
    h->perm.alloc(n);
    h->key.alloc(n);
    const MortonKeys K = morton_buffers(h);
    k_gather_sorted<<<ceil_div(n, BLK), BLK, 0, s>>>(tp, icloud, sidx, n, h->x.p, h->y.p, h->z.p, h->perm.p,
                                                      h->key.p, icloud ? h->scloud.p : nullptr, K);
    LAUNCH_CHECK();
    return K;
}

void check_finite(const egt_ctx* h, const std::vector<uint32_t>& rep) {
    if (rep[report_of(h).bad()]) throw ArgError{EGT_ERR_INVALID_ARG, "input coordinates contain NaN or Inf"};
}

// The host's cloud table: places and sizes, before a build, and the cubes from its report.
void place_clouds(egt_ctx* h, int nclouds, const int64_t* offsets) {
    h->nclouds = nclouds;
    h->clouds.assign(nclouds, CloudDev{});
    for (int c = 0; c < nclouds; ++c) {
        h->clouds[c].base = offsets[c];
        h->clouds[c].n = offsets[c + 1] - offsets[c];
    }
    h->dclouds.alloc(nclouds);
}
void set_cubes(egt_ctx* h, const std::vector<uint32_t>& rep) {
    const uint32_t* cube = rep.data() + report_of(h).cubes();
    for (int c = 0; c < h->nclouds; ++c) {
        float mm[2];
        std::memcpy(mm, cube + 2 * c, sizeof(mm));
        CloudDev& cd = h->clouds[c];
        cd.min_extent = mm[0];
        cd.extent = mm[1] - mm[0];
        cd.max_extent = mm[1];
    }
    h->min_extent = h->clouds[0].min_extent;
    h->max_extent = h->clouds[0].max_extent;
}

void build_search_structure(egt_ctx* h, const MortonKeys& K, std::vector<uint32_t>& rep, hipEvent_t done);

}  // namespace

void build_grid(egt_ctx* h, const float* dx, const float* dy, const float* dz) {
    const int64_t n = h->n;
    hipStream_t s = h->stream;
    Scratch& sc = h->scratch;
    Event e0, e1;
    HIP_CHECK(hipEventRecord(e0, s));

    // bounding cube
    const int64_t offsets[2] = {0, n};
    place_clouds(h, 1, offsets);
    const Report R = report_of(h);
    uint32_t* rep = R.dev(h);
    const int nbp = std::min<int64_t>(1024, std::max<int64_t>(1, ceil_div(n, BLK)));
    float* dpart = sc.get<float>(8, std::max<size_t>((size_t)nbp * MM_WORDS, n));  // the Morton keys' size
    k_minmax_partial<<<nbp, BLK, 0, s>>>(dx, dy, dz, n, dpart);
    LAUNCH_CHECK();
    k_cloud_cube<<<1, 64, 0, s>>>(dpart, nbp, n, h->dclouds.p, rep + R.bad(), rep + R.cubes());
    LAUNCH_CHECK();
    const MortonKeys K = sort_into_sorted_space(h, dx, dy, dz, nullptr);
    std::vector<uint32_t> hr;
    build_search_structure(h, K, hr, e1);
    set_cubes(h, hr);
    HIP_CHECK(hipEventElapsedTime(&h->stats.grid_ms, e0, e1));
}

void build_grid_batch(egt_ctx* h, const float* dx, const float* dy, const float* dz, const int64_t* offsets,
                      int nclouds) {
    const int64_t n = h->n;
    hipStream_t s = h->stream;
    Scratch& sc = h->scratch;
    Event e0, e1;
    HIP_CHECK(hipEventRecord(e0, s));
    place_clouds(h, nclouds, offsets);
    h->in_off.alloc(nclouds + 1);
    HIP_CHECK(hipMemcpyAsync(h->in_off.p, offsets, (nclouds + 1) * sizeof(int64_t), hipMemcpyHostToDevice, s));
    int32_t* icloud = sc.get<int32_t>(21, n);
    k_cloud_of<<<ceil_div(n, BLK), BLK, 0, s>>>(h->in_off.p, nclouds, n, icloud);
    LAUNCH_CHECK();
    const Report R = report_of(h);
    uint32_t* rep = R.dev(h);
    int* mm = sc.get<int>(8, std::max<size_t>((size_t)nclouds * 6, n));  // the Morton keys' size
    k_minmax_init<<<ceil_div(nclouds * 6, BLK), BLK, 0, s>>>(mm, nclouds, rep + R.bad());
    LAUNCH_CHECK();
    // one group a wave while that leaves few waves, then more groups and fewer sends
    const int groups = (int)std::min<int64_t>(16, std::max<int64_t>(1, n / ((int64_t)8192 * 64 * MM_ROUNDS)));
    k_cloud_minmax<<<ceil_div(n, (int64_t)BLK * MM_ROUNDS * groups), BLK, 0, s>>>(dx, dy, dz, icloud, n, groups, mm,
                                                                                 rep + R.bad());
    LAUNCH_CHECK();
    k_cloud_cubes<<<ceil_div(nclouds, BLK), BLK, 0, s>>>(mm, h->in_off.p, nclouds, h->dclouds.p, rep + R.cubes());
    LAUNCH_CHECK();
    const MortonKeys K = sort_into_sorted_space(h, dx, dy, dz, icloud);
    std::vector<uint32_t> hr;
    build_search_structure(h, K, hr, e1);
    set_cubes(h, hr);
    HIP_CHECK(hipEventElapsedTime(&h->stats.grid_ms, e0, e1));
}

namespace {
// The Morton order (from the sort keys K) and the level tables of the sorted points; rep: the report, done: recorded when the work is queued
// (if not null). Synchronizes the stream.
void build_search_structure(egt_ctx* h, const MortonKeys& K, std::vector<uint32_t>& rep, hipEvent_t done) {
    const int64_t n = h->n;
    hipStream_t s = h->stream;
    Scratch& sc = h->scratch;
    const int log2B = ilog2(h->B);
    const bool batch = h->nclouds > 1;
    uint32_t* order = K.idx;
    // Morton order of the fine cells, points of a cell in sub-code order: stable sort by sub code, then by cell code
    const bool by_cloud = sort_segments(K.sub, order, max_cloud(h), 3 * SUB, batch ? h->in_off.p : nullptr, h->nclouds,
                                        K.code, 3 * log2B, s);
    if (!by_cloud) {
        uint32_t* code = sc.get<uint32_t>(12, n);
        radix_sort_pairs(K.sub, order, n, 3 * SUB, s, sc, false);
        k_gather_u32<<<ceil_div(n, BLK), BLK, 0, s>>>(K.code, order, n, code);
        LAUNCH_CHECK();
        radix_sort_pairs(code, order, n, 3 * log2B, s, sc);
    }
    if (batch) h->mcloud.alloc(n);
    if (batch && !by_cloud) {
        // second stable pass by cloud: Morton order within each cloud, clouds in input order
        uint32_t* cl = sc.get<uint32_t>(22, n);
        k_gather_cloud<<<ceil_div(n, BLK), BLK, 0, s>>>(h->scloud.p, order, n, cl);
        LAUNCH_CHECK();
        radix_sort_pairs(cl, order, n, std::max(1, ceil_log2(h->nclouds)), s, sc, false);
    }
    h->mpts.alloc(n);
    h->mcell.alloc(n);
    h->mvcell.alloc(n);
    h->mcode.alloc(n);
    h->morder.alloc(n);
    h->minv.alloc(n);
    k_morton_points<<<ceil_div(n, BLK), BLK, 0, s>>>(K.spts, batch ? h->scloud.p : nullptr,
                                                      order, n, K.a, K.ba, h->B, log2B, h->mpts.p, h->mcell.p,
                                                      reinterpret_cast<unsigned long long*>(h->mvcell.p), h->mcode.p,
                                                      batch ? h->mcloud.p : nullptr, h->morder.p, h->minv.p);
    LAUNCH_CHECK();
    const int32_t* mcl = batch ? h->mcloud.p : nullptr;

    // level tables: every level's cells are counted, ranked and (below) inserted together
    const Report R = report_of(h);
    h->nlev = R.nl;
    const int nc = h->nclouds, nl = h->nlev;
    // room for the starts of every level: at most min(n, cells of the level's grid over all clouds) each
    std::vector<size_t> soff(nl + 1, 0);
    LevelStarts ls{};
    for (int l = 0; l < nl; ++l) {
        const double grid_cells = (double)nc * std::pow((double)(h->B >> l), 3.0);
        soff[l + 1] = soff[l] + (size_t)std::min<double>((double)n, grid_cells);
        ls.soff[l] = soff[l];
    }
    uint32_t* starts = sc.get<uint32_t>(38, soff[nl]);
    const int nb = ceil_div(n, LV_TILE);
    uint32_t* tiles = nb > 1 ? sc.get<uint32_t>(9, (size_t)nl * nb) : nullptr;
    uint32_t* drep = R.dev(h);
    uint32_t* dtot = drep + R.counts();  // per level: total, then the cloud bases
    if (nb > 1) {
        k_level_count<<<nb, BLK, 0, s>>>(h->mcode.p, mcl, n, nl, nb, tiles);
        LAUNCH_CHECK();
        k_level_scan<<<nl, LVS_BLK, 0, s>>>(tiles, nb, dtot, nc + 1);
        LAUNCH_CHECK();
    }
    k_level_starts<<<nb, BLK, 0, s>>>(h->mcode.p, mcl, n, nl, nb, tiles, ls, starts, dtot, nc + 1);
    LAUNCH_CHECK();
    // The tables are sized by the levels' cell counts, which takes one trip to the host, or, up to TABLE_BOUND cells,
    // by the bounds above, which takes none.
    rep.resize(R.words());
    auto read_back = [&](size_t words) {
        fetch(h->lane, {{rep.data(), drep, words * sizeof(uint32_t)}});
        check_finite(h, rep);
    };
    const bool by_bound = soff[nl] <= TABLE_BOUND;
    if (!by_bound) read_back(R.words());
    LevelInsert li{};
    li.nl = nl;
    for (int l = 0; l < nl; ++l) {
        const uint64_t cells = by_bound ? soff[l + 1] - soff[l] : rep[R.counts() + (size_t)l * (nc + 1)];
        // Twice the cells at least, and eight times on the coarse levels, whose tables are small beside the fine ones:
        // a wave's search waits for its longest probe chain. Search, us, twice everywhere -> eight times on coarse
        // levels: torus 1M k=16 1122 -> 1047, 16M k=40 32300 -> 31890; mixture 4M k=40 12976 -> 12776, 16M 57136 ->
        // 55434; builds unchanged (eight times on all levels: the same searches, builds 3-10% slower).
        // (A slot is a 32-bit number: beyond 2^28 cells there is no room for eight.)
        const uint64_t room = by_bound || 4 * cells > (uint64_t)n || cells > (1ull << 28) ? 2 : 8;
        uint32_t log2cap = 6;
        while ((1ull << log2cap) < room * cells) ++log2cap;
        h->lev[l].log2cap = li.log2cap[l] = log2cap;
        h->lev[l].offset = li.offset[l] = li.slots;
        li.first[l + 1] = li.first[l] + (int64_t)cells;
        li.soff[l] = soff[l];
        li.slots += 1ull << log2cap;
    }
    h->htab.alloc(li.slots);
    k_level_init<<<(int)std::min<uint64_t>(1024, (2 * li.slots + BLK - 1) / BLK), BLK, 0, s>>>(
        li, reinterpret_cast<uint64_t*>(h->htab.p), h->dlev.p);
    LAUNCH_CHECK();
    // (a batch of very many points has more cells, over all levels, than one launch takes threads)
    in_launches(ceil_div(li.first[nl], BLK), MAX_GROUPS, [&](int64_t first, int64_t groups) {
        k_level_insert<<<(unsigned)groups, BLK, 0, s>>>(li, starts, n, h->mcode.p, mcl, dtot, nc + 1, h->htab.p,
                                                        h->dlev.p, first);
        LAUNCH_CHECK();
    });
    if (done) HIP_CHECK(hipEventRecord(done, s));
    read_back(by_bound ? R.words() : R.bad() + 1);
    h->cloud_cells.assign((size_t)nc * nl, 0);
    for (int l = 0; l < nl; ++l) {
        const uint32_t* tl = &rep[R.counts() + (size_t)l * (nc + 1)];
        for (int c = 0; c < nc; ++c) {
            const uint32_t end = c + 1 < nc ? tl[1 + c + 1] : tl[0];
            h->cloud_cells[(size_t)c * nl + l] = end - (c > 0 ? tl[1 + c] : 0);
        }
        LevelDev d;
        std::memcpy(&d, &rep[l * (sizeof(LevelDev) / sizeof(uint32_t))], sizeof(d));
        h->lev[l].cells = tl[0];
        h->lev[l].max_count = d.max_count;
    }
}
}  // namespace

namespace {
__global__ void __launch_bounds__(BLK) k_rekey(const float* __restrict__ x, const float* __restrict__ y,
                                                const float* __restrict__ z, int64_t n, int32_t* __restrict__ key,
                                                MortonKeys K) {
    const int64_t s = (int64_t)blockIdx.x * BLK + threadIdx.x;
    if (s >= n) return;
    const float px = x[s], py = y[s], pz = z[s];
    const uint32_t cx = (uint32_t)cell_of(px, K.a, K.ba, K.B), cy = (uint32_t)cell_of(py, K.a, K.ba, K.B),
                   cz = (uint32_t)cell_of(pz, K.a, K.ba, K.B);
    const uint32_t k = cx | (cy << K.log2B) | (cz << (2 * K.log2B));
    key[s] = (int32_t)k;
    morton_keys(K, s, px, py, pz, k);
}
}  // namespace

// After smoothing moved the points: recompute each point's fine cell and rebuild the Morton search
// structure (the sorted-space order itself is kept).
void refresh_search_structure(egt_ctx* h) {
    const MortonKeys K = morton_buffers(h);
    k_rekey<<<ceil_div(h->n, BLK), BLK, 0, h->stream>>>(h->x.p, h->y.p, h->z.p, h->n, h->key.p, K);
    LAUNCH_CHECK();
    std::vector<uint32_t> rep;
    build_search_structure(h, K, rep, nullptr);
    h->search_stale = false;
}

void run_output(egt_ctx* h, float* x, float* y, float* z) {
    const int64_t n = h->n;
    hipStream_t s = h->stream;
    float* ox = h->scratch.get<float>(9, 3 * n);
    k_output<<<ceil_div(n, BLK), BLK, 0, s>>>(h->x.p, h->y.p, h->z.p, h->perm.p,
                                              h->nclouds > 1 ? h->scloud.p : nullptr, h->dclouds.p, n,
                                              h->min_extent, h->max_extent - h->min_extent, ox, ox + n, ox + 2 * n);
    LAUNCH_CHECK();
    const size_t bytes = n * sizeof(float);
    fetch(h->lane, {{x, ox, bytes}, {y, ox + n, bytes}, {z, ox + 2 * n, bytes}});
}

void run_knn_original(egt_ctx* h, int32_t* out) {
    const int64_t n = h->n, k = h->k;
    hipStream_t s = h->stream;
    int32_t* tmp = h->scratch.get<int32_t>(9, n * k);
    k_knn_original<<<ceil_div(n * k, BLK), BLK, 0, s>>>(h->knn.p, h->perm.p, n, (int)k, tmp);
    LAUNCH_CHECK();
    fetch(h->lane, {{out, tmp, n * k * sizeof(int32_t)}});
}

void run_knn_original_cloud(egt_ctx* h, int cloud, int32_t* out) {
    const CloudDev& c = h->clouds[cloud];
    hipStream_t s = h->stream;
    const int64_t cnt = c.n * c.k;
    int32_t* tmp = h->scratch.get<int32_t>(9, std::max<int64_t>(cnt, 1));
    k_knn_original_cloud<<<std::max(1, ceil_div(cnt, BLK)), BLK, 0, s>>>(h->knn.p, h->perm.p, c, c.base, tmp);
    LAUNCH_CHECK();
    fetch(h->lane, {{out, tmp, cnt * sizeof(int32_t)}});
}

uint32_t morton3(uint32_t x, uint32_t y, uint32_t z) { return morton_code(x, y, z); }

}  // namespace egt
