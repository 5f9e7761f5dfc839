// PCA normals and their orientation over a minimum spanning forest of the neighbour graph.
//
// Reference: Normal_CUDA::GetNormals Normal_CUDA.cu:304-775 with calculateNormal :87-144, getEdgeNumber /
// fillEdges :61-85, :146-175, mst() CUDA_MST.cu:423-460 (Boruvka), BFS bfs.cu:63-111 (sign propagation).
//
// 1. PCA: one thread per point; centroid of the point and its neighbours, covariance of the neighbours,
//    eigenvector of the smallest eigenvalue by cyclic Jacobi (egt_device.h).
// 2. Edges: every undirected edge {u < v} of the rows once, in (u, v) order: row u owns it when it lists v,
//    otherwise row v does; per-u buckets come from a counting pass + prefix sum and are sorted by v.
//    Weight max(0, 1 - |n_u . n_v|); edge key = (weight bits << 32) | edge id, a total order equal to
//    (weight, u, v).
// 3. Boruvka with parity: each component takes its minimum-key edge; mutual pairs keep the smaller id as
//    root; hooks carry the parity bit par(u) ^ par(v) ^ (n_u . n_v < 0); pointer jumping on packed
//    (target << 1 | parity) words resolves roots and parities. The forest is the unique minimum spanning
//    forest under the key order.
// 4. Orientation: each tree's root is u of its lightest edge; a vertex flips when its parity differs from
//    the root's, which equals the reference's BFS rule "flip the child when n_parent . n_child < 0".
#include <algorithm>
#include "egt_device.h"
#include "egt_internal.h"

namespace egt {
namespace {

constexpr int NBLK = 256;
constexpr uint64_t KEY_EMPTY = ~0ull;

// One thread per Morton position; neighbours from the Morton-order CSR (slot order of the rows), points
// from the Morton float4 copy. Writes the normal of sorted point s = mpts[m].w. The neighbour loops fetch four
// neighbours at a time (indices clamped to the row, so every load is valid) and add them in slot order.
__global__ void __launch_bounds__(NBLK) k_pca(const float4* __restrict__ mpts, const int32_t* __restrict__ rowptr,
                                               const int32_t* __restrict__ col, int64_t n, float* __restrict__ nx,
                                               float* __restrict__ ny, float* __restrict__ nz) {
    const int64_t m = (int64_t)blockIdx.x * NBLK + threadIdx.x;
    if (m >= n) return;
    const float4 p = mpts[m];
    const int32_t i = __float_as_int(p.w);
    const int32_t e0 = rowptr[m], e1 = rowptr[m + 1];
    float sx = p.x, sy = p.y, sz = p.z;
    int counter = 1;
    for (int32_t e = e0; e < e1; e += 4) {
        float4 q[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) q[u] = mpts[col[min(e + u, e1 - 1)]];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if (e + u < e1) {
                sx += q[u].x;
                sy += q[u].y;
                sz += q[u].z;
                ++counter;
            }
        }
    }
    const float cx = sx / (float)counter, cy = sy / (float)counter, cz = sz / (float)counter;
    float a00 = 0, a01 = 0, a02 = 0, a11 = 0, a12 = 0, a22 = 0;
    for (int32_t e = e0; e < e1; e += 4) {
        float4 q[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) q[u] = mpts[col[min(e + u, e1 - 1)]];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if (e + u < e1) {
                const float dx = q[u].x - cx, dy = q[u].y - cy, dz = q[u].z - cz;
                a00 = __builtin_fmaf(dx, dx, a00);
                a01 = __builtin_fmaf(dx, dy, a01);
                a02 = __builtin_fmaf(dx, dz, a02);
                a11 = __builtin_fmaf(dy, dy, a11);
                a12 = __builtin_fmaf(dy, dz, a12);
                a22 = __builtin_fmaf(dz, dz, a22);
            }
        }
    }
    float vx, vy, vz;
    eig3_smallest(a00, a01, a02, a11, a12, a22, vx, vy, vz);
    const float nrm = __builtin_sqrtf(__builtin_fmaf(vz, vz, __builtin_fmaf(vy, vy, vx * vx)));
    nx[i] = vx / nrm;
    ny[i] = vy / nrm;
    nz[i] = vz / nrm;
}

// pass 0: count per owner u and record which CSR entries emit an edge; pass 1: write v into u's bucket.
// Walks the Morton-order CSR (the same rows as the sorted-space neighbour lists, holes removed). Entry (i, nb)
// emits the edge {i, nb} when i < nb, or when i > nb and row nb does not list i (pass 0 scans nb's compact
// CSR row for that and stores the answer in own[], which pass 1 reads). Edges with u = i go to the row's own
// bucket: one atomic per row reserves them (order within a bucket is free: k_edge_sort sorts it; pass 0 keeps
// their count per row in lcount[]); only the edges owned by another row (u = nb) take an atomic each.
// EDGE_LANES lanes share a row, entry by entry: a row's scans of other rows are chains of three dependent loads, and a
// thread a row ran about four of them one after the other. Normals with 1 / 4 / 8 lanes: 4M-point torus 6.83 / 6.36 /
// 6.42 ms, cluster mixture 8.23 / 7.68 / 7.71, 100,000 points 0.39 / 0.38 / 0.40.
constexpr int EDGE_LANES = 4;
template <int PASS>
__global__ void __launch_bounds__(NBLK) k_edges(const int32_t* __restrict__ rowptr, const int32_t* __restrict__ col,
                                                 const int32_t* __restrict__ morder, int64_t n,
                                                 uint32_t* __restrict__ cnt, uint8_t* __restrict__ own,
                                                 uint8_t* __restrict__ lcount, int32_t* __restrict__ ev,
                                                 int64_t first_group) {
    const int64_t m = ((first_group + blockIdx.x) * NBLK + threadIdx.x) / EDGE_LANES;
    const int r = (int)threadIdx.x % EDGE_LANES, g0 = (__lane_id() / EDGE_LANES) * EDGE_LANES;
    const bool row = m < n;
    const int32_t i = row ? morder[m] : 0;
    const int32_t e0 = row ? rowptr[m] : 0, len = row ? rowptr[m + 1] - e0 : 0;
    // the lanes' flags of one row, as a mask of EDGE_LANES bits
    auto row_mask = [&](bool f) { return (uint32_t)(__ballot(f) >> g0) & ((1u << EDGE_LANES) - 1u); };
    if (PASS == 0) {
        uint32_t local = 0;  // edges of this row with u = i
        for (int b = 0; __ballot(b < len); b += EDGE_LANES) {
            const bool act = b + r < len;
            bool emit = false, mine = false;
            if (act) {
                const int32_t m2 = col[e0 + b + r], nb = morder[m2];
                emit = nb != i;
                mine = emit && nb > i;
                if (emit && !mine) {
                    bool listed = false;  // does row nb list i? then row nb owns the edge
                    const int32_t f1 = rowptr[m2 + 1];
                    for (int32_t f = rowptr[m2]; f < f1; f += 4) {
                        int32_t c4[4];
#pragma unroll
                        for (int v = 0; v < 4; ++v) c4[v] = col[min(f + v, f1 - 1)];
#pragma unroll
                        for (int v = 0; v < 4; ++v) listed = listed || c4[v] == (int32_t)m;
                    }
                    emit = !listed;
                    if (emit) atomicAdd(&cnt[nb], 1u);
                }
                own[e0 + b + r] = emit ? 1 : 0;
            }
            local += (uint32_t)__popc(row_mask(mine));
        }
        if (row && r == 0) {
            lcount[m] = (uint8_t)local;  // a row has at most 64 entries
            if (local) atomicAdd(&cnt[i], local);
        }
    } else {
        const uint32_t local = row ? lcount[m] : 0u;
        uint32_t p = r == 0 && local ? atomicAdd(&cnt[i], local) : 0u;
        p = __shfl(p, g0, 64);
        for (int b = 0; __ballot(b < len); b += EDGE_LANES) {
            const int32_t e = e0 + b + r;
            const bool ow = b + r < len && own[e];
            const int32_t nb = ow ? morder[col[e]] : i;
            const uint32_t mask = row_mask(nb > i);
            if (nb > i) ev[p + __popc(mask & ((1u << r) - 1u))] = nb;
            else if (ow) ev[atomicAdd(&cnt[nb], 1u)] = i;
            p += (uint32_t)__popc(mask);
        }
    }
}

__global__ void __launch_bounds__(NBLK) k_edge_sort(const uint32_t* __restrict__ off, int64_t n,
                                                     const uint32_t* __restrict__ m,
                                                     int32_t* __restrict__ ev, int32_t* __restrict__ eu) {
    const int64_t u = (int64_t)blockIdx.x * NBLK + threadIdx.x;
    if (u >= n) return;
    const uint32_t b = off[u], e = u + 1 < n ? off[u + 1] : *m;
    if (e - b <= 16) {  // the common case: sorted in registers by a 16-wide bitonic network, padded with INT_MAX
        int32_t r[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) r[i] = b + i < e ? ev[b + i] : INT32_MAX;
#pragma unroll
        for (int k = 2; k <= 16; k <<= 1) {
#pragma unroll
            for (int j = k >> 1; j > 0; j >>= 1) {
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const int l = i ^ j;
                    if (l > i) {
                        const int32_t x = r[i], y = r[l];
                        const bool up = (i & k) == 0;
                        r[i] = up ? min(x, y) : max(x, y);
                        r[l] = up ? max(x, y) : min(x, y);
                    }
                }
            }
        }
#pragma unroll
        for (int i = 0; i < 16; ++i)
            if (b + i < e) {
                ev[b + i] = r[i];
                eu[b + i] = (int32_t)u;
            }
        return;
    }
    for (uint32_t a = b + 1; a < e; ++a) {  // insertion sort of the bucket by v
        const int32_t t = ev[a];
        uint32_t c = a;
        while (c > b && ev[c - 1] > t) {
            ev[c] = ev[c - 1];
            --c;
        }
        ev[c] = t;
    }
    for (uint32_t a = b; a < e; ++a) eu[a] = (int32_t)u;
}

__global__ void __launch_bounds__(NBLK) k_edge_attr(const int32_t* __restrict__ eu, const int32_t* __restrict__ ev,
                                                     const uint32_t* __restrict__ m, const float* __restrict__ nx,
                                                     const float* __restrict__ ny, const float* __restrict__ nz,
                                                     uint64_t* __restrict__ ekey, uint8_t* __restrict__ erel,
                                                     float* __restrict__ ew) {
    const uint32_t e = blockIdx.x * NBLK + threadIdx.x;
    if (e >= *m) return;
    const int32_t u = eu[e], v = ev[e];
    const float dot = __builtin_fmaf(nz[u], nz[v], __builtin_fmaf(ny[u], ny[v], nx[u] * nx[v]));
    const float w = fmaxf(0.0f, 1.0f - __builtin_fabsf(dot));
    ew[e] = w;
    ekey[e] = ((uint64_t)__float_as_uint(w) << 32) | e;
    erel[e] = dot < 0.0f ? 1 : 0;
}

// Every vertex its own root. H (hook word: target << 1 | parity) is only ever read for roots, and a root's word
// stays its own until it hooks, so it is set once.
__global__ void __launch_bounds__(NBLK) k_bv_init(int64_t n, int32_t* __restrict__ comp, uint8_t* __restrict__ par,
                                                   uint64_t* __restrict__ best, uint64_t* __restrict__ tmin,
                                                   uint32_t* __restrict__ H, uint32_t* __restrict__ state, uint32_t m) {
    const int64_t v = (int64_t)blockIdx.x * NBLK + threadIdx.x;
    if (v < 4) state[v] = v == 2 ? m : 0u;
    if (v >= n) return;
    comp[v] = (int32_t)v;
    par[v] = 0;
    best[v] = KEY_EMPTY;
    tmin[v] = KEY_EMPTY;
    H[v] = (uint32_t)v << 1;
}

// atomicMin(base[idx], val) for the active lanes of a wave. Edges come in edge-id order, so lanes that share
// an endpoint's component often form runs: when a wave has any, a segmented inclusive min-scan over the lanes
// (log2(64) steps, a step merging the lane d below when it has the same target) leaves each run's minimum in
// its last lane, the only one of the run still to issue. Lanes that share a target without being adjacent may
// merge too, which is harmless: their values go to the same address. Late in Boruvka most edges join a few
// large components, so the remaining lanes often share a few targets without being adjacent: the target of
// the first remaining lane is then reduced over the wave and issued once, for up to 4 targets, as long as
// each is shared by at least two lanes; the rest issue their own atomics. Call from all lanes.
__device__ inline void wave_atomic_min(uint64_t* base, int32_t idx, uint64_t val, bool active) {
    const int lane = __lane_id();
    // A value that cannot lower the one already there (which only ever falls) needs no atomic: normals of a 4M-point
    // torus 8.3 -> 6.9 ms, of a 4M-point cluster mixture 10.9 -> 8.3.
    active = active && val < __hip_atomic_load(&base[idx], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const int32_t k = active ? idx : -1 - lane;  // inactive lanes: distinct keys that match no target
    unsigned long long v = active ? (unsigned long long)val : ~0ull;
    bool issue = active;
    const int32_t kp = __shfl_up(k, 1, 64);
    if (__ballot(active && lane > 0 && kp == k) != 0) {
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int32_t ok = __shfl_up(k, d, 64);
            const unsigned long long ov = __shfl_up(v, d, 64);
            if (lane >= d && ok == k && ov < v) v = ov;
        }
        const int32_t kn = __shfl_down(k, 1, 64);
        issue = active && (lane == 63 || kn != k);
    }
    for (int r = 0; r < 4; ++r) {
        const uint64_t amask = __ballot(issue);
        if (!amask) return;
        const int leader = __ffsll((unsigned long long)amask) - 1;
        const int32_t lk = __shfl(k, leader, 64);
        const bool mine = issue && k == lk;
        if (__popcll(__ballot(mine)) < 2) break;
        unsigned long long t = mine ? v : ~0ull;
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) {
            const unsigned long long o = __shfl_xor(t, d, 64);
            t = o < t ? o : t;
        }
        if (lane == leader) atomicMin((unsigned long long*)&base[lk], t);
        issue = issue && !mine;
    }
    if (issue) atomicMin((unsigned long long*)&base[idx], v);
}

// Block-level variant: when all active lanes of the block target one address, one atomic per block.
__device__ inline void block_atomic_min(uint64_t* base, int32_t idx, uint64_t val, bool active) {
    __shared__ int32_t widx[NBLK / 64];
    __shared__ unsigned long long wval[NBLK / 64];
    __shared__ int wstate[NBLK / 64];  // 0 idle, 1 uniform, 2 mixed
    const int wid = threadIdx.x / 64;
    const uint64_t amask = __ballot(active);
    int state = 0;
    int32_t lidx = 0;
    unsigned long long v = ~0ull;
    if (amask) {
        const int leader = __ffsll((unsigned long long)amask) - 1;
        lidx = __shfl(idx, leader, 64);
        state = __ballot(active && idx != lidx) == 0 ? 1 : 2;
        v = active ? (unsigned long long)val : ~0ull;
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) {
            const unsigned long long o = __shfl_xor(v, d, 64);
            v = o < v ? o : v;
        }
    }
    if (__lane_id() == 0) {
        widx[wid] = lidx;
        wval[wid] = v;
        wstate[wid] = state;
    }
    __syncthreads();
    if (state == 2 && active) atomicMin((unsigned long long*)&base[idx], (unsigned long long)val);
    if (threadIdx.x == 0) {
        bool all_same = true;
        int32_t bidx = -1;
        unsigned long long bv = ~0ull;
        for (int w = 0; w < NBLK / 64; ++w) {
            if (wstate[w] != 1) continue;
            if (bidx < 0) bidx = widx[w];
            if (widx[w] != bidx) all_same = false;
            bv = wval[w] < bv ? wval[w] : bv;
        }
        if (bidx >= 0) {
            if (all_same) {
                atomicMin((unsigned long long*)&base[bidx], bv);
            } else {
                for (int w = 0; w < NBLK / 64; ++w)
                    if (wstate[w] == 1) atomicMin((unsigned long long*)&base[widx[w]], wval[w]);
            }
        }
    }
}

// The alive-edge count is read from device memory (*mcount). The edge kernels of a round loop over it with a
// grid capped at BV_GRID blocks, so a round with few edges left costs a few microseconds, not a launch over
// the host's stale bound.
// After the first round the alive edges are 16-byte records of their key (whose low word is the edge) and the roots at
// their ends, which the merge that keeps them knows: a round then reads each edge in one piece, where an index into
// the edge arrays led to five more reads, two of them random. Normals of a
// torus / a cluster mixture: 100,000 points 0.38 -> 0.34 ms, 1M 1.45 -> 1.40, 4M 6.37 -> 6.07 / 7.71 -> 7.24.
constexpr int BV_GRID = 4096;
__device__ inline uint4 bv_record(const uint4* __restrict__ alive, uint32_t t, const int32_t* __restrict__ eu,
                                  const int32_t* __restrict__ ev, const uint64_t* __restrict__ ekey) {
    if (alive) return alive[t];
    const uint64_t key = ekey[t];  // first round: every vertex is its own root
    return make_uint4((uint32_t)key, (uint32_t)(key >> 32), (uint32_t)eu[t], (uint32_t)ev[t]);
}
__global__ void __launch_bounds__(NBLK) k_bv_best(const int32_t* __restrict__ eu, const int32_t* __restrict__ ev,
                                                   const uint64_t* __restrict__ ekey, const uint4* __restrict__ alive,
                                                   const uint32_t* __restrict__ mcount, uint64_t* __restrict__ best) {
    const uint32_t m = *mcount;
    for (uint32_t t0 = blockIdx.x * NBLK; t0 < m; t0 += gridDim.x * NBLK) {  // block-uniform bound
        const uint32_t t = t0 + threadIdx.x;
        int32_t cu = 0, cv = 0;
        uint64_t key = 0;
        bool act = t < m;
        if (act) {
            const uint4 a = bv_record(alive, t, eu, ev, ekey);
            cu = (int32_t)a.z;
            cv = (int32_t)a.w;
            act = cu != cv;
            key = ((uint64_t)a.y << 32) | a.x;
        }
        wave_atomic_min(best, cu, key, act);
        wave_atomic_min(best, cv, key, act);
    }
}

// Hooks every root with a lightest edge to the root at the edge's other end. No hook count is kept: a round
// hooks at least one root exactly when edges between components are alive at its start, which the alive-edge
// count already tells (a shared counter took one atomic per wave on one address, about 0.7 ms a round on a
// 4M-point cloud).
__global__ void __launch_bounds__(NBLK) k_bv_hook(int64_t n, const int32_t* __restrict__ eu,
                                                   const int32_t* __restrict__ ev, const uint8_t* __restrict__ erel,
                                                   const int32_t* __restrict__ comp, const uint8_t* __restrict__ par,
                                                   const uint64_t* __restrict__ best, uint32_t* __restrict__ H,
                                                   uint8_t* __restrict__ msf, uint64_t* __restrict__ best1,
                                                   uint32_t* __restrict__ next_count) {
    const int64_t c = (int64_t)blockIdx.x * NBLK + threadIdx.x;
    if (c == 0) *next_count = 0;
    if (best1 && c < n) best1[c] = best[c];  // first round: every vertex's lightest edge
    if (c < n && comp[c] == c) {
        const uint64_t b = best[c];
        if (b != KEY_EMPTY) {
            const uint32_t e = (uint32_t)b;
            const int32_t u = eu[e], v = ev[e];
            const int32_t cu = comp[u], cv = comp[v];
            const int32_t other = cu == (int32_t)c ? cv : cu;
            if (!(best[other] == b && (int32_t)c < other)) {  // mutual pair: the smaller id stays root
                H[c] = ((uint32_t)other << 1) | (uint32_t)(par[u] ^ par[v] ^ erel[e]);
                msf[e] = 1;
            }
        }
    }
}

// Follows hook pointers to the root. The hook graph is a forest (edge keys are a strict total order and
// mutual pairs keep one root), so every walk ends; the walk is still capped at n steps and a cap hit is
// reported through *overflow instead of spinning.
__global__ void __launch_bounds__(NBLK) k_bv_jump(int64_t n, const int32_t* __restrict__ comp,
                                                   uint32_t* __restrict__ H, uint32_t* __restrict__ overflow) {
    const int64_t c = (int64_t)blockIdx.x * NBLK + threadIdx.x;
    if (c >= n || comp[c] != c) return;
    uint32_t w = H[c];
    int64_t steps = 0;
    for (;;) {
        const uint32_t t = w >> 1;
        const uint32_t w2 = __hip_atomic_load(&H[t], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if ((w2 >> 1) == t) break;
        w = (w2 & ~1u) | ((w ^ w2) & 1u);
        if (++steps > n) {
            atomicAdd(overflow, 1u);
            break;
        }
    }
    __hip_atomic_store(&H[c], w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Relabels every vertex to its new root and keeps the edges that still join two components (the rest can never be
// chosen again) for the next round, with their new roots. The edge half does not wait for the vertex half: H leads
// from an old root to the new one. A workgroup filters BV_CHUNK edges
// at a time and reserves its place in the output with one atomic, so the kept edges stay in id order within a
// chunk only; the minima do not depend on the order, and runs of equal endpoints survive.
constexpr int BV_CHUNK = 8 * NBLK;
__global__ void __launch_bounds__(NBLK) k_bv_merge(int64_t n, int32_t* __restrict__ comp, uint8_t* __restrict__ par,
                                                    const uint32_t* __restrict__ H, uint64_t* __restrict__ best,
                                                    const int32_t* __restrict__ eu, const int32_t* __restrict__ ev,
                                                    const uint64_t* __restrict__ ekey, const uint4* __restrict__ alive,
                                                    const uint32_t* __restrict__ mcount, uint4* __restrict__ out,
                                                    uint32_t* __restrict__ out_count, int vblocks) {
    __shared__ uint32_t wcount[NBLK / 64][8];
    __shared__ uint32_t base;
    if ((int)blockIdx.x < vblocks) {
        const int64_t v = (int64_t)blockIdx.x * NBLK + threadIdx.x;
        if (v >= n) return;
        const uint32_t w = H[comp[v]];
        const int32_t root = (int32_t)(w >> 1);
        comp[v] = root;
        par[v] ^= (uint8_t)(w & 1u);
        if (root == (int32_t)v) best[v] = KEY_EMPTY;
        return;
    }
    const uint32_t m = *mcount;
    const int lane = __lane_id(), wid = threadIdx.x / 64;
    const uint32_t nblk = gridDim.x - (uint32_t)vblocks;
    for (uint32_t t0 = (blockIdx.x - (uint32_t)vblocks) * BV_CHUNK; t0 < m; t0 += nblk * BV_CHUNK) {
        uint4 ed[8];
        uint64_t keep[8];
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            const uint32_t t = t0 + r * NBLK + threadIdx.x;
            ed[r] = bv_record(alive, min(t, m - 1), eu, ev, ekey);
        }
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            const uint32_t t = t0 + r * NBLK + threadIdx.x;
            ed[r].z = H[ed[r].z] >> 1;
            ed[r].w = H[ed[r].w] >> 1;
            const bool k = t < m && ed[r].z != ed[r].w;
            keep[r] = __ballot(k);
            if (lane == 0) wcount[wid][r] = (uint32_t)__popcll(keep[r]);
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            uint32_t run = 0;
            for (int r = 0; r < 8; ++r)
                for (int w = 0; w < NBLK / 64; ++w) {
                    const uint32_t c = wcount[w][r];
                    wcount[w][r] = run;
                    run += c;
                }
            base = run ? atomicAdd(out_count, run) : 0u;
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < 8; ++r)
            if ((keep[r] >> lane) & 1ull)
                out[base + wcount[wid][r] + (uint32_t)__popcll(keep[r] & ((1ull << lane) - 1ull))] = ed[r];
        __syncthreads();
    }
}

// Lightest edge of each tree = minimum over its vertices of their lightest incident edge (round-1 best).
__global__ void __launch_bounds__(NBLK) k_tree_min(int64_t n, const int32_t* __restrict__ comp,
                                                    const uint64_t* __restrict__ best1, uint64_t* __restrict__ tmin) {
    const int64_t v = (int64_t)blockIdx.x * NBLK + threadIdx.x;
    const bool act = v < n && best1[v] != KEY_EMPTY;
    block_atomic_min(tmin, act ? comp[v] : 0, act ? best1[v] : 0ull, act);
}

__global__ void __launch_bounds__(NBLK) k_orient(int64_t n, const int32_t* __restrict__ comp,
                                                  const uint8_t* __restrict__ par, const uint64_t* __restrict__ tmin,
                                                  const int32_t* __restrict__ eu, float* __restrict__ nx,
                                                  float* __restrict__ ny, float* __restrict__ nz) {
    const int64_t v = (int64_t)blockIdx.x * NBLK + threadIdx.x;
    if (v >= n) return;
    const uint64_t t = tmin[comp[v]];
    if (t == KEY_EMPTY) return;
    const int32_t root = eu[(uint32_t)t];
    if (par[v] ^ par[root]) {
        nx[v] = -nx[v];
        ny[v] = -ny[v];
        nz[v] = -nz[v];
    }
}

// The whole forest and orientation of a small cloud in one workgroup: components, hook words and lightest edges in
// LDS, every round over all edges. A round in launches is four of them (ten before, with a wait every second
// round), a few us each whatever they do: GetNormals' device time 0.48 -> 0.10 ms at 1,500 points, 0.66 -> 0.27 at
// 8,192; with four launches a round 0.68 -> 0.33 at 20,000, 1.92 -> 1.55 at 1M.
constexpr int BVS_BLOCK = 1024, BVS_PER = 8, BVS_MAX = BVS_BLOCK * BVS_PER;  // vertices
constexpr size_t bvs_lds(int64_t n) { return (size_t)n * (sizeof(uint64_t) + 2 * sizeof(uint32_t)); }
__global__ void __launch_bounds__(BVS_BLOCK) k_bv_small(int n, const uint32_t* __restrict__ mcount,
                                                         const int32_t* __restrict__ eu,
                                                         const int32_t* __restrict__ ev,
                                                         const uint64_t* __restrict__ ekey,
                                                         const uint8_t* __restrict__ erel, uint8_t* __restrict__ msf,
                                                         float* __restrict__ nx, float* __restrict__ ny,
                                                         float* __restrict__ nz, uint32_t* __restrict__ trees) {
    extern __shared__ uint64_t lds[];
    const uint32_t m = *mcount;
    uint64_t* best = lds;
    uint32_t* comp = reinterpret_cast<uint32_t*>(lds + n);  // root << 1 | parity to it
    uint32_t* H = comp + n;                                 // hook word of a root: target << 1 | parity
    __shared__ uint32_t alive, ntrees;
    const int tid = threadIdx.x;
    uint64_t first[BVS_PER];  // the vertex's lightest edge
#pragma unroll
    for (int i = 0; i < BVS_PER; ++i) {
        const int v = tid + i * BVS_BLOCK;
        first[i] = KEY_EMPTY;
        if (v < n) {
            comp[v] = (uint32_t)v << 1;
            H[v] = (uint32_t)v << 1;
            best[v] = KEY_EMPTY;
        }
    }
    for (uint32_t e = tid; e < m; e += BVS_BLOCK) msf[e] = 0;
    if (tid == 0) ntrees = 0;
    for (int round = 0; round < 64; ++round) {
        if (tid == 0) alive = 0;
        __syncthreads();
        bool any = false;
        for (uint32_t e = tid; e < m; e += BVS_BLOCK) {
            const uint32_t cu = comp[eu[e]] >> 1, cv = comp[ev[e]] >> 1;
            if (cu == cv) continue;
            any = true;
            const unsigned long long k = ekey[e];
            for (const uint32_t c : {cu, cv})
                if (k < __hip_atomic_load(&best[c], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP))
                    atomicMin((unsigned long long*)&best[c], k);
        }
        if (any) alive = 1;
        __syncthreads();
        if (!alive) break;
        uint32_t w[BVS_PER];
#pragma unroll
        for (int i = 0; i < BVS_PER; ++i) {  // hook
            const int c = tid + i * BVS_BLOCK;
            if (c >= n || comp[c] >> 1 != (uint32_t)c) continue;
            const uint64_t b = best[c];
            if (round == 0) first[i] = b;
            if (b == KEY_EMPTY) continue;
            const uint32_t e = (uint32_t)b;
            const uint32_t wu = comp[eu[e]], wv = comp[ev[e]];
            const uint32_t other = wu >> 1 == (uint32_t)c ? wv >> 1 : wu >> 1;
            if (!(best[other] == b && (uint32_t)c < other)) {  // mutual pair: the smaller id stays root
                H[c] = (other << 1) | ((wu ^ wv ^ (uint32_t)erel[e]) & 1u);
                msf[e] = 1;
            }
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < BVS_PER; ++i) {  // follow the hooks; the hook graph is a forest, a walk has at most n steps
            const int c = tid + i * BVS_BLOCK;
            w[i] = 0;
            if (c >= n || comp[c] >> 1 != (uint32_t)c) continue;
            w[i] = H[c];
            for (int step = 0; step < n; ++step) {
                const uint32_t t = w[i] >> 1, w2 = H[t];
                if (w2 >> 1 == t) break;
                w[i] = (w2 & ~1u) | ((w[i] ^ w2) & 1u);
            }
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < BVS_PER; ++i) {
            const int c = tid + i * BVS_BLOCK;
            if (c < n && comp[c] >> 1 == (uint32_t)c) H[c] = w[i];
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < BVS_PER; ++i) {  // relabel (every lane its own vertices)
            const int v = tid + i * BVS_BLOCK;
            if (v >= n) continue;
            const uint32_t h = H[comp[v] >> 1];
            comp[v] = (h & ~1u) | ((comp[v] ^ h) & 1u);
            best[v] = KEY_EMPTY;
        }
        __syncthreads();
    }
    // orientation: the root of a tree is u of its lightest edge
#pragma unroll
    for (int i = 0; i < BVS_PER; ++i) {
        const int v = tid + i * BVS_BLOCK;
        if (v < n) best[v] = KEY_EMPTY;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < BVS_PER; ++i) {
        const int v = tid + i * BVS_BLOCK;
        if (v < n && first[i] != KEY_EMPTY) atomicMin((unsigned long long*)&best[comp[v] >> 1], first[i]);
    }
    __syncthreads();
    uint32_t roots = 0;
#pragma unroll
    for (int i = 0; i < BVS_PER; ++i) {
        const int v = tid + i * BVS_BLOCK;
        if (v >= n) continue;
        const uint64_t t = best[comp[v] >> 1];
        if (t == KEY_EMPTY) continue;
        roots += comp[v] >> 1 == (uint32_t)v ? 1u : 0u;
        if ((comp[v] ^ comp[eu[(uint32_t)t]]) & 1u) {
            nx[v] = -nx[v];
            ny[v] = -ny[v];
            nz[v] = -nz[v];
        }
    }
    if (roots) atomicAdd(&ntrees, roots);
    __syncthreads();
    if (tid == 0) *trees = ntrees;
}

// deterministic forest statistics: per-block partial sums, summed on the host in block order
__global__ void __launch_bounds__(NBLK) k_msf_stats(const uint8_t* __restrict__ msf, const float* __restrict__ ew,
                                                     const uint32_t* __restrict__ mcount, double* __restrict__ part_w,
                                                     uint32_t* __restrict__ part_c) {
    __shared__ double sw[NBLK];
    __shared__ uint32_t scnt[NBLK];
    double w = 0.0;
    uint32_t c = 0;
    // as many blocks as the edges fill, whatever the launch allowed for: the partial sums stay the same
    const uint32_t m = *mcount, stride = min(gridDim.x, max(1u, (m + NBLK - 1) / NBLK)) * NBLK;
    for (uint32_t e = blockIdx.x * NBLK + threadIdx.x; e < m && blockIdx.x * NBLK < stride; e += stride)
        if (msf[e]) {
            w += (double)ew[e];
            ++c;
        }
    sw[threadIdx.x] = w;
    scnt[threadIdx.x] = c;
    __syncthreads();
    for (int s = NBLK / 2; s > 0; s >>= 1) {
        if (threadIdx.x < s) {
            sw[threadIdx.x] += sw[threadIdx.x + s];
            scnt[threadIdx.x] += scnt[threadIdx.x + s];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        part_w[blockIdx.x] = sw[0];
        part_c[blockIdx.x] = scnt[0];
    }
}

__global__ void __launch_bounds__(NBLK) k_count_roots(int64_t n, const int32_t* __restrict__ comp,
                                                       const uint64_t* __restrict__ tmin, uint32_t* __restrict__ trees) {
    const int64_t v = (int64_t)blockIdx.x * NBLK + threadIdx.x;
    if (v >= n) return;
    if (comp[v] == v && tmin[v] != KEY_EMPTY) atomicAdd(trees, 1u);
}

__global__ void __launch_bounds__(NBLK) k_scatter_normals(const float* __restrict__ nx, const float* __restrict__ ny,
                                                           const float* __restrict__ nz, const int32_t* __restrict__ perm,
                                                           int64_t n, float* __restrict__ ox, float* __restrict__ oy,
                                                           float* __restrict__ oz) {
    const int64_t s = (int64_t)blockIdx.x * NBLK + threadIdx.x;
    if (s >= n) return;
    const int32_t o = perm[s];
    ox[o] = nx[s];
    oy[o] = ny[s];
    oz[o] = nz[s];
}

template <class T>
T* dalloc(DBuf<uint8_t>& b, size_t& off, size_t count) {
    off = (off + 255) & ~(size_t)255;
    T* p = reinterpret_cast<T*>(b.p + off);
    off += count * sizeof(T);
    return p;
}

}  // namespace

void run_normals(egt_ctx* h, float* nxh, float* nyh, float* nzh) {
    const int64_t n = h->n;
    hipStream_t s = h->stream;
    Event ev0, ev1;
    HIP_CHECK(hipEventRecord(ev0, s));
    const dim3 gn(ceil_div(n, NBLK)), blk(NBLK);

    float* nrm = h->scratch.get<float>(8, 6 * (size_t)n);
    float *nx = nrm, *ny = nrm + n, *nz = nrm + 2 * n;
    if (!h->csr_valid) build_csr_from_rows(h);
    k_pca<<<gn, blk, 0, s>>>(h->mpts.p, h->rowptr.p, h->col.p, n, nx, ny, nz);
    LAUNCH_CHECK();

    // canonical undirected edge list
    uint32_t* cnt = h->scratch.get<uint32_t>(9, n);
    uint32_t* off = h->scratch.get<uint32_t>(10, n);
    uint8_t* own = h->scratch.get<uint8_t>(11, std::max<int64_t>(h->nnz, 1) + n);
    uint8_t* lcount = own + std::max<int64_t>(h->nnz, 1);  // per Morton position: edges the row owns
    HIP_CHECK(hipMemsetAsync(cnt, 0, n * sizeof(uint32_t), s));
    auto edges = [&](auto kernel, int32_t* out) {
        in_launches(ceil_div(n, NBLK / EDGE_LANES), MAX_GROUPS, [&](int64_t first, int64_t groups) {
            kernel<<<(unsigned)groups, blk, 0, s>>>(h->rowptr.p, h->col.p, h->morder.p, n, cnt, own, lcount, out, first);
            LAUNCH_CHECK();
        });
    };
    edges(k_edges<0>, nullptr);
    // the edges' exact number sizes their arrays, or, where one workgroup builds the forest, the number of columns
    // does, which spares a trip to the host; the kernels read it where it lies
    const uint32_t* md = exclusive_scan_u32(h, cnt, off, n);
    uint32_t m = (uint32_t)h->nnz;
    if (n > BVS_MAX) fetch(h->lane, {{&m, md, sizeof(m)}});
    HIP_CHECK(hipMemcpyAsync(cnt, off, n * sizeof(uint32_t), hipMemcpyDeviceToDevice, s));
    DBuf<uint8_t> pool;
    const size_t mm = std::max<uint32_t>(m, 1);
    pool.alloc(mm * (4 + 4 + 8 + 1 + 1 + 4 + 32) + (size_t)n * (4 + 1 + 8 + 4 + 8 + 8) + 24 * 256 + 4096 * 12);
    size_t po = 0;
    int32_t* ev = dalloc<int32_t>(pool, po, mm);
    int32_t* eu = dalloc<int32_t>(pool, po, mm);
    uint64_t* ekey = dalloc<uint64_t>(pool, po, mm);
    uint8_t* erel = dalloc<uint8_t>(pool, po, mm);
    uint8_t* msf = dalloc<uint8_t>(pool, po, mm);
    float* ew = dalloc<float>(pool, po, mm);
    int32_t* comp = dalloc<int32_t>(pool, po, n);
    uint8_t* par = dalloc<uint8_t>(pool, po, n);
    uint64_t* best = dalloc<uint64_t>(pool, po, n);
    uint32_t* H = dalloc<uint32_t>(pool, po, n);
    uint64_t* tmin = dalloc<uint64_t>(pool, po, n);
    uint64_t* best1 = dalloc<uint64_t>(pool, po, n);
    uint4* alive_a = dalloc<uint4>(pool, po, mm);
    uint4* alive_b = dalloc<uint4>(pool, po, mm);
    uint32_t* state = dalloc<uint32_t>(pool, po, 4);  // hook-walk overflow, alive-edge counts (two), trees
    double* part_w = dalloc<double>(pool, po, 1024);
    uint32_t* part_c = dalloc<uint32_t>(pool, po, 1024);
    if (po > pool.n) throw ArgError{EGT_ERR_STATE, "normals pool overflow"};

    edges(k_edges<1>, ev);
    k_edge_sort<<<gn, blk, 0, s>>>(off, n, md, ev, eu);
    LAUNCH_CHECK();
    const dim3 gm(std::max(1, ceil_div(m, NBLK)));
    if (m > 0) {
        k_edge_attr<<<gm, blk, 0, s>>>(eu, ev, md, nx, ny, nz, ekey, erel, ew);
        LAUNCH_CHECK();
    }
    uint32_t* trees_d = state + 3;
    if (n <= BVS_MAX) {
        k_bv_small<<<1, BVS_BLOCK, bvs_lds(n), s>>>((int)n, md, eu, ev, ekey, erel, msf, nx, ny, nz, trees_d);
        LAUNCH_CHECK();
    } else {
        // Boruvka with parity. The alive-edge counts live in device memory, so rounds follow one another without a
        // host round trip: four launches each. A round at least halves the components and in practice leaves under
        // a third, so the host first looks (count, to stop once no edge joins two components, and the hook walk's
        // overflow flag) after about log2(n) / 2.4 rounds, then every second one. A round after convergence finds
        // no edge and changes nothing.
        HIP_CHECK(hipMemsetAsync(msf, 0, mm, s));
        k_bv_init<<<gn, blk, 0, s>>>(n, comp, par, best, tmin, H, state, m);
        LAUNCH_CHECK();
        int first_look = 0;
        while ((1ll << first_look) < n) ++first_look;
        first_look = (int)(first_look / 2.4);
        uint32_t* count[2] = {state + 2, state + 1};  // alive edges, this round and next; state[0]: overflow flag
        uint4* alive = nullptr;                       // null = all edges
        uint32_t bound = m;                           // host-side upper bound of the alive count
        for (int round = 0; round < 64 && bound > 0; ++round) {
            const int gb = std::min(BV_GRID, std::max(1, ceil_div(bound, NBLK)));
            const int gm2 = std::min(BV_GRID, std::max(1, ceil_div(bound, BV_CHUNK)));
            k_bv_best<<<gb, blk, 0, s>>>(eu, ev, ekey, alive, count[0], best);
            k_bv_hook<<<gn, blk, 0, s>>>(n, eu, ev, erel, comp, par, best, H, msf, round == 0 ? best1 : nullptr,
                                         count[1]);
            k_bv_jump<<<gn, blk, 0, s>>>(n, comp, H, state);
            uint4* out = alive == alive_a ? alive_b : alive_a;
            k_bv_merge<<<(int)gn.x + gm2, blk, 0, s>>>(n, comp, par, H, best, eu, ev, ekey, alive, count[0], out,
                                                       count[1], (int)gn.x);
            LAUNCH_CHECK();
            alive = out;
            std::swap(count[0], count[1]);
            if (round >= first_look && ((round - first_look) & 1) == 0) {
                uint32_t hs[3];
                fetch(h->lane, {{hs, state, sizeof(hs)}});
                if (hs[0]) throw ArgError{EGT_ERR_STATE, "spanning forest: hook walk exceeded n steps"};
                bound = hs[count[0] - state];
            }
        }

        // orientation
        if (m > 0) {
            k_tree_min<<<gn, blk, 0, s>>>(n, comp, best1, tmin);
            LAUNCH_CHECK();
        }
        k_orient<<<gn, blk, 0, s>>>(n, comp, par, tmin, eu, nx, ny, nz);
        LAUNCH_CHECK();
        k_count_roots<<<gn, blk, 0, s>>>(n, comp, tmin, trees_d);
        LAUNCH_CHECK();
    }
    HIP_CHECK(hipEventRecord(ev1, s));

    // statistics
    const int sb = std::min(1024, std::max(1, ceil_div(m, NBLK)));
    k_msf_stats<<<sb, blk, 0, s>>>(msf, ew, md, part_w, part_c);
    LAUNCH_CHECK();
    std::vector<double> hw(sb);
    std::vector<uint32_t> hc(sb);
    uint32_t trees = 0;

    // original order
    float* on = nrm + 3 * n;
    k_scatter_normals<<<gn, blk, 0, s>>>(nx, ny, nz, h->perm.p, n, on, on + n, on + 2 * n);
    LAUNCH_CHECK();
    const size_t bytes = n * sizeof(float);
    fetch(h->lane, {{hw.data(), part_w, sb * sizeof(double)},
                    {hc.data(), part_c, sb * sizeof(uint32_t)},
                    {&trees, trees_d, sizeof(uint32_t)},
                    {nxh, on, bytes},
                    {nyh, on + n, bytes},
                    {nzh, on + 2 * n, bytes}});
    HIP_CHECK(hipEventElapsedTime(&h->stats.normals_ms, ev0, ev1));
    double W = 0.0;
    int64_t C = 0;
    for (int b = 0; b < sb; ++b) {
        W += hw[b];
        C += hc[b];
    }
    h->stats.msf_weight = W;
    h->stats.msf_edges = C;
    h->stats.msf_trees = trees;
}

}  // namespace egt
