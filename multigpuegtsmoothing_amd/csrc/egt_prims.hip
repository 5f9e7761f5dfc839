// Device primitives for gfx950: exclusive prefix sum over uint32 and a stable LSD radix sort of
// (uint32 key, uint32 value) pairs. Wave64 throughout; blocks of 256 threads (4 waves).
#include <algorithm>
#include "egt_internal.h"

namespace egt {
namespace {

constexpr int SCAN_BLOCK = 256;
constexpr int SCAN_ITEMS = 8;
constexpr int SCAN_TILE = SCAN_BLOCK * SCAN_ITEMS;  // 2048

constexpr int SORT_BLOCK = 256;
constexpr int SORT_ITEMS = 16;
constexpr int SORT_TILE = SORT_BLOCK * SORT_ITEMS;  // 4096
constexpr int WAVE = 64;

__device__ inline uint32_t wave_incl_scan(uint32_t v) {
    const int lane = __lane_id();
#pragma unroll
    for (int d = 1; d < WAVE; d <<= 1) {
        const uint32_t t = __shfl_up(v, d, WAVE);
        if (lane >= d) v += t;
    }
    return v;
}

// Exclusive scan of one value per thread across a 256-thread block; returns the block total in *total.
__device__ inline uint32_t block_excl_scan(uint32_t v, uint32_t* lds4, uint32_t* total) {
    const int lane = __lane_id(), wid = threadIdx.x / WAVE;
    const uint32_t incl = wave_incl_scan(v);
    if (lane == WAVE - 1) lds4[wid] = incl;
    __syncthreads();
    uint32_t woff = 0, tot = 0;
#pragma unroll
    for (int w = 0; w < SCAN_BLOCK / WAVE; ++w) {
        const uint32_t s = lds4[w];
        if (w < wid) woff += s;
        tot += s;
    }
    __syncthreads();
    *total = tot;
    return incl - v + woff;
}

__global__ void __launch_bounds__(SCAN_BLOCK) k_scan_reduce(const uint32_t* __restrict__ in, int64_t n,
                                                             uint32_t* __restrict__ partial) {
    __shared__ uint32_t lds4[4];
    const int64_t base = (int64_t)blockIdx.x * SCAN_TILE;
    uint32_t s = 0;
#pragma unroll
    for (int r = 0; r < SCAN_ITEMS; ++r) {
        const int64_t i = base + (int64_t)r * SCAN_BLOCK + threadIdx.x;
        if (i < n) s += in[i];
    }
    uint32_t tot;
    (void)block_excl_scan(s, lds4, &tot);
    if (threadIdx.x == 0) partial[blockIdx.x] = tot;
}

// Per-block scan of SCAN_TILE items (thread t owns items [t*ITEMS, t*ITEMS+ITEMS) of the tile), adding the
// scanned block offset. total (if non-null) receives the grand total from the last block.
__global__ void __launch_bounds__(SCAN_BLOCK) k_scan_apply(const uint32_t* __restrict__ in, uint32_t* __restrict__ out,
                                                            int64_t n, const uint32_t* __restrict__ offsets,
                                                            uint32_t* __restrict__ total) {
    __shared__ uint32_t lds4[4];
    __shared__ uint32_t tile[SCAN_TILE];
    const int64_t base = (int64_t)blockIdx.x * SCAN_TILE;
#pragma unroll
    for (int r = 0; r < SCAN_ITEMS; ++r) {
        const int64_t i = base + (int64_t)r * SCAN_BLOCK + threadIdx.x;
        tile[r * SCAN_BLOCK + threadIdx.x] = i < n ? in[i] : 0u;
    }
    __syncthreads();
    uint32_t v[SCAN_ITEMS];
    uint32_t s = 0;
#pragma unroll
    for (int r = 0; r < SCAN_ITEMS; ++r) {
        v[r] = tile[threadIdx.x * SCAN_ITEMS + r];
        s += v[r];
    }
    uint32_t tot;
    uint32_t run = block_excl_scan(s, lds4, &tot) + (offsets ? offsets[blockIdx.x] : 0u);
#pragma unroll
    for (int r = 0; r < SCAN_ITEMS; ++r) {
        tile[threadIdx.x * SCAN_ITEMS + r] = run;
        run += v[r];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < SCAN_ITEMS; ++r) {
        const int64_t i = base + (int64_t)r * SCAN_BLOCK + threadIdx.x;
        if (i < n) out[i] = tile[r * SCAN_BLOCK + threadIdx.x];
    }
    if (total && blockIdx.x == gridDim.x - 1 && threadIdx.x == SCAN_BLOCK - 1) *total = run;
}

// Exclusive scan through per-level partial buffers: part(depth, count) returns room for count values at that
// recursion depth (allocated from a handle's scratch, or carved out of a fixed workspace).
template <class PartFn>
void scan_rec(const uint32_t* in, uint32_t* out, int64_t n, hipStream_t s, PartFn&& part, int depth,
              uint32_t* dtotal) {
    const int nb = ceil_div(n, SCAN_TILE);
    if (nb == 1) {
        k_scan_apply<<<1, SCAN_BLOCK, 0, s>>>(in, out, n, nullptr, dtotal);
        LAUNCH_CHECK();
        return;
    }
    if (depth >= 3) throw ArgError{EGT_ERR_UNSUPPORTED, "scan too large"};
    uint32_t* P = part(depth, 2 * (size_t)nb);
    k_scan_reduce<<<nb, SCAN_BLOCK, 0, s>>>(in, n, P);
    LAUNCH_CHECK();
    scan_rec(P, P + nb, nb, s, part, depth + 1, nullptr);
    k_scan_apply<<<nb, SCAN_BLOCK, 0, s>>>(in, out, n, P + nb, dtotal);
    LAUNCH_CHECK();
}

// ---------------------------------------------------------------------------------------------------
// LSD radix sort, BITS-bit digits (8: measured faster than three passes of 10 bits for 30-bit keys, 2.52 against
// 2.63 ms for the whole grid build of a 4M-point cloud and 46.8 against 48.4 ms for 55M points in 512 clouds:
// with 1024 digit values a 4096-key tile scatters runs of about 4 keys, which costs more than the pass saved).
// Pass structure: histogram per tile (digit-major count table), exclusive scan of the table, stable scatter.
// Stability inside a tile: wave w owns the contiguous sub-tile [w*1024, (w+1)*1024) and walks it in 16 rounds
// of 64 consecutive keys; lanes with equal digits are found with BITS ballots, ranked with mbcnt, and a
// per-wave per-digit LDS counter advanced by the lowest such lane.
constexpr int RADIX_BITS = 8;

// Three forms by size:
//  - up to SMALL_MAX keys: every pass in one workgroup's LDS, one launch;
//  - up to DIRECT_TILES tiles (of 1024 keys, then of 4096): a histogram per tile (tile-major), then a scatter whose
//    workgroups sum the histograms below their own tile themselves, two launches per pass;
//  - above: the counts are digit-major and scanned in launches of their own.
// A key of exactly 9 bits is one pass of 512 values. Bound: launches and a few dependent rounds up to about a
// million keys, the scattered stores above. Grid build (three sorts) with a scan per pass / now, in ms: 2,000 points
// 0.30 / 0.19, 16,384 0.40 / 0.26 (0.32 with one workgroup), 100,000 0.50 / 0.34, 1M 0.72 / 0.66, 4M 1.41 / 1.42.
constexpr int SMALL_BLOCK = 1024;
constexpr int SMALL_MAX = 8 * SMALL_BLOCK;
constexpr int DIRECT_TILES = 256;

template <int BITS, int ITEMS, bool TILE_MAJOR>
__global__ void __launch_bounds__(SORT_BLOCK) k_sort_hist(const uint32_t* __restrict__ keys, int64_t n, int shift,
                                                           uint32_t* __restrict__ counts, int nblocks) {
    constexpr int BINS = 1 << BITS;
    constexpr uint32_t MASK = BINS - 1;
    __shared__ uint32_t hist[BINS];
    for (int d = threadIdx.x; d < BINS; d += SORT_BLOCK) hist[d] = 0;
    __syncthreads();
    const int64_t base = (int64_t)blockIdx.x * SORT_BLOCK * ITEMS;
#pragma unroll 4
    for (int r = 0; r < ITEMS; ++r) {
        const int64_t i = base + (int64_t)r * SORT_BLOCK + threadIdx.x;
        if (i < n) atomicAdd(&hist[(keys[i] >> shift) & MASK], 1u);
    }
    __syncthreads();
    for (int d = threadIdx.x; d < BINS; d += SORT_BLOCK)
        counts[TILE_MAJOR ? (int64_t)blockIdx.x * BINS + d : (int64_t)d * nblocks + blockIdx.x] = hist[d];
}

// Stable rank of each of a wave's keys (ITEMS rounds of 64 consecutive keys) among the wave's keys with its digit;
// cnt (the wave's own row, zeroed) ends as the wave's digit counts. load runs ahead of round r.
template <int BITS, int ITEMS, class Load>
__device__ inline void wave_ranks(const uint32_t (&kk)[ITEMS], int64_t first, int64_t n, int shift, uint32_t* cnt,
                                  uint32_t (&pos)[ITEMS], Load&& load) {
    constexpr uint32_t MASK = (1u << BITS) - 1u;
    const int lane = __lane_id();
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const int64_t i = first + (int64_t)r * WAVE + lane;
        const bool valid = i < n;
        load(r, i, valid);
        const uint32_t digit = (kk[r] >> shift) & MASK;
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < BITS; ++b) {
            const uint64_t bal = __ballot((digit >> b) & 1u);
            peers &= ((digit >> b) & 1u) ? bal : ~bal;
        }
        const uint32_t rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(peers >> 32),
                                                        __builtin_amdgcn_mbcnt_lo((uint32_t)peers, 0u));
        const int leader = __ffsll((unsigned long long)peers) - 1;
        uint32_t old = 0;
        if (valid && lane == leader) old = atomicAdd(&cnt[digit], (uint32_t)__popcll(peers));
        old = __shfl(old, leader < 0 ? 0 : leader, WAVE);
        pos[r] = old + rank;
    }
}

// table: DIRECT, the tile-major histograms; else the scanned digit-major offsets.
template <int BITS, int ITEMS, bool DIRECT>
__global__ void __launch_bounds__(SORT_BLOCK) k_sort_scatter(const uint32_t* __restrict__ kin,
                                                              const uint32_t* __restrict__ vin,
                                                              uint32_t* __restrict__ kout, uint32_t* __restrict__ vout,
                                                              int64_t n, int shift,
                                                              const uint32_t* __restrict__ table, int nblocks) {
    constexpr int BINS = 1 << BITS, DPT = BINS / SORT_BLOCK;  // digits per thread
    static_assert(DPT * SORT_BLOCK == BINS, "whole digits per thread");
    constexpr uint32_t MASK = BINS - 1;
    __shared__ uint32_t wcnt[SORT_BLOCK / WAVE][BINS];
    __shared__ uint32_t goff[BINS];
    __shared__ uint32_t lds4[4];
    const int lane = __lane_id(), wid = threadIdx.x / WAVE;
    const int64_t base = (int64_t)blockIdx.x * SORT_BLOCK * ITEMS + (int64_t)wid * (WAVE * ITEMS);
    uint32_t kk[ITEMS], vv[ITEMS], pos[ITEMS];
    // the direct form fetches everything beside the histograms; the other one round by round, each used before the
    // next is fetched (4M keys: 36 us a pass against 47 with the loads hoisted to the front)
    auto load = [&](int r, int64_t i, bool valid) {
        kk[r] = valid ? kin[i] : 0u;
        vv[r] = valid ? vin[i] : 0u;
    };
    if (DIRECT) {
#pragma unroll
        for (int r = 0; r < ITEMS; ++r) {
            const int64_t i = base + (int64_t)r * WAVE + lane;
            load(r, i, i < n);
        }
        // digits DPT t .. DPT t + DPT - 1 of every tile, 16 tiles' counts in flight
        uint32_t below[DPT] = {}, total[DPT] = {};
        for (int b0 = 0; b0 < nblocks; b0 += 16) {
            uint32_t c[16][DPT];
#pragma unroll
            for (int u = 0; u < 16; ++u)
#pragma unroll
                for (int e = 0; e < DPT; ++e)
                    c[u][e] = table[(int64_t)min(b0 + u, nblocks - 1) * BINS + threadIdx.x * DPT + e];
#pragma unroll
            for (int u = 0; u < 16; ++u)
#pragma unroll
                for (int e = 0; e < DPT; ++e) {
                    if (b0 + u < (int)blockIdx.x) below[e] += c[u][e];
                    if (b0 + u < nblocks) total[e] += c[u][e];
                }
        }
        uint32_t sum = 0, all;
#pragma unroll
        for (int e = 0; e < DPT; ++e) sum += total[e];
        uint32_t run = block_excl_scan(sum, lds4, &all);
#pragma unroll
        for (int e = 0; e < DPT; ++e) {
            goff[threadIdx.x * DPT + e] = run + below[e];
            run += total[e];
        }
    } else {
        for (int d = threadIdx.x; d < BINS; d += SORT_BLOCK) goff[d] = table[(int64_t)d * nblocks + blockIdx.x];
    }
    for (int d = threadIdx.x; d < BINS; d += SORT_BLOCK)
        for (int w = 0; w < SORT_BLOCK / WAVE; ++w) wcnt[w][d] = 0;
    __syncthreads();
    wave_ranks<BITS, ITEMS>(kk, base, n, shift, wcnt[wid], pos, [&](int r, int64_t i, bool valid) {
        if (DIRECT) return;
        load(r, i, valid);
        asm volatile("" ::"v"(kk[r]), "v"(vv[r]) : "memory");  // used here: the rounds' loads stay apart
    });
    __syncthreads();
    for (int d = threadIdx.x; d < BINS; d += SORT_BLOCK) {  // per digit: exclusive prefix over the waves
        uint32_t run = 0;
#pragma unroll
        for (int w = 0; w < SORT_BLOCK / WAVE; ++w) {
            const uint32_t c = wcnt[w][d];
            wcnt[w][d] = run;
            run += c;
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const int64_t i = base + (int64_t)r * WAVE + lane;
        if (i < n) {
            const uint32_t digit = (kk[r] >> shift) & MASK;
            const uint32_t dst = goff[digit] + wcnt[wid][digit] + pos[r];
            kout[dst] = kk[r];
            vout[dst] = vv[r];
        }
    }
}

// Every pass of up to SMALL_BLOCK * ITEMS keys in one workgroup: keys and values stay in LDS between passes. With
// seg, workgroup b sorts the keys [seg[b], seg[b + 1]). With keys2, a second stable sort follows, by keys2[value].
template <int ITEMS>
__global__ void __launch_bounds__(SMALL_BLOCK) k_sort_small(uint32_t* __restrict__ keys, uint32_t* __restrict__ vals,
                                                             int n, int key_bits, const int64_t* __restrict__ seg,
                                                             const uint32_t* __restrict__ keys2, int key_bits2) {
    constexpr int NW = SMALL_BLOCK / WAVE, BINS = 256;
    __shared__ uint32_t sk[SMALL_BLOCK * ITEMS], sv[SMALL_BLOCK * ITEMS];
    __shared__ uint32_t wcnt[NW][BINS];
    __shared__ uint32_t goff[BINS];
    __shared__ uint32_t ws[BINS / WAVE];
    const int lane = __lane_id(), wid = threadIdx.x / WAVE;
    const int base = wid * WAVE * ITEMS;
    if (seg) {
        const int64_t first = seg[blockIdx.x];
        keys += first;
        vals += first;
        n = (int)(seg[blockIdx.x + 1] - first);
    }
    uint32_t kk[ITEMS], vv[ITEMS], pos[ITEMS];
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const int i = base + r * WAVE + lane;
        kk[r] = i < n ? keys[i] : 0u;
        vv[r] = i < n ? vals[i] : 0u;
    }
    for (int shift = 0;; shift += 8) {
        if (shift >= key_bits) {
            if (!keys2) break;
#pragma unroll
            for (int r = 0; r < ITEMS; ++r) kk[r] = base + r * WAVE + lane < n ? keys2[vv[r]] : 0u;
            keys2 = nullptr;
            key_bits = key_bits2;
            shift = 0;
        }
        for (int i = threadIdx.x; i < NW * BINS; i += SMALL_BLOCK) (&wcnt[0][0])[i] = 0;
        __syncthreads();
        wave_ranks<8, ITEMS>(kk, base, n, shift, wcnt[wid], pos, [](int, int64_t, bool) {});
        __syncthreads();
        uint32_t total = 0, incl = 0;
        if (threadIdx.x < BINS) {
#pragma unroll
            for (int w = 0; w < NW; ++w) {
                const uint32_t c = wcnt[w][threadIdx.x];
                wcnt[w][threadIdx.x] = total;
                total += c;
            }
            incl = wave_incl_scan(total);
            if (lane == WAVE - 1) ws[wid] = incl;
        }
        __syncthreads();
        if (threadIdx.x < BINS) {
            uint32_t off = incl - total;
            for (int w = 0; w < wid; ++w) off += ws[w];
            goff[threadIdx.x] = off;
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < ITEMS; ++r) {
            if (base + r * WAVE + lane < n) {
                const uint32_t digit = (kk[r] >> shift) & (BINS - 1);
                const uint32_t dst = goff[digit] + wcnt[wid][digit] + pos[r];
                sk[dst] = kk[r];
                sv[dst] = vv[r];
            }
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < ITEMS; ++r) {
            const int i = base + r * WAVE + lane;
            if (i < n) {
                kk[r] = sk[i];
                vv[r] = sv[i];
            }
        }
        // the next pass writes sk, sv and goff only after barriers that follow these reads
    }
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const int i = base + r * WAVE + lane;
        if (i < n) {
            keys[i] = kk[r];
            vals[i] = vv[r];
        }
    }
}

// Tiles of the sort at n keys: 1024 keys while the direct form has few enough of them, else 4096.
bool sort_small_tiles(int64_t n) { return n <= (int64_t)DIRECT_TILES * SORT_BLOCK * 4; }
int sort_tiles(int64_t n) { return ceil_div(n, sort_small_tiles(n) ? SORT_BLOCK * 4 : SORT_TILE); }

template <int BITS, class PartFn>
void radix_pass(const uint32_t* ki, const uint32_t* vi, uint32_t* ko, uint32_t* vo, int64_t n, int shift,
                hipStream_t s, uint32_t* cnt, uint32_t* off, PartFn&& part) {
    const int nb = sort_tiles(n);
    if (sort_small_tiles(n)) {
        k_sort_hist<BITS, 4, true><<<nb, SORT_BLOCK, 0, s>>>(ki, n, shift, cnt, nb);
        LAUNCH_CHECK();
        k_sort_scatter<BITS, 4, true><<<nb, SORT_BLOCK, 0, s>>>(ki, vi, ko, vo, n, shift, cnt, nb);
    } else if (nb <= DIRECT_TILES) {
        k_sort_hist<BITS, SORT_ITEMS, true><<<nb, SORT_BLOCK, 0, s>>>(ki, n, shift, cnt, nb);
        LAUNCH_CHECK();
        k_sort_scatter<BITS, SORT_ITEMS, true><<<nb, SORT_BLOCK, 0, s>>>(ki, vi, ko, vo, n, shift, cnt, nb);
    } else {
        k_sort_hist<BITS, SORT_ITEMS, false><<<nb, SORT_BLOCK, 0, s>>>(ki, n, shift, cnt, nb);
        LAUNCH_CHECK();
        scan_rec(cnt, off, ((int64_t)1 << BITS) * nb, s, part, 0, nullptr);
        k_sort_scatter<BITS, SORT_ITEMS, false><<<nb, SORT_BLOCK, 0, s>>>(ki, vi, ko, vo, n, shift, off, nb);
    }
    LAUNCH_CHECK();
}

// One stable LSD pass structure over explicit buffers (ak, av: n keys and values; cnt, off: one count per digit
// value and sort tile).
template <class PartFn>
void radix_passes(uint32_t* keys, uint32_t* vals, int64_t n, int key_bits, hipStream_t s, uint32_t* ak,
                  uint32_t* av, uint32_t* cnt, uint32_t* off, PartFn&& part, bool keep_keys) {
    uint32_t *ki = keys, *vi = vals, *ko = ak, *vo = av;
    int passes = 0;
    if (key_bits == 9) {
        radix_pass<9>(ki, vi, ko, vo, n, 0, s, cnt, off, part);
        std::swap(ki, ko);
        std::swap(vi, vo);
        ++passes;
    } else {
        for (int shift = 0; shift < key_bits; shift += RADIX_BITS, ++passes) {
            radix_pass<RADIX_BITS>(ki, vi, ko, vo, n, shift, s, cnt, off, part);
            std::swap(ki, ko);
            std::swap(vi, vo);
        }
    }
    if (passes & 1) {
        if (keep_keys) HIP_CHECK(hipMemcpyAsync(keys, ki, n * sizeof(uint32_t), hipMemcpyDeviceToDevice, s));
        HIP_CHECK(hipMemcpyAsync(vals, vi, n * sizeof(uint32_t), hipMemcpyDeviceToDevice, s));
    }
}

// Sorts of at most max_len <= SMALL_MAX pairs each, in one launch.
void sort_small(uint32_t* keys, uint32_t* vals, int64_t max_len, int key_bits, const int64_t* seg, int nseg,
                const uint32_t* keys2, int key_bits2, hipStream_t s) {
    const int n = (int)max_len;
    if (n <= 2 * SMALL_BLOCK)
        k_sort_small<2><<<nseg, SMALL_BLOCK, 0, s>>>(keys, vals, n, key_bits, seg, keys2, key_bits2);
    else if (n <= 4 * SMALL_BLOCK)
        k_sort_small<4><<<nseg, SMALL_BLOCK, 0, s>>>(keys, vals, n, key_bits, seg, keys2, key_bits2);
    else
        k_sort_small<8><<<nseg, SMALL_BLOCK, 0, s>>>(keys, vals, n, key_bits, seg, keys2, key_bits2);
    LAUNCH_CHECK();
}

// Sorts up to SMALL_MAX pairs in one launch; false above.
bool radix_small(uint32_t* keys, uint32_t* vals, int64_t n, int key_bits, hipStream_t s) {
    if (n > SMALL_MAX) return false;
    sort_small(keys, vals, n, key_bits, nullptr, 1, nullptr, 0, s);
    return true;
}

__global__ void __launch_bounds__(SCAN_BLOCK) k_sum_u64(const uint32_t* __restrict__ in, int64_t n,
                                                         unsigned long long* __restrict__ total) {
    uint64_t s = 0;
    for (int64_t i = (int64_t)blockIdx.x * SCAN_BLOCK + threadIdx.x; i < n; i += (int64_t)gridDim.x * SCAN_BLOCK)
        s += in[i];
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) s += __shfl_xor(s, d, WAVE);
    if (__lane_id() == 0 && s) atomicAdd(total, (unsigned long long)s);
}

}  // namespace

static DBuf<uint32_t>& part_buf(Scratch& sc, int i);

uint64_t sum_u32(egt_ctx* h, const uint32_t* in, int64_t n) {
    hipStream_t s = h->stream;
    unsigned long long* t = reinterpret_cast<unsigned long long*>(h->scratch.get<uint64_t>(36, 1));
    HIP_CHECK(hipMemsetAsync(t, 0, sizeof(uint64_t), s));
    if (n > 0) {
        k_sum_u64<<<(int)std::min<int64_t>(2048, ceil_div(n, SCAN_BLOCK)), SCAN_BLOCK, 0, s>>>(in, n, t);
        LAUNCH_CHECK();
    }
    uint64_t total = 0;
    fetch(h->lane, {{&total, t, sizeof(total)}});
    return total;
}

namespace {
// Scan partials from the handle's scratch (buffers 0-2, one per recursion depth).
auto scratch_parts(Scratch& sc) {
    return [&sc](int depth, size_t count) {
        DBuf<uint32_t>& P = part_buf(sc, depth);
        P.alloc(count);
        return P.p;
    };
}
}  // namespace

const uint32_t* exclusive_scan_u32(egt_ctx* h, const uint32_t* in, uint32_t* out, int64_t n) {
    DBuf<uint32_t>& tot = part_buf(h->scratch, 3);
    tot.alloc(1);
    scan_rec(in, out, n, h->stream, scratch_parts(h->scratch), 0, tot.p);
    return tot.p;
}

bool sort_segments(uint32_t* keys, uint32_t* vals, int64_t max_len, int key_bits, const int64_t* seg, int nseg,
                   const uint32_t* keys2, int key_bits2, hipStream_t s) {
    if (max_len > SMALL_MAX) return false;
    sort_small(keys, vals, max_len, key_bits, seg, nseg, keys2, key_bits2, s);
    return true;
}

void radix_sort_pairs(uint32_t* keys, uint32_t* vals, int64_t n, int key_bits, hipStream_t s, Scratch& sc,
                      bool keep_keys) {
    if (n <= 1 || radix_small(keys, vals, n, key_bits, s)) return;
    const int nb = sort_tiles(n);
    DBuf<uint32_t>& ak = part_buf(sc, 4);
    DBuf<uint32_t>& av = part_buf(sc, 5);
    DBuf<uint32_t>& cnt = part_buf(sc, 6);
    DBuf<uint32_t>& off = part_buf(sc, 7);
    const size_t bins = (size_t)1 << (key_bits == 9 ? 9 : RADIX_BITS);
    ak.alloc(n);
    av.alloc(n);
    cnt.alloc(bins * nb);
    off.alloc(bins * nb);
    radix_passes(keys, vals, n, key_bits, s, ak.p, av.p, cnt.p, off.p, scratch_parts(sc), keep_keys);
}

size_t radix_sort_workspace_words(int64_t n) {
    const int64_t nb = sort_tiles(n);
    const int64_t c = ((int64_t)1 << (RADIX_BITS + 1)) * nb;  // count and offset tables, a 9-bit digit's at most
    const int64_t p0 = (c + SCAN_TILE - 1) / SCAN_TILE, p1 = (p0 + SCAN_TILE - 1) / SCAN_TILE;
    const int64_t p2 = (p1 + SCAN_TILE - 1) / SCAN_TILE;
    return (size_t)(2 * n + 2 * c + 2 * (p0 + p1 + p2));
}

void radix_sort_pairs_ws(uint32_t* keys, uint32_t* vals, int64_t n, int key_bits, hipStream_t s, uint32_t* ws) {
    if (n <= 1 || radix_small(keys, vals, n, key_bits, s)) return;
    const int64_t nb = sort_tiles(n), c = ((int64_t)1 << (RADIX_BITS + 1)) * nb;
    const int64_t p0 = (c + SCAN_TILE - 1) / SCAN_TILE, p1 = (p0 + SCAN_TILE - 1) / SCAN_TILE;
    uint32_t* ak = ws;
    uint32_t* av = ak + n;
    uint32_t* cnt = av + n;
    uint32_t* off = cnt + c;
    uint32_t* parts = off + c;  // depth 0: 2 p0 words, depth 1: 2 p1, depth 2: the rest
    auto part = [parts, p0, p1](int depth, size_t) {
        return depth == 0 ? parts : (depth == 1 ? parts + 2 * p0 : parts + 2 * (p0 + p1));
    };
    radix_passes(keys, vals, n, key_bits, s, ak, av, cnt, off, part, true);
}

static DBuf<uint32_t>& part_buf(Scratch& sc, int i) { return sc.bufs[i]; }

}  // namespace egt
