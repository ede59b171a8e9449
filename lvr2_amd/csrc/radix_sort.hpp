// LSD radix sort of (u64 key, u32 value) pairs and an exclusive scan, hand-written for
// gfx950.  Replaces the host-side thrust::sort_by_key of LBVHIndex::build
// (src/liblvr2/reconstruction/cuda/LBVHIndex.cu:138, 532).
//
// One pass = 8 key bits, two launches: (1) per-tile digit counts, and their sums over groups of 16 tiles;
// (2) a stable scatter whose blocks find their own offsets: for each digit the counts of the groups
// before, of the group's tiles before, and of all smaller digits (at most 64 + 16 coalesced rows of a table in
// L2).  Above 4M keys (more than 1,024 tiles) the rows would be too many and a scan over the table
// takes their place (three more launches).
// A block's waves take contiguous runs of the tile and rank them on their own: match masks (8 ballots per key)
// and digit counters of the wave's own in LDS, no barrier until the four waves' counts meet.  With 16
// steps of three barriers each, a scan in between and tiles of 4,096 keys for every size, a pass over 30,000
// keys had taken 25 us in three launches and over 1.2M keys 54 us in five: now 12 us and 35 us in two.
// The passes are bound by launch latency up to about 1M keys, by the scattered 12-byte stores above.
#pragma once

#include <algorithm>

#include "common.hpp"

namespace lvrhip {

constexpr int RS_THREADS = 256;
constexpr int RS_WAVES = RS_THREADS / kWave;
constexpr int RS_RADIX = 256;
constexpr int RS_GROUP = 16;        // tiles per group
constexpr int RS_MAX_TILES = 1024;  // most tiles whose offsets the scatter finds by itself
constexpr int64_t RS_SMALL = 1 << 20;  // up to here 4 keys per thread (tiles of 1,024), else 16: blocks enough
                                       // for every CU matter more than the rows of counts they read

template <int ITEMS>
constexpr int rs_tile() { return RS_THREADS * ITEMS; }

// key i of the wave's run: tile, wave, step r
template <int ITEMS>
__device__ __forceinline__ int64_t rs_entry(int r)
{
    return (int64_t)blockIdx.x * rs_tile<ITEMS>() + (int64_t)(threadIdx.x / kWave) * (ITEMS * kWave) + r * kWave +
           lane_id();
}

// kScan: the counts digit-major for a scan over the table; else tile-major, with the groups' sums
template <int ITEMS, bool kScan>
static __global__ __launch_bounds__(RS_THREADS) void rs_hist_kernel(const uint64_t* __restrict__ keys, int64_t n,
                                                                    int shift, uint32_t* __restrict__ cnt, int ntiles,
                                                                    uint32_t* __restrict__ group)
{
    __shared__ uint32_t h[RS_RADIX];
    const int tid = threadIdx.x;
    h[tid] = 0;
    __syncthreads();
    uint32_t d[ITEMS];
#pragma unroll
    for (int r = 0; r < ITEMS; r++) {
        const int64_t i = rs_entry<ITEMS>(r);
        d[r] = i < n ? (uint32_t)(keys[i] >> shift) & 255u : ~0u;
    }
#pragma unroll
    for (int r = 0; r < ITEMS; r++)
        if (d[r] != ~0u) atomicAdd(&h[d[r]], 1u);
    __syncthreads();
    if constexpr (kScan) {
        cnt[(int64_t)tid * ntiles + blockIdx.x] = h[tid];
    } else {
        cnt[(int64_t)blockIdx.x * RS_RADIX + tid] = h[tid];
        if (h[tid]) atomicAdd(&group[(blockIdx.x / RS_GROUP) * RS_RADIX + tid], h[tid]);
    }
}

// One 4096-entry segment of an in-place exclusive scan by a 1024-thread block: entries
// [base, base + 4096) get carry + their exclusive prefix within the segment; returns the
// segment's total (on every thread).
constexpr int SCAN_SEG = 4096;
__device__ __forceinline__ uint32_t scan_segment(uint32_t* __restrict__ a, int64_t len, int64_t base, uint32_t carry,
                                                 uint32_t* wsum)
{
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    uint32_t v[4];
    uint32_t s = 0;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        int64_t i = base + (int64_t)tid * 4 + j;
        v[j] = i < len ? a[i] : 0u;
        s += v[j];
    }
    // inclusive wave scan of per-thread sums
    uint32_t incl = s;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        uint32_t y = __shfl_up(incl, o, 64);
        if (lane >= o) incl += y;
    }
    if (lane == 63) wsum[wave] = incl;
    __syncthreads();
    uint32_t wpre = 0, tot = 0;
    for (int w = 0; w < 16; w++) {
        uint32_t x = wsum[w];
        if (w < wave) wpre += x;
        tot += x;
    }
    uint32_t run = carry + wpre + incl - s;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        int64_t i = base + (int64_t)tid * 4 + j;
        if (i < len) a[i] = run;
        run += v[j];
    }
    __syncthreads();  // wsum is reused by the next segment
    return tot;
}

// In-place exclusive scan of a[0..len) with one 1024-thread block, one segment per step.
static __global__ __launch_bounds__(1024) void scan_exclusive_kernel(uint32_t* __restrict__ a, int64_t len,
                                                              uint32_t* __restrict__ total)
{
    __shared__ uint32_t wsum[16];
    uint32_t carry = 0;
    for (int64_t base = 0; base < len; base += SCAN_SEG) carry += scan_segment(a, len, base, carry, wsum);
    if (threadIdx.x == 0 && total) *total = carry;
}

// Multi-block form for long tables (the radix sort's digit table: 256 entries per 4096 keys):
// (1) each block sums its segment, (2) one block scans the segment sums, (3) each block scans
// its segment from its carry.
static __global__ __launch_bounds__(1024) void scan_segsum_kernel(const uint32_t* __restrict__ a, int64_t len,
                                                           uint32_t* __restrict__ sums)
{
    __shared__ uint32_t wsum[16];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t base = (int64_t)blockIdx.x * SCAN_SEG;
    uint32_t s = 0;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        int64_t i = base + (int64_t)tid * 4 + j;
        s += i < len ? a[i] : 0u;
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) s += __shfl_xor(s, o, 64);
    if (lane == 0) wsum[wave] = s;
    __syncthreads();
    if (tid == 0) {
        uint32_t t = 0;
        for (int w = 0; w < 16; w++) t += wsum[w];
        sums[blockIdx.x] = t;
    }
}

static __global__ __launch_bounds__(1024) void scan_segapply_kernel(uint32_t* __restrict__ a, int64_t len,
                                                             const uint32_t* __restrict__ carry)
{
    __shared__ uint32_t wsum[16];
    scan_segment(a, len, (int64_t)blockIdx.x * SCAN_SEG, carry[blockIdx.x], wsum);
}

// Exclusive scan of a[0..len) in place; sums holds ceil(len / 4096) entries.
inline void scan_exclusive(uint32_t* a, int64_t len, uint32_t* sums, hipStream_t st)
{
    const int64_t nseg = ceil_div(len, SCAN_SEG);
    if (nseg <= 4) {
        scan_exclusive_kernel<<<1, 1024, 0, st>>>(a, len, nullptr);
        LVRHIP_LAUNCH_CHECK();
        return;
    }
    scan_segsum_kernel<<<(unsigned)nseg, 1024, 0, st>>>(a, len, sums);
    LVRHIP_LAUNCH_CHECK();
    scan_exclusive_kernel<<<1, 1024, 0, st>>>(sums, nseg, nullptr);
    LVRHIP_LAUNCH_CHECK();
    scan_segapply_kernel<<<(unsigned)nseg, 1024, 0, st>>>(a, len, sums);
    LVRHIP_LAUNCH_CHECK();
}

template <int ITEMS, bool kScan>
static __global__ __launch_bounds__(RS_THREADS) void rs_scatter_kernel(const uint64_t* __restrict__ kin,
                                                                       const uint32_t* __restrict__ vin,
                                                                       uint64_t* __restrict__ kout,
                                                                       uint32_t* __restrict__ vout, int64_t n,
                                                                       int shift, const uint32_t* __restrict__ cnt,
                                                                       int ntiles, const uint32_t* __restrict__ group)
{
    __shared__ uint32_t wcnt[RS_WAVES][RS_RADIX];  // the waves' digit counts, then their digits' offsets
    __shared__ uint32_t wsum[RS_WAVES];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
#pragma unroll
    for (int w = 0; w < RS_WAVES; w++) wcnt[w][tid] = 0;
    uint64_t key[ITEMS];
    uint32_t val[ITEMS], rank[ITEMS];
#pragma unroll
    for (int r = 0; r < ITEMS; r++) {
        const int64_t i = rs_entry<ITEMS>(r);
        key[r] = i < n ? kin[i] : 0ull;
        val[r] = i < n ? vin[i] : 0u;
    }
    // where this tile's keys of digit `tid` start
    uint32_t at = 0;
    if constexpr (kScan) {
        at = cnt[(int64_t)tid * ntiles + blockIdx.x];
    } else {
        const int t = (int)blockIdx.x, g = t / RS_GROUP, ng = (ntiles + RS_GROUP - 1) / RS_GROUP;
        uint32_t total = 0;
#pragma unroll 16
        for (int j = 0; j < ng; j++) {
            const uint32_t c = group[j * RS_RADIX + tid];
            total += c;
            at += j < g ? c : 0u;
        }
#pragma unroll
        for (int j = 0; j < RS_GROUP; j++) {
            const int tj = g * RS_GROUP + j;
            if (tj < t) at += cnt[(int64_t)tj * RS_RADIX + tid];
        }
        uint32_t incl = total;  // keys of smaller digits: a scan over the block
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t y = __shfl_up(incl, o, 64);
            if (lane >= o) incl += y;
        }
        if (lane == 63) wsum[wave] = incl;
        at += incl - total;
    }
    __syncthreads();
    if constexpr (!kScan)
        for (int w = 0; w < wave; w++) at += wsum[w];
    // ranks within the wave's run, digit by digit in its order
    volatile uint32_t* wc = wcnt[wave];
    const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
#pragma unroll
    for (int r = 0; r < ITEMS; r++) {
        const bool valid = rs_entry<ITEMS>(r) < n;
        const uint32_t d = (uint32_t)(key[r] >> shift) & 255u;
        uint64_t peers = ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; b++) {
            const bool bit = (d >> b) & 1u;
            const uint64_t bal = ballot(bit);
            peers &= bit ? bal : ~bal;
        }
        const uint32_t pre = wc[d];
        rank[r] = pre + (uint32_t)__popcll(peers & lt_mask);
        __builtin_amdgcn_wave_barrier();  // every lane has read before the first of the peers writes
        if (valid && (peers & lt_mask) == 0) wc[d] = pre + (uint32_t)__popcll(peers);
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < RS_WAVES; w++) {
        const uint32_t c = wcnt[w][tid];
        wcnt[w][tid] = at;
        at += c;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ITEMS; r++) {
        if (rs_entry<ITEMS>(r) < n) {
            const uint32_t o = wcnt[wave][(uint32_t)(key[r] >> shift) & 255u] + rank[r];
            kout[o] = key[r];
            vout[o] = val[r];
        }
    }
}

inline int64_t rs_tiles(int64_t n)
{
    return ceil_div(std::max<int64_t>(n, 1), n <= RS_SMALL ? rs_tile<4>() : rs_tile<16>());
}
// Entries the radix sort's table must hold for n keys: the digit counts, then the groups' sums of up to
// eight passes or the scan's segment sums.
inline size_t rs_hist_size(int64_t n)
{
    const int64_t t = rs_tiles(n), len = (int64_t)RS_RADIX * t;
    return (size_t)(len + (t <= RS_MAX_TILES ? 8 * (int64_t)RS_RADIX * ceil_div(t, (int64_t)RS_GROUP) : ceil_div(len, SCAN_SEG)));
}

inline int rs_passes(int end_bit, int begin_bit = 0) { return (end_bit - begin_bit + 7) / 8; }

template <int ITEMS, bool kScan>
inline void rs_run(uint64_t* kin, uint32_t* vin, uint64_t* kout, uint32_t* vout, int64_t n, uint32_t* hist,
                   hipStream_t st, int end_bit, int begin_bit)
{
    const int ntiles = (int)rs_tiles(n);
    uint32_t* extra = hist + (size_t)RS_RADIX * ntiles;
    const int64_t grp = (int64_t)RS_RADIX * ceil_div(ntiles, RS_GROUP);
    if (!kScan) {
        const int64_t len = grp * rs_passes(end_bit, begin_bit);
        fill_u32_kernel<<<(unsigned)ceil_div(len, 256), 256, 0, st>>>(extra, len, 0u);
        LVRHIP_LAUNCH_CHECK();
    }
    for (int shift = begin_bit; shift < end_bit; shift += 8) {
        rs_hist_kernel<ITEMS, kScan><<<ntiles, RS_THREADS, 0, st>>>(kin, n, shift, hist, ntiles, extra);
        LVRHIP_LAUNCH_CHECK();
        if (kScan) scan_exclusive(hist, (int64_t)RS_RADIX * ntiles, extra, st);
        rs_scatter_kernel<ITEMS, kScan><<<ntiles, RS_THREADS, 0, st>>>(kin, vin, kout, vout, n, shift, hist, ntiles,
                                                                      extra);
        LVRHIP_LAUNCH_CHECK();
        if (!kScan) extra += grp;
        std::swap(kin, kout);
        std::swap(vin, vout);
    }
}

// Stable sort of n (key, value) pairs by key bits [begin_bit, end_bit), 8 bits per pass, at most 64 bits.  The
// result ends in (keys, vals); the input is there too if the number of passes (rs_passes) is even, else in
// (ktmp, vtmp).  hist must hold rs_hist_size(n) entries.
inline void radix_sort_pairs(uint64_t* keys, uint32_t* vals, uint64_t* ktmp, uint32_t* vtmp, int64_t n,
                             uint32_t* hist, hipStream_t st, int end_bit = 64, int begin_bit = 0)
{
    if (n < 1) return;
    uint64_t *kin = keys, *kout = ktmp;
    uint32_t *vin = vals, *vout = vtmp;
    if (rs_passes(end_bit, begin_bit) & 1) {
        std::swap(kin, kout);
        std::swap(vin, vout);
    }
    if (n <= RS_SMALL)
        rs_run<4, false>(kin, vin, kout, vout, n, hist, st, end_bit, begin_bit);
    else if (rs_tiles(n) <= RS_MAX_TILES)
        rs_run<16, false>(kin, vin, kout, vout, n, hist, st, end_bit, begin_bit);
    else
        rs_run<16, true>(kin, vin, kout, vout, n, hist, st, end_bit, begin_bit);
}

}  // namespace lvrhip
