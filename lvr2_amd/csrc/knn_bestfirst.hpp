// Exact kNN for small k by best-first traversal, one lane per query.
//
// The tile kernel (knn_tile.hpp) serves large neighbourhoods (the adaptive normals' k = 2kn ..
// 32kn) well, but a signed-distance query needs only kd (5 .. 30) neighbours, and for lattice
// vertices just off a very dense surface its radius attempts must close in on the k-th distance
// to within micrometres, tile after tile.  A best-first search needs no radius: each lane keeps
// its t best keys (fp32 d^2, point index) sorted in registers and prunes the tree with the t-th,
// which tightens as points are found.  It replaces AdaptiveKSearchSurface::distance's kSearch
// (AdaptiveKSearchSurface.tcc:414-457, called from PointsetGrid.tcc:123-149) and
// SearchKDTree::kSearch / radiusSearch (KDTree.tcc:331-387) for k <= BF_KMAX.
//
// A lane keeps a pool of subtrees not yet entered, each with a lower bound of its distance.  A step
// takes the nearest of them and descends from it, always to the nearest child (BvhNode4: four
// grandchildren per node), until it reaches a leaf; what is left of every node passed (its other
// children within the bound) goes into the pool as one entry.  The search ends when the pool's nearest
// entry is beyond the t-th key.
// The order decides the work: a depth-first stack (nearest child first) returns to the siblings of
// its first leaf, near the query or not, while the bound is still wide.  On the lattice vertices of the
// 4M-point room (t = 10) that scanned 21 leaves and expanded about 50 nodes per query; taking the nearest
// pool entry after every leaf scans 8.6 and expands 37 (a strict best-first queue: 7.7 and 25, but it
// holds four times the entries).  Signed distances at 700,000 vertices of that lattice, sort included:
// 5.17 -> 1.19 ms (1.00 with the rest of the call's launches).
// The few queries whose lane stack overflows (hundreds of leaves within their bound) are searched
// again by a whole wave each (bf_knn_wave_kernel), and the tile kernel takes any that outgrow
// that stack too.
// Box distances are monotone lower bounds of the fp32 d^2 of every point in the box, so a box
// is skipped only when none of its points can enter the list: the result is the exact t
// smallest keys, identical to the tile kernel's.
#pragma once

#include "adjoint.hpp"
#include "common.hpp"
#include "knn_tile.hpp"
#include "lbvh.hpp"
#include "sinks.hpp"

namespace lvrhip {

constexpr int BF_THREADS = 64;  // one wave per workgroup
// A lane's pool: BF_POOL entries in LDS, then BF_SPILL more in global memory (a few lanes in 10,000).
// An entry is a node with the mask of its children still to be entered (the top 4 bits), and the upper
// 16 bits of the smallest of their box distances: rounded towards zero, so still a lower bound.  24
// entries of 6 bytes are 9.2 KB per wave: 17 waves per CU by LDS (99 % of the room's queries never hold
// more than 21).
constexpr int BF_POOL = 24;
constexpr int BF_SPILL = 40;
constexpr uint32_t BF_NODE_MASK = 0x0FFFFFFFu;  // node index of an entry (n < 2^32 points: nodes < 2^28)
typedef uint32_t __attribute__((may_alias)) bf_word;  // two 16-bit distances read as one word
struct BfPool {
    uint32_t ref[BF_POOL][BF_THREADS];
    alignas(4) uint16_t d[BF_POOL / 2][BF_THREADS][2];  // slots 2 w and 2 w + 1 of a lane share a word; 0xFFFF: free
};

constexpr int BF_KMAX = 32;
// key of an empty list slot: above every key of a finite d^2 (and of d^2 = inf with a real index)
constexpr uint64_t BF_EMPTY = 0x7F800000FFFFFFFFull;
constexpr uint64_t BF_NONE = 0x7FE0000000000000ull;  // no candidate: above every key, a finite double

// Keys as doubles.  A key's upper word is a non-negative float's bits (at most 0x7F800000), so as a
// double it is positive and finite, and doubles order like the 64-bit integers they are made of: a
// compare-exchange is one v_min_f64 and one v_max_f64 (full rate on gfx950) where 64-bit integers take a
// compare and four selects.  Tiny keys (d^2 = 0) are denormal doubles, which the double unit keeps.
__device__ __forceinline__ double bf_as_f64(uint64_t k) { return __longlong_as_double((long long)k); }
__device__ __forceinline__ uint64_t bf_as_u64(double k) { return (uint64_t)__double_as_longlong(k); }
__device__ __forceinline__ double bf_min(double a, double b)
{
    double r;
    asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ double bf_max(double a, double b)
{
    double r;
    asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ void bf_cas(double& a, double& b)
{
    const double lo = bf_min(a, b), hi = bf_max(a, b);
    a = lo;
    b = hi;
}

// Batcher's odd-even merge sort of c[0, 16) (63 compare-exchanges).
__device__ __forceinline__ void bf_sort16(double (&c)[16])
{
#pragma unroll
    for (int p = 1; p < 16; p *= 2)
#pragma unroll
        for (int k = p; k >= 1; k /= 2)
#pragma unroll
            for (int j = k % p; j + k < 16; j += 2 * k)
#pragma unroll
                for (int i = 0; i < k; i++)
                    if (i + j + k < 16 && (i + j) / (2 * p) == (i + j + k) / (2 * p)) bf_cas(c[i + j], c[i + j + k]);
}

// Sort a bitonic sequence (ascending, then descending) in x[B, B + N), N <= 16.  It is taken as the end of
// a 16-entry one whose first 16 - N entries are below every key: a compare-exchange with one of those
// changes nothing and is left out.
template <int B, int N, int SZ>
__device__ __forceinline__ void bf_bitonic(double (&x)[SZ])
{
    constexpr int PAD = 16 - N;
#pragma unroll
    for (int d = 8; d >= 1; d /= 2)
#pragma unroll
        for (int i = PAD; i < 16; i++)
            if ((i & d) == 0 && i + d < 16) bf_cas(x[B + i - PAD], x[B + i + d - PAD]);
}

// The t smallest keys seen so far, ascending in key[K - t, K).  The slots below K - t hold 0, which
// stays first, so the t-th key is always key[K - 1] and every index into the arrays is a compile-time
// constant.  Unfilled slots hold `empty`, above every key that may enter.
template <int K>
struct BfList {
    static_assert(K <= 16 || K == 32, "list lengths up to 16, or 32");
    double k[K];
    uint64_t key[K];  // after finish(): the keys, and
    uint32_t sp[K];   // the sorted position of each key's point (~0: empty)
    uint64_t empty;

    __device__ __forceinline__ void init(int t, uint64_t e)
    {
        empty = e;
#pragma unroll
        for (int j = 0; j < K; j++) k[j] = bf_as_f64(j < K - t ? 0ull : e);
    }
    __device__ __forceinline__ uint64_t worst() const { return bf_as_u64(k[K - 1]); }
    // d^2 of the t-th key: the pruning bound
    __device__ __forceinline__ float bound() const { return bitsf((uint32_t)(worst() >> 32)); }
    // every one of the t slots holds a point
    __device__ __forceinline__ bool full() const { return sp[K - 1] != ~0u; }

    // the K smallest of the list and the 16 sorted candidates c
    __device__ __forceinline__ void merge(const double (&c)[16])
    {
        if constexpr (K <= 16) {
#pragma unroll
            for (int i = 0; i < K; i++) k[i] = bf_min(k[i], c[K - 1 - i]);
            bf_bitonic<0, K>(k);
        } else {
            // the candidates against the larger half, then the halves against each other
#pragma unroll
            for (int i = 0; i < 16; i++) k[16 + i] = bf_min(k[16 + i], c[15 - i]);
            bf_bitonic<16, 16>(k);
#pragma unroll
            for (int i = 0; i < 8; i++) {  // k[i] with k[31 - i]: both halves become bitonic
                bf_cas(k[i], k[31 - i]);
                bf_cas(k[15 - i], k[16 + i]);
            }
            bf_bitonic<0, 16>(k);
            bf_bitonic<16, 16>(k);
        }
    }

    // keys and sorted positions for the consumer
    __device__ __forceinline__ void finish(const uint32_t* __restrict__ rank, int t)
    {
#pragma unroll
        for (int j = 0; j < K; j++) {
            key[j] = bf_as_u64(k[j]);
            sp[j] = j >= K - t && key[j] < empty ? rank[(uint32_t)key[j]] : ~0u;
        }
    }
};

// The leaf's points whose key beats the current t-th: sorted by a network and merged into the list, with
// no loop and no branch per point (the search's leaf work is the same for every lane of the wave; taking
// the points in one by one had run as many rounds as the busiest lane had improving points).
template <int K>
__device__ __forceinline__ void bf_scan_leaf(const BvhView& bv, int leaf, float qx, float qy, float qz, BfList<K>& L)
{
    const float4* p = bv.pts4 + (size_t)leaf * LEAF;
    float4 v[LEAF];
#pragma unroll
    for (int j = 0; j < LEAF; j++) v[j] = p[j];
    static_assert(LEAF == 16, "the sorting network");
    double c[LEAF];
    const uint64_t w = L.worst();
    bool any = false;
#pragma unroll
    for (int j = 0; j < LEAF; j++) {
        const float d = d2_contract(qx, qy, qz, v[j].x, v[j].y, v[j].z);
        const uint64_t key = make_key(d, fbits(v[j].w));
        // padding slots have NaN coordinates: their keys are above every bound
        const bool in = key < w;
        any = any || in;
        c[j] = bf_as_f64(in ? key : BF_NONE);
    }
    if (ballot(any) == 0) return;
    bf_sort16(c);
    L.merge(c);
}

__device__ __forceinline__ float bf_child_d2(const float* f, int k, float qx, float qy, float qz)
{
    return box_d2(f[6 * k], f[6 * k + 1], f[6 * k + 2], f[6 * k + 3], f[6 * k + 4], f[6 * k + 5], qx, qy, qz, qx, qy,
                  qz);
}

// The pool of lane `lane`: which slots are free, and how many entries were spilled.
struct BfLane {
    uint32_t free;  // bit i: slot i of the LDS pool is free
    int nspill;
    uint2* spill;  // this lane's spilled entries (ref, d), interleaved with the wave's other lanes
    int spill_cap;
    int lanes;  // of the wave that search, and have a spill area
};

// Puts an entry into the pool; false if neither the LDS slots nor the spill area hold it.
__device__ __forceinline__ bool bf_put(BfPool& pool, BfLane& ln, int lane, uint32_t ref, uint32_t d16, float bound)
{
    if (ln.free == 0u) {  // drop the entries the bound has left behind
#pragma unroll
        for (int i = 0; i < BF_POOL; i++) {
            const uint32_t e = pool.d[i / 2][lane][i & 1];
            if (bitsf(e << 16) > bound) {
                ln.free |= 1u << i;
                pool.d[i / 2][lane][i & 1] = 0xFFFFu;
            }
        }
    }
    if (ln.free == 0u) {
        if (ln.nspill == ln.spill_cap) return false;
        ln.spill[(size_t)ln.nspill * ln.lanes] = make_uint2(ref, d16);
        ln.nspill++;
        return true;
    }
    const int slot = __ffs((int)ln.free) - 1;
    ln.free &= ln.free - 1u;
    pool.ref[slot][lane] = ref;
    pool.d[slot / 2][lane][slot & 1] = (uint16_t)d16;
    return true;
}

// Takes the nearest entry within the bound out of the pool; false if there is none.
__device__ __forceinline__ bool bf_take(BfPool& pool, BfLane& ln, int lane, float bound, uint32_t& ref)
{
    for (;;) {
        // minimum of (d, slot) over all slots, two per LDS word; a free slot's d is above every bound
        uint32_t m = ~0u;
        const bf_word* w = reinterpret_cast<const bf_word*>(&pool.d[0][lane][0]);
#pragma unroll
        for (int i = 0; i < BF_POOL / 2; i++) {
            const uint32_t x = w[i * BF_THREADS];
            const uint32_t e0 = (x << 16) | (uint32_t)(2 * i), e1 = (x & 0xFFFF0000u) | (uint32_t)(2 * i + 1);
            m = min(m, min(e0, e1));
        }
        if (bitsf(m & 0xFFFF0000u) <= bound) {  // (a free slot: NaN, never)
            const int slot = (int)(m & 0xFFFFu);
            ref = pool.ref[slot][lane];
            pool.d[slot / 2][lane][slot & 1] = 0xFFFFu;
            ln.free |= 1u << slot;
            return true;
        }
        if (ln.nspill == 0) return false;
        // every LDS entry is beyond the bound: free them all and bring spilled ones back
#pragma unroll
        for (int i = 0; i < BF_POOL; i++) pool.d[i / 2][lane][i & 1] = 0xFFFFu;
        ln.free = (1u << BF_POOL) - 1u;
        while (ln.nspill > 0 && ln.free != 0u) {
            ln.nspill--;
            const uint2 e = ln.spill[(size_t)ln.nspill * ln.lanes];
            const int slot = __ffs((int)ln.free) - 1;
            ln.free &= ln.free - 1u;
            pool.ref[slot][lane] = e.x;
            pool.d[slot / 2][lane][slot & 1] = (uint16_t)e.y;
        }
    }
}

// The search of one lane; returns false if its pool overflowed (the list is then incomplete).
template <int K>
__device__ __forceinline__ bool bf_search(const BvhView& bv, BfPool& pool, BfLane& ln, int lane, float qx, float qy,
                                          float qz, BfList<K>& L, int& leaves, int& nodes)
{
    constexpr int NONE = EMPTY4;
    if (bv.nleaf <= 1) {
        bf_scan_leaf<K>(bv, 0, qx, qy, qz, L);
        leaves++;
        return true;
    }
#pragma unroll
    for (int i = 0; i < BF_POOL; i++) pool.d[i / 2][lane][i & 1] = 0xFFFFu;
    ln.free = (1u << BF_POOL) - 1u;
    ln.nspill = 0;
    int cur = 0;          // the node to expand next (NONE: take one from the pool)
    uint32_t want = 15u;  // its children still to be entered
    for (;;) {
        // descend until the lane holds a leaf; then the lanes scan their leaves together
        int leaf = -1;
        const float bound = L.bound();
        for (;;) {
            if (cur == NONE) {
                uint32_t e;
                if (!bf_take(pool, ln, lane, bound, e)) break;
                cur = (int)(e & BF_NODE_MASK);
                want = e >> 28;
            }
            nodes++;
            const BvhNode4 nd = bv.nodes4[cur];
            const float* f = reinterpret_cast<const float*>(nd.b);
            const int c[4] = {nd.r.x, nd.r.y, nd.r.z, nd.r.w};
            float d[4], best = INFINITY;
            int next = NONE, bk = 0;
            uint32_t rest = 0u;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                d[k] = bf_child_d2(f, k, qx, qy, qz);
                const bool in = c[k] != EMPTY4 && ((want >> k) & 1u) && d[k] <= bound;
                if (!in) d[k] = INFINITY;
                rest |= in ? 1u << k : 0u;
                if (in && (next == NONE || d[k] < best)) {
                    best = d[k];
                    next = c[k];
                    bk = k;
                }
            }
            if (next == NONE) {
                cur = NONE;
                continue;
            }
            rest &= ~(1u << bk);
            if (rest != 0u) {
                float dr = INFINITY;
#pragma unroll
                for (int k = 0; k < 4; k++) dr = k == bk ? dr : fminf(dr, d[k]);
                if (!bf_put(pool, ln, lane, (uint32_t)cur | (rest << 28), fbits(dr) >> 16, bound)) return false;
            }
            cur = next;
            want = 15u;
            if (cur < 0) {
                leaf = -1 - cur;
                cur = NONE;
                break;
            }
        }
        if (leaf < 0) return true;  // nothing left within the bound: the list is final
        bf_scan_leaf<K>(bv, leaf, qx, qy, qz, L);
        leaves++;
    }
}

// One lane per query i < m (queries in Morton order for locality): Out(i, list, t, ok, q)
// consumes the result.  empty: the key an unfilled slot holds (BF_EMPTY, or (r^2, 0) to keep
// only points with d^2 < r^2).
// Outputs that know a neighbour set of the query beforehand declare kPrefill = true and
// first_bound(i, t, x, y, z, empty): a key above the t-th, which the search starts from.
template <class O, class = void>
struct bf_prefills : std::false_type {
};
template <class O>
struct bf_prefills<O, std::void_t<decltype(O::kPrefill)>> : std::integral_constant<bool, O::kPrefill> {
};

// stats (optional, KS_* counters of knn_tile.hpp): waves (KS_TILES), the largest leaf count of a
// lane summed over waves (KS_ATTEMPTS: a wave runs as long as its slowest lane), points scanned
// (KS_CANDIDATES), nodes expanded (KS_POPS), queries left to the next pass (KS_REFINE),
// queries resolved (KS_RESOLVED), shader-clock cycles per wave (KS_CY_TOTAL).
template <int K, class Out>
__device__ __forceinline__ void bf_stats(unsigned long long* stats, bool valid, bool ok, int leaves, int nodes,
                                         unsigned long long c0)
{
    int lmax = leaves, lsum = leaves, nsum = nodes, bad = (valid && !ok) ? 1 : 0, good = (valid && ok) ? 1 : 0;
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        lmax = max(lmax, shfl_xor(lmax, o));
        lsum += shfl_xor(lsum, o);
        nsum += shfl_xor(nsum, o);
        bad += shfl_xor(bad, o);
        good += shfl_xor(good, o);
    }
    if (lane_id() == 0) {
        atomicAdd(&stats[KS_TILES], 1ull);
        atomicAdd(&stats[KS_ATTEMPTS], (unsigned long long)lmax);
        atomicAdd(&stats[KS_CANDIDATES], (unsigned long long)lsum * LEAF);
        atomicAdd(&stats[KS_POPS], (unsigned long long)nsum);
        atomicAdd(&stats[KS_REFINE], (unsigned long long)bad);
        atomicAdd(&stats[KS_RESOLVED], (unsigned long long)good);
        atomicAdd(&stats[KS_CY_TOTAL], cycles() - c0);
    }
}

// One lane per query (queries in Morton order), chunks of per_wave (at most 64) consecutive queries per
// wave: fewer for a smaller batch (bf_per_wave).  With
// a work queue (QUEUE_SEGS counters QUEUE_STRIDE apart, zeroed before the launch; the grid is
// then the waves the device holds at once) the chunks are dealt like the tile kernel's runs:
// blocks of QUEUE_CHUNK consecutive chunks to the XCDs in turn, each XCD taking from its own
// counter and then helping the others, so neighbouring chunks share an L2 and the costly regions
// of a cloud are spread over all XCDs.  Without a queue, wave b takes chunk b.
//
// Query i is (qx[i qs], qy[i qs], qz[i qs]): qs = 1 for SoA coordinates, 3 for an AoS buffer
// (qy = qx + 1, qz = qx + 2).  spill: spill_cap entries for each of the per_wave lanes of each wave of the
// grid (all 64 lanes' would be 20 KB per wave, 64 times what a batch of one query per wave can use).
template <int K, class Out>
__global__ __launch_bounds__(BF_THREADS) void bf_knn_kernel(const BvhView bv, const float* __restrict__ qx,
                                                            const float* __restrict__ qy,
                                                            const float* __restrict__ qz, int qs, int64_t m,
                                                            int t, uint64_t empty, Out out,
                                                            unsigned long long* stats, uint32_t* queue, uint2* spill,
                                                            int spill_cap, int per_wave, uint32_t* left,
                                                            uint32_t* left_count)
{
    __shared__ BfPool pool;
    const int lane = threadIdx.x;
    const int64_t nchunks = (m + per_wave - 1) / per_wave;
    const int xcd = (int)(blockIdx.x % QUEUE_SEGS);
    int seg_k = 0;
    bool once = false;
    for (;;) {
        int64_t chunk = -1;
        if (queue) {
            chunk = queue_take(queue, nchunks, xcd, seg_k);
        } else if (!once) {
            chunk = blockIdx.x;
            once = true;
        }
        if (chunk < 0 || chunk >= nchunks) break;
        const unsigned long long c0 = stats ? cycles() : 0ull;
        const int64_t i = lane < per_wave ? chunk * per_wave + lane : m;
        int leaves = 0, nodes = 0;
        bool ok = true;
        if (i < m) {  // no barrier in the search: lanes are independent
            const float x = qx[i * qs], y = qy[i * qs], z = qz[i * qs];
            uint64_t start = empty;
            if constexpr (bf_prefills<Out>::value) start = out.first_bound(i, t, x, y, z, empty);
            BfList<K> L;
            L.init(t, start);
            BfLane ln{0u, 0, spill + (size_t)blockIdx.x * spill_cap * per_wave + lane, spill_cap, per_wave};
            ok = bf_search<K>(bv, pool, ln, lane, x, y, z, L, leaves, nodes);
            L.finish(bv.rank, t);
            // the queries left go to the next pass, in any order: each result is its query's own
            if (!out.template emit<K>(i, L, t, ok, x, y, z)) left[atomicAdd(left_count, 1u)] = (uint32_t)i;
            ok = ok && L.full();
        }
        if (stats) bf_stats<K, Out>(stats, i < m, ok, leaves, nodes, c0);
    }
}

// Zeroes a search's work queue and the counts of the queries its passes leave.
static __global__ void bf_reset_kernel(uint32_t* queue, int n, uint32_t* count1, uint32_t* count2)
{
    for (int i = threadIdx.x; i < n; i += blockDim.x) queue[i] = 0u;
    if (threadIdx.x == 0) {
        *count1 = 0u;
        *count2 = 0u;
    }
}
constexpr int BF_WAVE_STACK = 4096;
constexpr int BF_WAVE_BLOCKS = 1024;  // waves striding over the list

__device__ __forceinline__ uint64_t wave_min_u64(uint64_t v)
{
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        const uint64_t w = shfl_xor(v, o);
        v = w < v ? w : v;
    }
    return v;
}

// Wave-cooperative best-first search for the queries list[0, *count) (list NULL: all of them, a
// small batch): the ones
// whose lane pool overflowed (a very dense or a far-off neighbourhood, hundreds of leaves deep).  One
// wave per query: a greedy descent to a seed leaf; then every step pops up to 64 stack entries
// at once, the lanes expand their nodes (children within the bound pushed) or scan their leaves,
// and the t smallest keys of the list and the scanned points are extracted by t rounds of a
// wave-wide minimum.  Lane j holds the j-th key of the list in a register.  The serial chain is
// the tree depth plus leaves / 64 steps, not one step per node or leaf.  A query whose stack
// outgrows BF_WAVE_STACK entries is left to the tile kernel.
template <int K, class Out>
__global__ __launch_bounds__(BF_THREADS) void bf_knn_wave_kernel(const BvhView bv, const float* __restrict__ qx,
                                                                 const float* __restrict__ qy,
                                                                 const float* __restrict__ qz, int qs,
                                                                 const uint32_t* __restrict__ list,
                                                                 const uint32_t* __restrict__ count, int64_t all,
                                                                 int t, uint64_t empty, Out out,
                                                                 unsigned long long* stats, uint32_t* left,
                                                                 uint32_t* left_count)
{
    __shared__ uint2 stk[BF_WAVE_STACK];
    __shared__ uint64_t fkey[BF_KMAX];
    __shared__ uint32_t fsp[BF_KMAX];
    const int lane = threadIdx.x;
    const int64_t n = list ? (int64_t)*count : all;
    const int root = bv.nleaf > 1 ? 0 : leaf_ref(0);
    for (int64_t j = blockIdx.x; j < n; j += gridDim.x) {
        const unsigned long long c0 = stats ? cycles() : 0ull;
        const int64_t i = list ? (int64_t)list[j] : j;
        const float x = qx[i * qs], y = qy[i * qs], z = qz[i * qs];
        // lane j < t holds the j-th smallest key so far (empty: none)
        uint64_t bk = empty;
        uint32_t bs = ~0u;
        uint64_t worst = empty;  // the t-th key (uniform)
        int leaves = 0, nodes = 0;
        // seed leaf: greedy descent (every lane computes the same path)
        int ref = root;
        while (ref >= 0) {
            const BvhNode4 nd = bv.nodes4[ref];
            const float* f = reinterpret_cast<const float*>(nd.b);
            const int rr[4] = {nd.r.x, nd.r.y, nd.r.z, nd.r.w};
            float bd = INFINITY;
            int next = rr[0];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const float d = bf_child_d2(f, k, x, y, z);
                if (rr[k] != EMPTY4 && d < bd) {
                    bd = d;
                    next = rr[k];
                }
            }
            ref = next;
        }
        const int seed = -1 - ref;
        if (root >= 0 && lane == 0) stk[0] = make_uint2((uint32_t)root, 0u);
        int sp = root >= 0 ? 1 : 0;
        bool ok = true;
        bool first = true;
        while (first || sp > 0) {
            // this step's entries: the seed leaf first, then up to 64 popped entries
            int leaf = -1, node = -1;
            if (first) {
                if (lane == 0) leaf = seed;
            } else {
                const int w = min(BF_THREADS, sp);
                if (lane < w) {
                    const uint2 e = stk[sp - 1 - lane];
                    if (!(bitsf(e.y) > bitsf((uint32_t)(worst >> 32)))) {
                        const int r = (int)e.x;
                        if (r < 0) {
                            if (-1 - r != seed) leaf = -1 - r;
                        } else {
                            node = r;
                        }
                    }
                }
                sp -= w;
            }
            first = false;
            const float bound = bitsf((uint32_t)(worst >> 32));
            // nodes: children within the bound onto the stack
            int c[4] = {EMPTY4, EMPTY4, EMPTY4, EMPTY4};
            float d[4] = {0, 0, 0, 0};
            if (node >= 0) {
                nodes++;
                const BvhNode4 nd = bv.nodes4[node];
                const float* f = reinterpret_cast<const float*>(nd.b);
                const int rr[4] = {nd.r.x, nd.r.y, nd.r.z, nd.r.w};
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    d[k] = bf_child_d2(f, k, x, y, z);
                    if (rr[k] != EMPTY4 && d[k] <= bound) c[k] = rr[k];
                }
            }
            int npush = 0;
#pragma unroll
            for (int k = 0; k < 4; k++) npush += __popcll(ballot(c[k] != EMPTY4));
            if (sp + npush > BF_WAVE_STACK) {
                ok = false;
                break;
            }
            __syncthreads();  // the pops above read the slots the pushes overwrite
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const uint64_t m4 = ballot(c[k] != EMPTY4);
                if (c[k] != EMPTY4) stk[sp + mbcnt(m4)] = make_uint2((uint32_t)c[k], fbits(d[k]));
                sp += __popcll(m4);
            }
            __syncthreads();
            // leaves: the scanned keys below the t-th are candidates (~0: none)
            uint64_t ck[LEAF];
            bool any = false;
            if (leaf >= 0) {
                leaves++;
                const float4* pp = bv.pts4 + (size_t)leaf * LEAF;
#pragma unroll
                for (int q = 0; q < LEAF; q++) {
                    const float4 v = pp[q];
                    const float dd = d2_contract(x, y, z, v.x, v.y, v.z);
                    const uint64_t key = make_key(dd, fbits(v.w));
                    ck[q] = (dd == dd && key < worst) ? key : ~0ull;
                    any = any || ck[q] != ~0ull;
                }
            } else {
#pragma unroll
                for (int q = 0; q < LEAF; q++) ck[q] = ~0ull;
            }
            if (ballot(any) == 0) continue;
            // the new list: t rounds, each taking the smallest remaining key of the old list
            // (lane j's bk) and the candidates, to lane r
            uint64_t nk = empty;
            uint32_t ns = ~0u;
            bool own = lane < t && bk != empty;  // this lane's list entry is still unplaced
            for (int r = 0; r < t; r++) {
                uint64_t lm = own ? bk : ~0ull;
                int li = LEAF;  // LEAF: the list entry
#pragma unroll
                for (int q = 0; q < LEAF; q++) {
                    if (ck[q] < lm) {
                        lm = ck[q];
                        li = q;
                    }
                }
                const uint64_t gm = wave_min_u64(lm);
                if (gm == ~0ull || !(gm < empty)) break;  // nothing left below the bound
                const bool mine = lm == gm;  // keys are unique: exactly one lane
                const int src = __ffsll((long long)ballot(mine)) - 1;
                uint32_t s_ = ~0u;
                if (mine) {
                    if (li == LEAF) {
                        s_ = bs;
                        own = false;
                    } else {
                        s_ = (uint32_t)(leaf * LEAF + li);
#pragma unroll
                        for (int q = 0; q < LEAF; q++)
                            if (q == li) ck[q] = ~0ull;
                    }
                }
                s_ = (uint32_t)shfl((int)s_, src);
                if (lane == r) {
                    nk = gm;
                    ns = s_;
                }
            }
            bk = nk;
            bs = ns;
            // the t-th key (empty while fewer than t are known)
            worst = (uint64_t)shfl((long long)bk, t - 1);
        }
        // the list to lane 0 through LDS
        if (lane < t) {
            fkey[lane] = bk;
            fsp[lane] = bs;
        }
        __syncthreads();
        if (lane == 0) {
            BfList<K> L;
            L.empty = empty;
#pragma unroll
            for (int q = 0; q < K; q++) {
                const int o = q - (K - t);
                L.key[q] = q < K - t ? 0ull : fkey[o];
                L.sp[q] = q < K - t ? ~0u : fsp[o];
            }
            if (!out.template emit<K>(i, L, t, ok, x, y, z)) left[atomicAdd(left_count, 1u)] = (uint32_t)i;
        }
        if (stats) {
            const int lsum = wave_sum_int(leaves), nsum = wave_sum_int(nodes);
            if (lane == 0) {
                atomicAdd(&stats[KS_TILES], 1ull);
                atomicAdd(&stats[KS_CANDIDATES], (unsigned long long)lsum * LEAF);
                atomicAdd(&stats[KS_POPS], (unsigned long long)nsum);
                atomicAdd(&stats[KS_RESOLVED], ok ? 1ull : 0ull);
                atomicAdd(&stats[KS_REFINE], ok ? 0ull : 1ull);
                atomicAdd(&stats[KS_CY_TOTAL], cycles() - c0);
            }
        }
        __syncthreads();
    }
}

// Signed distance from the sorted list: positions and normals summed in ascending key order
// (tcc:435-449).  emit returns whether the query is resolved: false for a search that overflowed or found too few points.
struct BfSdfOut {
    const float* px;
    const float* py;
    const float* pz;
    const float* nx;
    const float* ny;
    const float* nz;
    const uint32_t* qorig;  // query position -> caller's index (NULL: the same)
    float voxel;
    float* out_proj;
    float* out_eucl;
    uint8_t* out_invalid;

    template <int K>
    __device__ __forceinline__ bool emit(int64_t i, const BfList<K>& L, int t, bool ok, float qx, float qy,
                                         float qz) const
    {
        // an unfilled slot (NaN coordinates) sorts last: the tile kernel handles such queries
        ok = ok && L.full();
        if (!ok) return false;
        float ax = 0, ay = 0, az = 0, bx = 0, by = 0, bz = 0;
        float v[K][6];
#pragma unroll
        for (int j = 0; j < K; j++) {
            if (j >= K - t) {
                const uint32_t s = L.sp[j];
                v[j][0] = px[s];
                v[j][1] = py[s];
                v[j][2] = pz[s];
                v[j][3] = nx[s];
                v[j][4] = ny[s];
                v[j][5] = nz[s];
            }
        }
#pragma unroll
        for (int j = 0; j < K; j++) {
            if (j >= K - t) {
                ax += v[j][0];
                ay += v[j][1];
                az += v[j][2];
                bx += v[j][3];
                by += v[j][4];
                bz += v[j][5];
            }
        }
        sdf_emit(ax, ay, az, bx, by, bz, t, qx, qy, qz, voxel, qorig ? qorig[i] : (uint32_t)i, out_proj, out_eucl,
                 out_invalid);
        return true;
    }
};

// Reverse pass of the signed distance (SinkSdfAdjoint's sums, adjoint.hpp) from the sorted list.
struct BfSdfAdjointOut {
    const float* px;
    const float* py;
    const float* pz;
    const float* nx;
    const float* ny;
    const float* nz;
    const uint32_t* qorig;  // query position -> caller's index
    const float* w;         // dL/dproj per caller index
    float* gpx;             // dL/dp and dL/dn, sorted positions
    float* gpy;
    float* gpz;
    float* gnx;
    float* gny;
    float* gnz;

    template <int K>
    __device__ __forceinline__ bool emit(int64_t i, const BfList<K>& L, int t, bool ok, float qx, float qy,
                                         float qz) const
    {
        ok = ok && L.full();
        if (!ok) return false;
        const float wv = w[qorig[i]];
        if (wv == 0.0f) return true;
        float ax = 0, ay = 0, az = 0, bx = 0, by = 0, bz = 0;
#pragma unroll
        for (int j = 0; j < K; j++) {
            if (j >= K - t) {
                const uint32_t s = L.sp[j];
                ax += px[s];
                ay += py[s];
                az += pz[s];
                bx += nx[s];
                by += ny[s];
                bz += nz[s];
            }
        }
        SdfGrad g;
        if (!sdf_grad(ax, ay, az, bx, by, bz, t, qx, qy, qz, wv, g)) return true;
#pragma unroll
        for (int j = 0; j < K; j++) {
            if (j >= K - t) {
                const uint32_t s = L.sp[j];
                atomicAdd(&gpx[s], g.px);
                atomicAdd(&gpy[s], g.py);
                atomicAdd(&gpz[s], g.pz);
                atomicAdd(&gnx[s], g.nx);
                atomicAdd(&gny[s], g.ny);
                atomicAdd(&gnz[s], g.nz);
            }
        }
        return true;
    }
};

// kSearch rows in the caller's order: row j < t the j-th key (index, d^2), the rest -1 / +inf.
// With a radius (empty = (r^2, 0)) the unfilled slots are padding too, and count[row] = the
// number of neighbours found.
struct BfRowsOut {
    const uint32_t* qorig;
    int k;
    int32_t* idx;
    float* d2;
    int32_t* count;  // optional

    template <int K>
    __device__ __forceinline__ bool emit(int64_t i, const BfList<K>& L, int t, bool ok, float, float, float) const
    {
        if (!ok) return false;
        const size_t row = qorig[i];
        int found = 0;
#pragma unroll
        for (int j = 0; j < K; j++) {
            if (j >= K - t) {
                const int o = j - (K - t);
                const bool real = L.sp[j] != ~0u;
                idx[row * k + o] = real ? (int32_t)(uint32_t)L.key[j] : -1;
                if (d2) d2[row * k + o] = real ? bitsf((uint32_t)(L.key[j] >> 32)) : INFINITY;
                found += real ? 1 : 0;
            }
        }
        for (int o = t; o < k; o++) {
            idx[row * k + o] = -1;
            if (d2) d2[row * k + o] = INFINITY;
        }
        if (count) count[row] = found;
        return true;
    }
};

// PointsetSurface::getInterpolatedNormal (PointsetSurface.tcc:61-74): a Normal starts as
// (0, 1, 0) (Normal.hpp:62); each of the ki nearest points' normals is normalised
// (Normal(x, y, z), Normal.tcc:49-54) and added; the sum is divided by ki and returned as is
// (the copy into the return value does not normalise again).
struct BfMeanNormalOut {
    const float* nx;
    const float* ny;
    const float* nz;
    const uint32_t* qorig;
    int ki;
    float* out;  // caller order, 3 floats per query

    template <int K>
    __device__ __forceinline__ bool emit(int64_t i, const BfList<K>& L, int t, bool ok, float, float, float) const
    {
        ok = ok && L.full();
        if (!ok) return false;
        float rx = 0.0f, ry = 1.0f, rz = 0.0f;
#pragma unroll
        for (int j = 0; j < K; j++) {
            if (j >= K - t) {
                const uint32_t s = L.sp[j];
                float x = nx[s], y = ny[s], z = nz[s];
                if (!(x == 0.0f && y == 0.0f && z == 0.0f)) {
                    const float l = sqrtf(x * x + y * y + z * z);
                    x /= l;
                    y /= l;
                    z /= l;
                }
                rx += x;
                ry += y;
                rz += z;
            }
        }
        const float c = (float)ki;
        rx /= c;
        ry /= c;
        rz /= c;
        const size_t o = 3 * (size_t)qorig[i];
        out[o] = rx;
        out[o + 1] = ry;
        out[o + 2] = rz;
        return true;
    }
};

// The centroid of the neighbours (BilinearFastBox::optimizePlanarFaces, BilinearFastBox.tcc:172-186):
// a zero vector plus each neighbour's position in ascending order, divided by their number.
struct BfCentroidOut {
    const float4* pts;  // sorted points
    const uint32_t* qorig;
    float* out;  // caller order, 3 floats per query
    // optional: the query's vertex (caller index -> vertex id) and, per vertex, the t neighbours
    // (sorted positions) of its last search, which a later search of the vertex starts from
    // (first_bound): their keys at the new position bound the search at once.  The result is the
    // same exact neighbour set.
    const uint32_t* vid;
    uint32_t* nbr;
    bool prefill;
    uint32_t npts;  // sorted positions
    static constexpr bool kPrefill = true;

    // the t neighbours of the vertex's last search are t different points of the cloud (every pass that
    // resolves a query saves them, the tile kernel's too, or ~0 where it found fewer): the t-th key is at most
    // the largest of their keys at the new position
    __device__ __forceinline__ uint64_t first_bound(int64_t i, int t, float qx, float qy, float qz,
                                                    uint64_t empty) const
    {
        if (!prefill || !vid || !nbr) return empty;
        const size_t v = vid[qorig[i]];
        uint64_t top = 0;
        for (int j = 0; j < t; j++) {
            const uint32_t s = nbr[v * t + j];
            if (s >= npts) return empty;
            const float4 p = pts[s];
            const float d = d2_contract(qx, qy, qz, p.x, p.y, p.z);
            if (!(d == d)) return empty;
            const uint64_t key = make_key(d, fbits(p.w));
            top = key > top ? key : top;
        }
        return top < empty ? top + 1 : empty;
    }

    template <int K>
    __device__ __forceinline__ bool emit(int64_t i, const BfList<K>& L, int t, bool ok, float qx, float qy,
                                         float qz) const
    {
        if (!ok) return false;
        if (vid && nbr) {
            const size_t v = vid[qorig[i]];
#pragma unroll
            for (int j = 0; j < K; j++)  // compile-time slots: the list stays in registers
                if (j >= K - t) nbr[v * t + (j - (K - t))] = L.sp[j];
        }
        float cx = 0.0f, cy = 0.0f, cz = 0.0f;
        int nk = 0;
#pragma unroll
        for (int j = 0; j < K; j++) {
            if (j >= K - t && L.sp[j] != ~0u) {
                const float4 p = pts[L.sp[j]];
                cx += p.x;
                cy += p.y;
                cz += p.z;
                nk++;
            }
        }
        const size_t o = 3 * (size_t)qorig[i];
        if (nk == 0) {  // nothing found: the position stays
            out[o] = qx;
            out[o + 1] = qy;
            out[o + 2] = qz;
            return true;
        }
        const float c = (float)nk;
        out[o] = cx / c;
        out[o + 1] = cy / c;
        out[o + 2] = cz / c;
        return true;
    }
};

}  // namespace lvrhip
