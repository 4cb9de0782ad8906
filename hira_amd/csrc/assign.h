// What the nearest-centroid kernels (assign_mfma.hip, and the vector-ALU one of build.hip) share
// with the index build around them: the counting of the items a centroid takes, done by the
// assignment itself, and the operand tiles of the centroids for the matrix cores.
#pragma once

#include "search.h"

namespace hira {

// Bucketing fused into an assignment launch (counts NULL: the launch only assigns).
//   counts  (T, K), 1 << count_log2 apart  zero when the round starts; counts[a] += 1 for every item assigned to a.  The
//                        value the item's increment returned is its place in the bucket:
//   members (T, K, places)  the first `places` items of every bucket, in order of arrival, and
//   dists   (T, K, places)  their distances (NULL: a Lloyd round, which asks for none)
//   places_log2, count_log2 bucket_places_log2, bucket_count_log2 of the fan-out
//   big     (T, K)       the buckets with more than kWaveBucket members, big_count (T) of them
//   more    (T, n_c)     (centroid, item) of the items behind those, more_count (T) of them, their
//   more_dist (T, n_c)   distances by item.  Such buckets are rare (a few seeds of a Lloyd round);
//                        what works on them looks for their items here.
//   lost    (T, n_c), lost_count (T)  packing: the items that have no nearest centroid (not numbers)
// With the places fixed there is no prefix sum over the counts, no tail of a launch that waits for
// it and no launch that sorts the items into buckets (4.3 + 5 us a round at 8 x 32768 items).
//   zero    (T)          a counter the launch clears (the list of the round after it), or NULL
// Counters of trees (big_count, more_count, lost_count, zero, and the lists' lengths) lie kCounterStride apart: at
// one address, or in one line of memory, an addition waits for the one before it (9 ns each; 8 x 1024
// workgroups adding to eight neighbours took 67 us).
// places = sixteen times the fan-out, the mean of a bucket, rounded up to a power of two between
// kWaveBucket and kBucketCap: 128 bytes a key of workspace at fan-outs of 4, 8 and 16, 64 at 32, less than
// 256 from 3 on.  (256 places whatever the fan-out took 512 bytes a key at 4 and 2 KiB at 1.  Eight times
// the fan-out: what lies behind the places costs 8 x 20000 rows at a fan-out of 16 2 %.)
constexpr int kBucketCap = 256;
constexpr int kWaveBucket = 64;
static_assert(kWaveBucket == 1 << 6 && kBucketCap == 1 << 8, "bucket_places_log2");
static inline int bucket_places_log2(int bf) { return bf <= 4 ? 6 : bf <= 8 ? 7 : 8; }
// Counters of neighbouring buckets lie half a fan-out apart (its power of two): additions to one line of memory wait for each
// other (9 ns each, and a round makes a fan-out of them for each of the counters in it).  Side by side, 32 a line: builds of 8 x 8192 keys 238.5
// us, now 222.5, 8 x 4001 194 / 186, 8 x 20000 at a fan-out of 64 410 / 385, 8 x 32768 564 / 558.
static inline int bucket_count_log2(int bf) { return bf <= 2 ? 0 : bf <= 4 ? 1 : bf <= 8 ? 2 : bf <= 16 ? 3 : bf <= 32 ? 4 : 5; }
constexpr int kCounterStride = 32;
struct AssignCounting {
    int32_t* counts;
    int32_t* members;
    float* dists;
    int32_t* big;
    int32_t* big_count;
    int2* more;
    int32_t* more_count;
    float* more_dist;
    int32_t* lost;
    int32_t* lost_count;
    int32_t* zero;
    int places_log2, count_log2;
};

// item `it` of tree t was assigned to centroid k, at distance d (k < 0: to none)
__device__ __forceinline__ void count_item(const AssignCounting& ac, int t, int K, int n_c, int k, int it, float d) {
    if (k < 0) {
        if (ac.dists != nullptr) ac.lost[(size_t)t * n_c + atomicAdd(&ac.lost_count[t * kCounterStride], 1)] = it;
        return;
    }
    const size_t b = (size_t)t * K + k;
    const int pos = atomicAdd(&ac.counts[b << ac.count_log2], 1);
    if (pos == kWaveBucket) ac.big[(size_t)t * K + atomicAdd(&ac.big_count[t * kCounterStride], 1)] = k;
    if (pos < 1 << ac.places_log2) {
        ac.members[(b << ac.places_log2) + pos] = it;
        if (ac.dists != nullptr) ac.dists[(b << ac.places_log2) + pos] = d;
    } else {  // (one atomic for the lanes of the wave that are here)
        const unsigned long long here = __ballot(1);
        const int lane = threadIdx.x & 63, leader = __ffsll((long long)here) - 1;
        int base = 0;
        if (lane == leader) base = atomicAdd(&ac.more_count[t * kCounterStride], __popcll(here));
        base = __shfl(base, leader, 64);
        ac.more[(size_t)t * n_c + base + __popcll(here & ((1ull << lane) - 1ull))] = make_int2(k, it);
        if (ac.dists != nullptr) ac.more_dist[(size_t)t * n_c + it] = d;
    }
}

// The centroids that still take items, put side by side (packing rounds from the second on: most
// blocks are full by then, and a round multiplies every unplaced item with every centroid it is
// given).  ids (T, K): the centroids with room, in increasing order; count (T): how many; the
// assignment then walks tiles and norms holding only those (same arrays' shapes as the full ones)
// and translates the column it finds back through ids.  Both NULL: all centroids, as they lie.
struct AssignOpen {
    const int32_t* count;
    const int32_t* ids;
};

// Exclusive prefix sums of n numbers by a workgroup of 256 threads, 1024 numbers a step; every
// thread returns the total.
template <typename Load, typename Store>
__device__ __forceinline__ int block_exclusive_scan(int n, Load load, Store store) {
    __shared__ int32_t s_w[4];
    __shared__ int32_t s_carry;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (threadIdx.x == 0) s_carry = 0;
    __syncthreads();
    for (int base = 0; base < n; base += 1024) {
        const int k0 = base + (int)threadIdx.x * 4;
        int v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = k0 + j < n ? load(k0 + j) : 0;
        const int mine = v[0] + v[1] + v[2] + v[3];
        int inc = mine;  // inclusive scan in the wave
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int o = __shfl_up(inc, off, 64);
            if (lane >= off) inc += o;
        }
        if (lane == 63) s_w[wave] = inc;
        __syncthreads();
        int before = s_carry;
        for (int w = 0; w < wave; ++w) before += s_w[w];
        int run = before + inc - mine;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (k0 + j < n) store(k0 + j, run);
            run += v[j];
        }
        __syncthreads();
        if (threadIdx.x == 255) s_carry = before + inc;
        __syncthreads();
    }
    return s_carry;
}

// ---- centroids as operands of v_mfma_f32_16x16x32_bf16 --------------------------------------
// A tile holds 16 centroids of up to 32 * KS columns (zeros behind the last one), each split into two
// bf16 numbers, c = hi + lo: 2 * KS * 64 chunks of 16 bytes, chunk (half, s, kb, i) at half*KS*64 + s*64 +
// kb*16 + i = columns [s*32 + kb*8, +8) of centroid i of the tile.  A tree has Kt tiles (whole stages
// of the assignment kernels).  Beside them, per centroid (T, Kt*16):
//   n2   ||hi + lo||^2, +inf for a centroid that takes no items
//   lo   a bound of ||c - hi||: what a score made of `hi` alone can be off by, per unit of ||x||
struct CentroidTiles {
    uint4* tiles;
    float* n2;
    float* lo;
};

// Eight numbers as two bf16 halves each, v = hi + lo; joined to ss: the squares of hi + lo, to ls: those of v - hi.
__device__ __forceinline__ void split_bf16(const float (&v)[8], uint4& hi, uint4& lo, float& ss, float& ls) {
    uint32_t h[4], l[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        h[e] = pack_bf16(v[2 * e], v[2 * e + 1]);
        const float d0 = v[2 * e] - bf16_lo(h[e]), d1 = v[2 * e + 1] - bf16_hi(h[e]);
        l[e] = pack_bf16(d0, d1);
        const float w0 = bf16_lo(h[e]) + bf16_lo(l[e]), w1 = bf16_hi(h[e]) + bf16_hi(l[e]);
        ss += w0 * w0;
        ls += d0 * d0;
        ss += w1 * w1;
        ls += d1 * d1;
    }
    hi = make_uint4(h[0], h[1], h[2], h[3]);
    lo = make_uint4(l[0], l[1], l[2], l[3]);
}

// Columns 8 j .. 8 j + 7 of centroid k of tree t (zeros behind the last one) into its tile; `lanes` (a power of two, at
// least 4 KS) consecutive lanes hold a centroid.
__device__ __forceinline__ void emit_columns(const float (&v)[8], int j, int lanes, bool have, int KS, int Kt, int t, int k,
                                             bool usable, const CentroidTiles& ct) {
    float ss = 0.0f, ls = 0.0f;
    if (have && j < KS * 4) {
        const int s = j >> 2, kb = j & 3, i = k & 15;
        uint4* out = ct.tiles + ((size_t)t * Kt + (k >> 4)) * (size_t)(2 * KS * 64);
        uint4 hi, lo;
        split_bf16(v, hi, lo, ss, ls);
        out[s * 64 + kb * 16 + i] = hi;
        out[KS * 64 + s * 64 + kb * 16 + i] = lo;
    }
    ss = group_sum_of(ss, lanes);
    ls = group_sum_of(ls, lanes);
    if (have && j == 0) {
        ct.n2[(size_t)t * Kt * 16 + k] = usable ? ss : INFINITY;
        // (1e-5 of ||c|| per 32 columns: what the roundings of two sums of products can be worth)
        ct.lo[(size_t)t * Kt * 16 + k] = sqrtf(ls) * 1.0001f + (float)KS * 1e-5f * sqrtf(ss);
    }
}

// Centroid k of tree t, D fp32 numbers at c (LDS or memory), into its tile; called by the 64
// lanes of one wave.
__device__ __forceinline__ void emit_centroid(const float* c, int D, int KS, int Kt, int t, int k,
                                              bool usable, const CentroidTiles& ct) {
    const int j = threadIdx.x & 63;
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = j < KS * 4 && j * 8 + e < D ? c[j * 8 + e] : 0.0f;
    emit_columns(v, j, 32, true, KS, Kt, t, k, usable, ct);
}

// What an assignment launch works on.
struct AssignJob {
    const void* x;          // (T, n_c, D) items
    int n_c;
    const int32_t* n_live;  // (T): the first so many of them only, or NULL
    size_t x_tree_stride;
    int dtype, D, num_trees;
    CentroidTiles ct;       // centroids as operand tiles (all, or the open ones)
    const float* cent;      // (T, K, D) fp32
    int K;
    const int32_t* list;    // NULL: all items, else the items list[0 .. *list_count) of each tree
    const int32_t* list_count;
    int32_t* assign;        // (T, n_c) and
    float* dist;            // (T, n_c): where the result goes if nothing is counted
    AssignCounting counting;
    AssignOpen open;
    int after_approx;       // the approximate pass has been over it: only what it left is left
    int32_t* unsure;        // (T, n_c) / (T): items the approximate pass leaves to an exact one
    int32_t* unsure_count;
};

// Grids of `blocks` workgroups to each of `trees` trees, trees in the fast index: workgroups go to the eight XCDs in
// turn by their number, so a tree's run behind the same L2s in one launch after the other, and what a launch
// wrote is there for the next.  (Trees in the slow index: every tile and bucket came from another XCD's L2 or
// from memory; builds of 8 x 32768 keys 729 -> 703 us, of 8 x 131072 3440 -> 3410.)
static inline dim3 tree_grid(long long blocks, int trees) {
    const long long y = blocks < 32768 ? (blocks > 0 ? blocks : 1) : 32768;
    return dim3((unsigned)trees, (unsigned)y, (unsigned)((blocks + y - 1) / y > 0 ? (blocks + y - 1) / y : 1));
}
__device__ __forceinline__ int tree_block() { return (int)(blockIdx.y + blockIdx.z * gridDim.y); }
__device__ __forceinline__ int tree_blocks() { return (int)(gridDim.y * gridDim.z); }

// (all trees together) more items than this on a list, and the approximate pass takes it
constexpr int kApproxListItems = 256 * 256;

__device__ __forceinline__ int items_of(const AssignJob& job, int t) {
    if (job.list != nullptr) return job.list_count[t * kCounterStride];
    return job.n_live != nullptr ? min(max(job.n_live[t], 0), job.n_c) : job.n_c;
}
// what was found for item `it`: into its bucket, or as it is
__device__ __forceinline__ void put_result(const AssignJob& job, int t, int it, int k, float d) {
    if (job.counting.counts != nullptr) {
        count_item(job.counting, t, job.K, job.n_c, k, it, d);
    } else {
        job.assign[(size_t)t * job.n_c + it] = k;
        job.dist[(size_t)t * job.n_c + it] = d;
    }
}

// The current device, for what is asked once per kernel and device.
constexpr int kMaxDevices = 64;
static inline int current_device() {
    int dev = 0;
    return hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < kMaxDevices ? dev : -1;
}
// (more than 64 KiB of dynamic LDS has to be asked for: once per kernel and device)
static inline int ask_for_lds(const void* kernel, size_t smem, int* asked, int dev) {
    if (dev < 0) return fail(HIRA_ELAUNCH, "assignment: no current device");
    if (__atomic_load_n(&asked[dev], __ATOMIC_RELAXED) == 0) {
        if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess)
            return fail(HIRA_ELAUNCH, "assignment: %zu bytes of LDS refused", smem);
        __atomic_store_n(&asked[dev], 1, __ATOMIC_RELAXED);
    }
    return HIRA_OK;
}

// assign_mfma.hip
int assign_ks(int dtype, int D);        // KS of the operand tiles for rows of D columns, 0: none
bool assign_exact_on_mfma(int dtype, int D);
bool assign_approx_pays(int dtype, int D, int K);
int assign_tiles(int K);
int launch_cent_prep(int dim, const float* cent, int K, int num_trees, const int32_t* fill, int bf,
                     void* tiles, float* cn2, hipStream_t s);
int launch_assign_mfma(const AssignJob& job, hipStream_t s);
int launch_assign_approx(const AssignJob& job, hipStream_t s);
int launch_open_centroids(int KS, const CentroidTiles& ct, const int32_t* fill, int bf, int K,
                          int num_trees, int32_t* open_ids, int32_t* open_count,
                          const CentroidTiles& open, hipStream_t s);

}  // namespace hira
