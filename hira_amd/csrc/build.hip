// Index build: bottom-up k-means-style ball tree in the fixed-fan-out layout.
//
// For each level l = 1 .. L-1 the n_c items of the level below (keys for l = 1, the
// centres of level l-1 above that) are clustered into K = ceil(n_c / bf) groups of at most
// bf items:
//   1. K initial centroids = evenly strided, seeded sample of the items;
//   2. `niter` Lloyd rounds: nearest-centroid assignment, then centroid = mean of members
//      (members are bucketed and summed in a fixed order, so the result is reproducible);
//   3. capacity packing: every item proposes to its nearest centroid that still has room,
//      each centroid takes the closest proposers first (the rule of the reference's GPU
//      build, indexer/cuda.py:247-307), the rest try again against the centroids that are
//      not full yet; what is still unplaced after `pack_rounds` fills free slots in order
//      (the reference drops such items into random free slots, indexer/cuda.py:309-334);
//   4. the centre of a block = mean of the items that ended up in it, rounded to the
//      storage dtype.
// Then the levels are laid out top-down (children of slot p at [p*bf, (p+1)*bf)), keys and
// values are gathered once into slot order, and radii are taken bottom-up from the final
// layout: r_p = max over children (||c_child - c_p|| + r_child), the bound of
// indexer/cpu.py:286-309 / indexer/cuda.py:114-198, against the ROUNDED centres and
// nudged up by a few ulp so that rounding never makes a ball too small.
#include "assign.h"
#include "cluster.h"
#include "small_levels.h"

namespace hira {

// ------------------------------------------------------------------------------------
// small helpers
// ------------------------------------------------------------------------------------
// what the phases of a level count, per tree: items on the two lists, items behind the buckets (of
// this round, of the next), items the approximate assignment leaves, items without a centroid, large
// buckets (of this round, of the next)
constexpr int kBuildCounters = 8;

__global__ void k_fill_i32(int32_t* p, size_t n, int32_t v) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// Kernels with a wave per node: four nodes a workgroup (a workgroup of one wave costs its dispatch).
constexpr int kNodeThreads = 256;
static dim3 node_grid(int nodes, int trees) { return tree_grid((nodes + kNodeThreads / 64 - 1) / (kNodeThreads / 64), trees); }
__device__ __forceinline__ int node_of_wave() {
    return __builtin_amdgcn_readfirstlane(tree_block() * (kNodeThreads / 64) + (threadIdx.x >> 6));
}

// ------------------------------------------------------------------------------------
// 1. what a level starts from, in one launch: empty blocks, zero counters, the initial centroids: centroid k is item
//    floor((k + u_k) * n_c / K), u_k in [0,1) from the seed.
//    n_live != NULL: tree t holds n_live[t] <= n_c items, the first ones of its rows, and uses its first
//    K_t = ceil(n_t / bf) centroids only: the others count as full.
//    ct.tiles != NULL: the centroids also go into their operand tiles (those that count as full take no items); the
//    columns that pad the last stage of tiles are zeros that take no items.
//    `lanes` (a power of two) hold a centroid, eight columns each, so that a wave takes several: bound by its
//    instructions (the random number, the split into halves), 8 x 4096 centroids of 128 columns 13.5 us, 27 with a
//    centroid a wave, most of whose lanes had no columns.  With the filling as a launch of its own ahead a build took 1 to 5 us more
//    (8 x 8192 keys 253.5 -> 251.7, 4 x 5003 x 80 fp32 644 -> 640).
// ------------------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(kNodeThreads) void k_level_init(
    const void* x, int n_c, size_t x_tree_stride, int K, int bf, int D, uint64_t seed, float* cent, const int32_t* n_live, int32_t* fill,
    int32_t* slots, int32_t* counts, int32_t* counters /* (kBuildCounters, T) */,
    float* absmax /* (T, kAbsCopies, D) or NULL */, int Kt, CentroidTiles ct, int KS, int lanes, int count_log2) {
    constexpr int EPL = Elem<T>::kPerChunk, CH = 8 / EPL;
    const int t = blockIdx.x, lane = threadIdx.x & 63, j = lane % lanes;
    const int k = node_of_wave() * (64 / lanes) + lane / lanes, own = min(k, K - 1);
    const int n_t = n_live ? min(max(n_live[t], 0), n_c) : n_c;
    const int K_t = n_live ? min(max((n_t + bf - 1) / bf, 1), K) : K;
    // ---- the centroid's item: on its way while the arrays are filled ---------------------------------
    const long long idx = first_centroid(seed, t, own, max(n_t, 1), K_t);
    const size_t src = ((size_t)t * x_tree_stride + (size_t)idx) * D;
    uint4 raw[CH];
#pragma unroll
    for (int h = 0; h < CH; ++h) {
        raw[h] = make_uint4(0, 0, 0, 0);
        if ((j * CH + h) * EPL < D) raw[h] = load_chunk<T>(x, src, j * CH + h);
    }

    const int stride = tree_blocks() * blockDim.x, T_ = gridDim.x;
    const int i0 = tree_block() * blockDim.x + threadIdx.x;
    if (i0 < kBuildCounters) counters[(i0 * T_ + t) * kCounterStride] = 0;
    if (absmax != nullptr)
        for (int i = i0; i < kAbsCopies * D; i += stride) absmax[(size_t)t * kAbsCopies * D + i] = 0.0f;
    for (int i = i0; i < K; i += stride) {
        fill[(size_t)t * K + i] = i >= K_t ? bf : 0;
        counts[((size_t)t * K + i) << count_log2] = 0;
    }
    for (size_t i = i0; i < (size_t)K * bf; i += stride) slots[(size_t)t * K * bf + i] = -1;
    if (ct.tiles != nullptr) {
        const int pad = Kt * 16 - K, cpc = KS * 8;  // chunks of a column: hi and lo halves
        for (int i = i0; i < pad * cpc; i += stride) {
            const int kp = K + i / cpc, c = i % cpc;
            const int half = c / (KS * 4), jc = c % (KS * 4);
            ct.tiles[((size_t)t * Kt + (kp >> 4)) * (size_t)(2 * KS * 64) + half * KS * 64 + (jc >> 2) * 64 +
                     (jc & 3) * 16 + (kp & 15)] = make_uint4(0, 0, 0, 0);
        }
        for (int i = i0; i < pad; i += stride) {
            ct.n2[(size_t)t * Kt * 16 + K + i] = INFINITY;
            ct.lo[(size_t)t * Kt * 16 + K + i] = 0.0f;
        }
    }

    float v[8];
#pragma unroll
    for (int h = 0; h < CH; ++h) {
        float f[EPL];
        unpack<T>(raw[h], f);
#pragma unroll
        for (int e = 0; e < EPL; ++e) v[h * EPL + e] = f[e];
    }
    float* dst = cent + ((size_t)t * K + own) * D + j * 8;
#pragma unroll
    for (int h = 0; h < 2; ++h)  // (rows are whole fours)
        if (k < K && j * 8 + h * 4 < D) *reinterpret_cast<float4*>(dst + h * 4) = make_float4(v[h * 4], v[h * 4 + 1], v[h * 4 + 2], v[h * 4 + 3]);
    if (ct.tiles != nullptr) emit_columns(v, j, lanes, k < K, KS, Kt, t, own, own < K_t, ct);
}

// ------------------------------------------------------------------------------------
// 2. nearest centroid (vector-ALU kernel): argmin_k ||x_i - c_k||^2, lowest k on ties.
//    LPR lanes hold one item row; each lane group keeps PPG items in registers and walks the centroids, kAhead of
//    them asked for at a time.  `share` waves of a workgroup hold the same items and walk every share-th centroid, as
//    many as the chip has waves for; the best of theirs meet in LDS.  fill != NULL: centroids with fill[k] >= bf are
//    skipped.
//    Long lists are bound by the vector ALUs and the L2s that the centroids come from, short ones (what the approximate
//    pass leaves: a few hundred items a tree) by the walk's trips to memory, which is why they are shared out and
//    asked for several at a time: a wave to its items and a trip a centroid took such a list 317 us for 4 x 8000 fp32 items of 128
//    columns and 500 centroids, now 31; builds of 4 x 8000 keys at a fan-out of 16 1787 -> 501 us, of 8 x 20000 at 32
//    2335 -> 897, of 1 x 90000 at 8 32.8 -> 4.1 ms.
// ------------------------------------------------------------------------------------
constexpr int kPPG = 4;
constexpr int kSimpleThreads = 512;
constexpr int kSimpleWaves = kSimpleThreads / 64;
static_assert(kSimpleWaves == 1 << 3, "simple_share_log2");
constexpr int kSimpleBlocks = 1024;  // workgroups of all trees, at most: they go through a list in strides

// Waves that share a set of items, of which each of `trees` trees has `sets` (as a power of two): the number whose
// rounds of waves take least, a wave's items and its end as long as a dozen centroids.
__device__ __forceinline__ int simple_share_log2(int sets, int trees, int K) {
    constexpr int kFixed = 12, kOnChipLog2 = 12;
    int best = 0;
    long long least = 0;
#pragma unroll
    for (int s = 0; s <= 3; ++s) {
        const long long rounds = (((long long)sets * trees << s) + (1 << kOnChipLog2) - 1) >> kOnChipLog2;
        const long long cost = rounds * (kFixed + ((K + (1 << s) - 1) >> s));
        if (s == 0 || cost < least) {
            best = s;
            least = cost;
        }
    }
    return best;
}

template <typename T, int LPR>
__global__ __launch_bounds__(kSimpleThreads, 4) void k_assign_simple(const int32_t* fill, int bf, const AssignJob job) {
    constexpr int EPL = Elem<T>::kPerChunk, RPW = kWave / LPR, SET = RPW * kPPG;
    constexpr int kAhead = EPL == 8 ? 2 : 4;
    __shared__ float s_b[kSimpleWaves][SET];
    __shared__ int s_g[kSimpleWaves][SET];
    const int lane = lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int rg = lane / LPR, ch = lane % LPR;
    const int t = blockIdx.x;
    const int n_items = items_of(job, t), n_c = job.n_c, D = job.D, K = job.K;
    if (job.counting.zero != nullptr && blockIdx.y == 0 && threadIdx.x == 0) job.counting.zero[t * kCounterStride] = 0;
    const int sets = (n_items + SET - 1) / SET, share_log2 = simple_share_log2(sets, gridDim.x, K), share = 1 << share_log2;
    const int part = wave & (share - 1), per_block = kSimpleWaves >> share_log2;
    const bool chunk_ok = ch * EPL < D;
    const float* ct = job.cent + (size_t)t * K * D + (chunk_ok ? ch * EPL : 0);
    const int32_t* ft = fill ? fill + (size_t)t * K : nullptr;

    for (int b = blockIdx.y; b * per_block < sets; b += gridDim.y) {  // uniform
        const int first = (b * per_block + (wave >> share_log2)) * SET;
        float xf[kPPG][EPL], best[kPPG];
        int arg[kPPG];
#pragma unroll
        for (int p = 0; p < kPPG; ++p) {
            const int pos = first + p * RPW + rg;
            int item = -1;
            if (pos < n_items) item = job.list ? job.list[(size_t)t * n_c + pos] : pos;
            uint4 raw = make_uint4(0, 0, 0, 0);
            if (item >= 0 && chunk_ok) raw = load_chunk<T>(job.x, ((size_t)t * job.x_tree_stride + item) * D, ch);
            unpack<T>(raw, xf[p]);
            best[p] = INFINITY;
            arg[p] = -1;
        }
        // my centroids: part, part + share, ..., 64 of them looked up at a time
        for (int k0 = part; k0 < K && first < n_items; k0 += share * 64) {  // uniform in the wave
            const int kl = k0 + lane * share;
            unsigned long long left = __ballot(kl < K && !(ft && ft[min(kl, K - 1)] >= bf));
            while (left) {
                int k[kAhead];
                float4 c[kAhead][EPL / 4];
#pragma unroll
                for (int u = 0; u < kAhead; ++u) {  // (behind the last one: that one again)
                    k[u] = left ? k0 + (__ffsll((long long)left) - 1) * share : k[u > 0 ? u - 1 : 0];
                    left &= left - (left ? 1ull : 0ull);
#pragma unroll
                    for (int e = 0; e < EPL / 4; ++e)
                        c[u][e] = reinterpret_cast<const float4*>(ct + (size_t)k[u] * D)[e];
                }
#pragma unroll
                for (int u = 0; u < kAhead; ++u)
#pragma unroll
                    for (int p = 0; p < kPPG; ++p) {
                        float ss = 0.0f;
#pragma unroll
                        for (int e = 0; e < EPL / 4; ++e) {
                            const float cf[4] = {c[u][e].x, c[u][e].y, c[u][e].z, c[u][e].w};
#pragma unroll
                            for (int i = 0; i < 4; ++i) {
                                const float df = xf[p][e * 4 + i] - cf[i];
                                ss += df * df;
                            }
                        }
                        ss = group_sum<LPR>(chunk_ok ? ss : 0.0f);
                        if (ss < best[p]) {  // (centroids come in increasing order: ties keep the lower one)
                            best[p] = ss;
                            arg[p] = k[u];
                        }
                    }
            }
        }
        if (ch == 0) {
#pragma unroll
            for (int p = 0; p < kPPG; ++p) {
                s_b[wave][p * RPW + rg] = best[p];
                s_g[wave][p * RPW + rg] = arg[p];
            }
        }
        __syncthreads();
        if (part == 0) {
            for (int i = lane; i < SET && first + i < n_items; i += 64) {
                float d = s_b[wave][i];
                int g = s_g[wave][i];
                for (int w = wave + 1; w < wave + share; ++w) {  // uniform
                    const float od = s_b[w][i];
                    const int og = s_g[w][i];
                    if (og >= 0 && (g < 0 || od < d || (od == d && og < g))) {
                        d = od;
                        g = og;
                    }
                }
                put_result(job, t, job.list ? job.list[(size_t)t * n_c + first + i] : first + i, g, d);
            }
        }
        __syncthreads();
    }
}

// ------------------------------------------------------------------------------------
// 3. the buckets of a round: what the assignment left of it (assign.h)
// ------------------------------------------------------------------------------------
struct Buckets {
    int32_t* counts;          // (T, K), 1 << count_log2 apart; every kernel here leaves it zero for the round after it
    const int32_t* members;   // (T, K, places)
    const float* dists;       // (T, K, places)
    const int32_t* big;       // (T, K)
    const int32_t* big_count;   // (T)
    const int2* more;         // (T, n_c)
    const int32_t* more_count;  // (T)
    const float* more_dist;     // (T, n_c)
    int32_t* next_big_count;    // (T): the round after this one counts here; cleared by these kernels
    int32_t* next_more_count;   // (T): the same
    int32_t* unsure_count;      // (T): cleared by these kernels
    int places_log2, count_log2;
    __device__ int32_t& count(size_t b) const { return counts[b << count_log2]; }
    __device__ int places() const { return 1 << places_log2; }
    __device__ size_t first(size_t b) const { return b << places_log2; }  // place of bucket b (of all trees)
};

// f(item) for the items of bucket k among entries [e0, e1) of those that do not lie in `members`;
// called by the whole workgroup
template <typename F>
__device__ __forceinline__ void for_more(const Buckets& b, int t, int n_c, int k, int e0, int e1, F f) {
    constexpr int U = 8;  // entries on their way at a time
    const int2* more = b.more + (size_t)t * n_c;
    for (int e = e0 + (int)threadIdx.x; e < e1; e += U * (int)blockDim.x) {
        int2 v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = e + u * (int)blockDim.x < e1 ? more[e + u * (int)blockDim.x] : make_int2(-1, 0);
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (v[u].x == k) f(v[u].y);
    }
}

// The order in which a bucket's members arrive depends on the run; everything that follows works
// on them in a fixed order.  Most buckets have about `bf` members (32 or so): a wave has one to
// itself, ranks each lane's member against the others' in registers and works on without a barrier
// (kWaveBucket members at most; a workgroup per bucket spent its time on five barriers and on 224
// idle threads).  The larger ones, which the assignment has listed, take a workgroup each; the
// launch's first workgroups do those, so that the longest start first:
//   up to its places    every thread ranks its member against all others
//   more                a bit map of the members (means), a bitonic sorting network (packing)
constexpr int kWaves = 4;  // of a workgroup of the per-bucket kernels
// Workgroups of a tree for large buckets.  (An eighth of the buckets: 8 x 8192 keys 254 us a build, 248 with a quarter, 8 x 20000
// at a fan-out of 64 427 / 417; 512 instead of 256 at most: 8 x 131072 keys 3225 / 3235.)
static int large_blocks(int K) { return min(max(K / 4, 1), 256); }
constexpr int kBucketThreads = 256;

template <typename Key>
__device__ __forceinline__ void bitonic_sort(Key* a, int P) {  // (a barrier ahead of the first step)
    for (int k = 2; k <= P; k <<= 1)
        for (int j = k >> 1; j > 0; j >>= 1) {
            __syncthreads();
            for (int i = threadIdx.x; i < P; i += kBucketThreads) {
                const int x = i ^ j;
                if (x > i) {
                    const Key u = a[i], v = a[x];
                    if ((u > v) == ((i & k) == 0)) {
                        a[i] = v;
                        a[x] = u;
                    }
                }
            }
        }
    __syncthreads();
}

__device__ __forceinline__ int pow2_at_least(int n) {
    int p = 1;
    while (p < n) p <<= 1;
    return p;
}

// what the wave, or the workgroup, that has read the count of its bucket does for the round after it
// (behind a barrier: the count is read through the scalar cache, and only the wait there keeps this
// store from overtaking it; a bucket's other reader finds a large count, or none, and leaves it)
__device__ __forceinline__ void reset_count(const Buckets& b, int t, int k, int K) {
    b.count((size_t)t * K + k) = 0;
}
__device__ __forceinline__ void reset_round(const Buckets& b, int t) {  // (one thread of the tree)
    b.next_big_count[t * kCounterStride] = 0;
    b.next_more_count[t * kCounterStride] = 0;
    b.unsure_count[t * kCounterStride] = 0;
}

// ------------------------------------------------------------------------------------
// 4. Lloyd round: centroid = mean of the member rows: the members in the order of their item ids,
//    row e summed by row group e % R, the R sums added in order, so the result does not depend on the
//    order of arrival.  (A row is CPR threads of 16 bytes, R = 256 / CPR rows at a time: 256 threads of a
//    workgroup, or four times the 64 lanes of a wave.)  An empty centroid keeps its value.
//    ct.tiles != NULL: the new centroid also goes into its operand tile.
//    What bounds it is the latency of each bucket's chain (count, members, rows, sums): 6 us a workgroup of four
//    small ones, 20 to 45 us a large one (up to 1473 rows at 8 x 131072 items, beside a mean of 32), so what
//    counts is how many are on a compute unit: six workgroups (76 registers, 18 KiB), with fewer rows on their way in
//    each.  8 x 32768 rows of 256 bytes 26 us, 8 x 131072 75 us (33 and 92 with four workgroups of 108 registers, twice the
//    rows on their way and a quarter of the sums added up one load after the other).
// ------------------------------------------------------------------------------------
constexpr int kMeanMap = 2048;  // words of a bit map of item ids, for buckets beyond their places
constexpr int kMeanMapBits = kMeanMap * 32;

template <typename T>
__global__ __launch_bounds__(kBucketThreads, 6) void k_bucket_mean(
    const void* x, size_t x_tree_stride, int n_c, int K, int D, const Buckets bk,
    const int32_t* fill, int bf, float* cent, int Kt, const CentroidTiles ct, int KS, int large) {
    constexpr int EPL = Elem<T>::kPerChunk;
    constexpr int kPart = kBucketThreads * EPL;  // (R, D) partial sums, R * D <= 256 * EPL
    constexpr int kPiece = kWaveMeanPiece<T>;    // a quarter of them
    // one bucket: partial sums, ids in order or their bit map, counts of the bit map's stretches;
    // or, a wave each: a quarter of the partial sums
    __shared__ __attribute__((aligned(16))) float s_lds[kPart + kMeanMap + kBucketThreads];
    __shared__ uint32_t s_ids[kWaves][kWaveBucket];
    static_assert(kWaves * kPiece <= kPart, "a quarter for every wave");
    const int t = blockIdx.x, block = tree_block(), tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int CPR = D / EPL, R = kBucketThreads / CPR;
    auto usable = [&](int k) { return !(fill != nullptr && fill[(size_t)t * K + k] >= bf); };
    if (block == 0 && tid == 0) reset_round(bk, t);
    if (block >= large) {
        const int k = (block - large) * kWaves + wave;
        if (k >= K) return;
        uint32_t id = (uint32_t)bk.members[bk.first((size_t)t * K + k) + lane];  // (garbage from m on)
        const int m = __builtin_amdgcn_readfirstlane(bk.count((size_t)t * K + k));
        if (m <= 0 || m > kWaveBucket) return;
        if (lane >= m) id = 0xffffffffu;
        const int rank = wave_rank(id, m);
        if (lane < m) s_ids[wave][rank] = id;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        if (lane == 0) reset_count(bk, t, k, K);
        float* piece = s_lds + wave * kPiece;
        wave_mean<T, 1>(x, (size_t)t * x_tree_stride, [&](int e) { return s_ids[wave][e]; }, m, D, piece,
                        cent + ((size_t)t * K + k) * D);
        if (ct.tiles != nullptr) emit_centroid(piece, D, KS, Kt, t, k, usable(k), ct);
        return;
    }
    // ---- the large ones --------------------------------------------------------------------------
    float* s_part = s_lds;
    uint32_t* s_ord = reinterpret_cast<uint32_t*>(s_lds + kPart);
    int32_t* s_small = reinterpret_cast<int32_t*>(s_lds + kPart + kMeanMap);
    const int nbig = bk.big_count[t * kCounterStride];
    for (int i = block; i < nbig; i += large) {  // uniform
        const int k = bk.big[(size_t)t * K + i];
        const int m = bk.count((size_t)t * K + k);
        const int32_t* mem = bk.members + bk.first((size_t)t * K + k);
        __syncthreads();
        if (tid == 0) reset_count(bk, t, k, K);
        const int r = tid / CPR, c = tid % CPR;
        float acc[EPL];
#pragma unroll
        for (int e = 0; e < EPL; ++e) acc[e] = 0.0f;
        // rows [e0, e0 + n) in order, their ids at ids[0 .. n)
        auto add_rows = [&](const uint32_t* ids, int e0, int n) {
            constexpr int U = 4;  // rows on their way at a time
            if (r < R)
                for (int e = e0 + (r - e0 % R + R) % R; e < e0 + n; e += U * R) {
                    uint4 raw[U];
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        raw[u] = make_uint4(0, 0, 0, 0);
                        if (e + u * R < e0 + n)
                            raw[u] = load_chunk<T>(x, ((size_t)t * x_tree_stride + (int)ids[e + u * R - e0]) * D, c);
                    }
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        float f[EPL];
                        unpack<T>(raw[u], f);
                        if (e + u * R < e0 + n) {
#pragma unroll
                            for (int q = 0; q < EPL; ++q) acc[q] += f[q];
                        }
                    }
                }
        };
        if (m <= bk.places()) {
            const int mine = tid < m ? mem[tid] : 0x7fffffff;
            s_small[tid] = mine;
            __syncthreads();
            int rank = 0;
            for (int j = 0; j < m; ++j) rank += s_small[j] < mine;
            if (tid < m) s_ord[rank] = (uint32_t)mine;
            __syncthreads();
            add_rows(s_ord, 0, m);
        } else {
            // ids in ranges of kMeanMapBits: a bit per member, then the set bits in order, as many of
            // them at a time as there is room for in s_part
            uint32_t* piece = reinterpret_cast<uint32_t*>(s_part);
            constexpr int W = kMeanMap / kBucketThreads;
            const int others = bk.more_count[t * kCounterStride];
            int written = 0;
            for (int lo = 0; lo < n_c; lo += kMeanMapBits) {
                __syncthreads();
                const int per = min(W, (n_c - lo + 32 * kBucketThreads - 1) / (32 * kBucketThreads));
                for (int i = tid; i < per * kBucketThreads; i += kBucketThreads) s_ord[i] = 0;
                __syncthreads();
                auto mark = [&](int it) {
                    const int d = it - lo;
                    if (d >= 0 && d < kMeanMapBits) atomicOr(&s_ord[d >> 5], 1u << (d & 31));
                };
                if (tid < bk.places()) mark(mem[tid]);
                for_more(bk, t, n_c, k, 0, others, mark);
                __syncthreads();
                // thread `tid` owns the words [tid * per, (tid + 1) * per)
                const int in_range = block_exclusive_scan(
                    kBucketThreads, [&](int i) {
                        int n = 0;
                        for (int u = 0; u < per; ++u) n += __popc(s_ord[i * per + u]);
                        return n;
                    },
                    [&](int i, int v) { s_small[i] = v; });
                __syncthreads();
                for (int p0 = 0; p0 < in_range; p0 += kPart) {
                    int at = s_small[tid];
                    for (int u = 0; u < per; ++u) {
                        uint32_t bits = s_ord[tid * per + u];
                        while (bits) {
                            const int b = __ffs(bits) - 1;
                            bits &= bits - 1;
                            if (at >= p0 && at < p0 + kPart) piece[at - p0] = (uint32_t)(lo + (tid * per + u) * 32 + b);
                            ++at;
                        }
                    }
                    __syncthreads();
                    add_rows(piece, written + p0, min(kPart, in_range - p0));
                    __syncthreads();
                }
                written += in_range;
            }
        }
        __syncthreads();
        if (r < R) {
#pragma unroll
            for (int q = 0; q < EPL; ++q) s_part[r * D + c * EPL + q] = acc[q];
        }
        __syncthreads();
        const int rows = min(R, m);
        for (int j = tid; j < D; j += kBucketThreads) {
            float s = 0.0f;
            for (int q = 0; q < rows; ++q) s += s_part[q * D + j];
            const float v = s / (float)m;
            cent[((size_t)t * K + k) * D + j] = v;
            s_part[j] = v;  // (nobody else reads column j)
        }
        __syncthreads();
        if (ct.tiles != nullptr && wave == 0) emit_centroid(s_part, D, KS, Kt, t, k, usable(k), ct);
    }
}

// A wave per block (wave_block_mean).  Bound by the gather of the rows: 8 x 131072 rows of 256 bytes 44 us, 6.1 TB/s
// (60 with the centres rounded by shifts and stored a number at a time)
template <typename T>
__global__ __launch_bounds__(kNodeThreads) void k_block_mean(const void* x, size_t x_tree_stride, int K,
                                                             int D, const int32_t* slots, int bf, int lpr,
                                                             const float* cent, void* out_t) {
    const int k = node_of_wave(), t = blockIdx.x;
    if (k >= K) return;  // (the whole wave)
    wave_block_mean<T, 8>(x, (size_t)t * x_tree_stride, D,
                          (threadIdx.x & 63) < bf ? slots[((size_t)t * K + k) * bf + (threadIdx.x & 63)] : -1, bf, lpr,
                          ((size_t)t * K + k) * D, cent, out_t);
}

// ------------------------------------------------------------------------------------
// 5. capacity packing
// ------------------------------------------------------------------------------------
// The closest proposers of a bucket (by distance, then item id) take the free slots of the block in
// that order; the others go on the list of the next round.  A block that is full now takes no more
// items: its norm in the operand tiles becomes +inf.  (One addition to the list's length per
// workgroup: a tree's 1024 or 4096 buckets would queue up at it.)  What bounds it is the chain count,
// members, place on the list; first round of 8 x 131072 items 159 -> 60 us, of 8 x 32768 45 -> 14.
constexpr int kAcceptSort = 2048;  // keys sorted at a time; larger buckets in several goes, the
                                   // best `take` (at most 64) so far carried along

__global__ __launch_bounds__(kBucketThreads) void k_bucket_accept(
    const Buckets bk, int n_c, int K, int bf, int32_t* fill, int32_t* slots, int32_t* next_list,
    int32_t* next_count, int Kt, float* cn2, int large) {
    __shared__ uint64_t s_keys[kAcceptSort];
    __shared__ int32_t s_back[kWaves];
    __shared__ int32_t s_base, s_rej, s_n;
    const int t = blockIdx.x, block = tree_block(), tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int32_t* nl = next_list + (size_t)t * n_c;
    auto key_of = [](float d, int it) { return ((uint64_t)__float_as_uint(d) << 32) | (uint32_t)it; };
    auto filled = [&](int k, int f) {  // (one thread)
        fill[(size_t)t * K + k] = f;
        if (cn2 != nullptr && f >= bf) cn2[(size_t)t * Kt * 16 + k] = INFINITY;
    };
    if (block == 0 && tid == 0) reset_round(bk, t);
    if (block >= large) {
        const int k = (block - large) * kWaves + wave;
        int m = 0, f = 0, take = 0;
        uint64_t mine = 0;
        if (k < K) {
            const size_t b = (size_t)t * K + k;
            mine = key_of(bk.dists[bk.first(b) + lane], bk.members[bk.first(b) + lane]);  // (garbage from m on)
            m = __builtin_amdgcn_readfirstlane(bk.count(b));
            f = __builtin_amdgcn_readfirstlane(fill[b]);
            if (m > kWaveBucket) m = 0;
            take = max(min(m, bf - f), 0);
            if (lane == 0 && take > 0) filled(k, f + take);
        }
        if (lane >= m) mine = ~0ull;
        if (lane == 0) s_back[wave] = m - take;
        __syncthreads();
        if (lane == 0 && m > 0) reset_count(bk, t, k, K);
        if (tid == 0) {
            const int back = s_back[0] + s_back[1] + s_back[2] + s_back[3];
            s_base = back > 0 ? atomicAdd(&next_count[t * kCounterStride], back) : 0;
        }
        const int rank = wave_rank(mine, m);  // (the addition is on its way)
        __syncthreads();
        if (lane < m) {
            if (rank < take) {
                slots[((size_t)t * K + k) * bf + f + rank] = (int)(uint32_t)mine;
            } else {
                int at = s_base + rank - take;
                for (int w = 0; w < wave; ++w) at += s_back[w];
                nl[at] = (int)(uint32_t)mine;
            }
        }
        return;
    }
    // ---- the large ones --------------------------------------------------------------------------
    const int nbig = bk.big_count[t * kCounterStride];
    for (int i = block; i < nbig; i += large) {  // uniform
        const int k = bk.big[(size_t)t * K + i];
        const size_t b = (size_t)t * K + k;
        const int m = bk.count(b), f = fill[b];
        const int32_t* mem = bk.members + bk.first(b);
        const float* md = bk.dists + bk.first(b);
        const float* more_d = bk.more_dist + (size_t)t * n_c;
        int32_t* my_slots = slots + b * bf + f;
        const int take = max(min(m, bf - f), 0);
        __syncthreads();  // (everybody has read; what the bucket before left in LDS is used)
        if (tid == 0) {
            s_rej = 0;
            s_base = m > take ? atomicAdd(&next_count[t * kCounterStride], m - take) : 0;
            reset_count(bk, t, k, K);
            filled(k, f + take);
        }
        if (m <= bk.places()) {
            const uint64_t own = tid < m ? key_of(md[tid], mem[tid]) : ~0ull;
            s_keys[tid] = own;
            __syncthreads();
            int r = 0;
            for (int j = 0; j < m; ++j) r += s_keys[j] < own;
            if (tid < m) {
                if (r < take) my_slots[r] = (int)(uint32_t)own;
                else nl[s_base + r - take] = (int)(uint32_t)own;
            }
            continue;
        }
        // s_keys[0 .. n): the best so far and those not looked at yet; a kAcceptStep of the others at
        // a time is searched for the bucket's items
        constexpr int kAcceptStep = kAcceptSort - kBucketCap - 64;
        const int others = bk.more_count[t * kCounterStride];
        if (tid < bk.places()) s_keys[tid] = key_of(md[tid], mem[tid]);
        if (tid == 0) s_n = bk.places();
        for (int e0 = 0; e0 < others; e0 += kAcceptStep) {
            __syncthreads();
            for_more(bk, t, n_c, k, e0, min(e0 + kAcceptStep, others),
                     [&](int it) { s_keys[atomicAdd(&s_n, 1)] = key_of(more_d[it], it); });
            __syncthreads();
            const int n = s_n, P = pow2_at_least(n);
            for (int e = n + tid; e < P; e += kBucketThreads) s_keys[e] = ~0ull;
            bitonic_sort(s_keys, P);
            if (tid == 0) s_n = min(take, n);
        }
        __syncthreads();
        for (int r = tid; r < take; r += kBucketThreads) my_slots[r] = (int)(uint32_t)s_keys[r];
        if (m > take) {  // whoever lies behind the last one taken tries again
            const uint64_t last = take > 0 ? s_keys[take - 1] : 0ull;
            auto again = [&](float d, int it) {
                if (take == 0 || key_of(d, it) > last) nl[s_base + atomicAdd(&s_rej, 1)] = it;
            };
            if (tid < bk.places()) again(md[tid], mem[tid]);
            for_more(bk, t, n_c, k, 0, others, [&](int it) { again(more_d[it], it); });
        }
    }
}

// Whatever is still unplaced -- the list the last round left, and items that have no nearest
// centroid -- goes to the free slots in order: the u-th of them (by item id) takes the u-th free
// slot (by block, then slot).  A workgroup per tree: the ids in order through a bit map, then a walk over
// the blocks.  (Few or none are left as a rule.  Two launches over all items took 17 + 5 us at 8 x 32768
// items and 56 + 10 us at 8 x 131072.)
constexpr int kLeftThreads = 1024;
constexpr int kLeftWords = 16 * 1024;  // of the bit map: 512K ids at a time

// exclusive prefix sum over the workgroup; `total` is that of all
__device__ __forceinline__ int leftover_scan(int mine, int* s_w, int* total) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int inc = mine;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int o = __shfl_up(inc, off, 64);
        if (lane >= off) inc += o;
    }
    __syncthreads();
    if (lane == 63) s_w[wave] = inc;
    __syncthreads();
    int before = 0, all = 0;
    for (int w = 0; w < kLeftThreads / 64; ++w) {
        if (w < wave) before += s_w[w];
        all += s_w[w];
    }
    *total = all;
    return before + inc - mine;
}

__global__ __launch_bounds__(kLeftThreads) void k_leftover(
    const int32_t* list, const int32_t* list_count, const int32_t* lost, const int32_t* lost_count, int n_c,
    int K, int bf, const int32_t* fill, int32_t* sorted /* (T, n_c) */, int32_t* slots) {
    __shared__ uint32_t s_map[kLeftWords];
    __shared__ int s_w[kLeftThreads / 64];
    const int t = blockIdx.x, tid = threadIdx.x;
    const int nl = list_count[t * kCounterStride], total = nl + lost_count[t * kCounterStride];
    if (total == 0) return;
    const int32_t* lt = list + (size_t)t * n_c;
    const int32_t* xt = lost + (size_t)t * n_c;
    int32_t* st = sorted + (size_t)t * n_c;
    int done = 0, sum;
    for (int lo = 0; lo < n_c && done < total; lo += kLeftWords * 32) {  // uniform
        const int words = min(kLeftWords, (n_c - lo + 31) / 32), per = (words + kLeftThreads - 1) / kLeftThreads;
        __syncthreads();
        for (int i = tid; i < words; i += kLeftThreads) s_map[i] = 0;
        __syncthreads();
        for (int e = tid; e < total; e += kLeftThreads) {
            const int d = (e < nl ? lt[e] : xt[e - nl]) - lo;
            if (d >= 0 && d < words * 32) atomicOr(&s_map[d >> 5], 1u << (d & 31));
        }
        __syncthreads();
        int mine = 0;
        for (int i = tid * per; i < min((tid + 1) * per, words); ++i) mine += __popc(s_map[i]);
        int at = done + leftover_scan(mine, s_w, &sum);
        for (int i = tid * per; i < min((tid + 1) * per, words); ++i)
            for (uint32_t bits = s_map[i]; bits; bits &= bits - 1) st[at++] = lo + i * 32 + __ffs(bits) - 1;
        done += sum;
    }
    __threadfence_block();
    __syncthreads();
    int before = 0;  // free slots ahead
    for (int k0 = 0; k0 < K && before < total; k0 += kLeftThreads) {  // uniform
        const int k = k0 + tid;
        const int f = k < K ? fill[(size_t)t * K + k] : bf;
        const int room = max(bf - f, 0);
        const int at = before + leftover_scan(room, s_w, &sum);
        for (int j = 0; j < room && at + j < total; ++j) slots[((size_t)t * K + k) * bf + f + j] = st[at + j];
        before += sum;
    }
}

// ------------------------------------------------------------------------------------
// 6. final layout
// ------------------------------------------------------------------------------------
// One level: every node of level l gets its children's rows (keys and values, or block centres of level
// l - 1) into their slots, its radius and its count:
//   radius = max over children (||child - centre|| + r_child), -inf when there is none.
// A wave per node.  Which cluster lies in a slot is followed from the root down (the clusters of the top level
// lie in order; slots[i][k] are the children of cluster k of level i): a chain of l' < L loads that no launch
// has to prepare.  `lpr` lanes (a power of two) hold a row in 16-byte chunks (a chunk is contiguous in either
// layout), 64 / lpr children a step, eight steps on their way.  The rows are read once for all of it: bound
// by the bytes moved, 8 x 131072 keys and values of 256 bytes with their radii and the largest magnitude
// per channel 214 us, 5.0 TB/s.  (As launches of their own -- orders, keys, values, centres, radii,
// magnitudes -- a level-4 index of those took 360 us, now 235; 8 x 32768 keys, three levels, 82, now 50.)
struct PlaceLevel {
    const void* rows;                // (T, rows_stride, D) what the children are: keys as they came, or block centres
    size_t rows_stride;
    const int32_t* slots[HIRA_MAX_LEVELS];  // (T, K[i], bf)
    int32_t K[HIRA_MAX_LEVELS];
    int32_t num_levels, level, size, bf, D, lpr;
    void* child;                     // (T, child_stride, D) where they go
    size_t child_stride;
    int32_t child_layout, center_layout;
    const float* child_radii;        // (T, child_stride), or NULL: keys have none
    const void* cent;                // (T, K[level], D) the level's block centres
    void* top;                       // top level: where those go themselves, (T, out_stride, D)
    float* radii;                    // (T, out_stride)
    int32_t* counts;
    size_t out_stride;
    int32_t* perm;                   // level 1: (T, child_stride)
    const void* values_in;           // level 1: (T, rows_stride, vdim) -> (T, child_stride, vdim), or NULL
    void* values;
    int32_t vdim, lpr_v;             // (a value row in steps of lpr_v <= 64 lanes)
    // a subtree (level 1 of 2): nodes with children first, to slots from slot0 and nodes from node0 on; perm takes
    // pos[child], (T, rows_stride)
    const int32_t* pos;
    int32_t slot0, node0;
    float* absmax;                   // ABSMAX: (T, kAbsCopies, D) joined by the largest finite magnitudes per channel
};

// 16 bytes that nothing reads for a while: they push nothing out of the caches on their way
__device__ __forceinline__ void store_once(void* p, const uint4& v) {
    typedef __attribute__((ext_vector_type(4))) uint32_t vec4;
    __builtin_nontemporal_store(vec4{v.x, v.y, v.z, v.w}, reinterpret_cast<vec4*>(p));
}

template <typename T, bool ABSMAX>
__global__ __launch_bounds__(kNodeThreads) void k_place(const PlaceLevel pl) {
    constexpr int EPL = Elem<T>::kPerChunk;
    constexpr int U = 8;
    __shared__ float s_abs[ABSMAX ? kNodeThreads / 64 : 1][256];
    const int p = node_of_wave(), t = blockIdx.x, lane = threadIdx.x & 63;
    const int bf = pl.bf, D = pl.D, lpr = pl.lpr;
    const int rg = lane / lpr, ch = lane % lpr, groups = 64 / lpr;
    const bool chunk_ok = ch * EPL < D;
    float big[EPL];
#pragma unroll
    for (int e = 0; e < EPL; ++e) big[e] = 0.0f;
    if (p < pl.size) {  // (uniform in the wave)
        int id = p;  // the cluster that lies in slot p
        for (int i = pl.level; i < pl.num_levels - 1; ++i) id /= bf;
        for (int i = pl.num_levels - 1; i > pl.level; --i) {  // (from cluster `id` of level i to one of level i - 1)
            int at = p;
            for (int j = pl.level; j < i - 1; ++j) at /= bf;
            id = id >= 0 ? pl.slots[i][((size_t)t * pl.K[i] + id) * bf + at % bf] : -1;
        }
        if (pl.pos) {  // block p, if those with children come first (size = bf <= 64 blocks, filled from the first slot on)
            const unsigned long long full = __ballot(lane < bf && pl.slots[1][((size_t)t * bf + min(lane, bf - 1)) * bf] >= 0);
            const int n_full = __popcll(full);
            unsigned long long left = p < n_full ? full : ~full;
            for (int i = p < n_full ? p : p - n_full; i > 0; --i) left &= left - 1ull;
            id = __ffsll((long long)left) - 1;
        }
        const int own = max(id, 0);
        const int mine = lane < bf && id >= 0 ? pl.slots[pl.level][((size_t)t * pl.K[pl.level] + own) * bf + lane] : -1;
        const unsigned long long live = __ballot(mine >= 0);
        const size_t s0 = (size_t)t * pl.child_stride + pl.slot0 + (size_t)p * bf;  // slots of the children
        const float my_radius = mine >= 0 && pl.child_radii ? pl.child_radii[s0 + lane] : 0.0f;
        if (pl.perm && lane < bf)
            pl.perm[s0 + lane] = mine >= 0 && pl.pos ? pl.pos[(size_t)t * pl.rows_stride + mine] : mine;
        const uint4 craw = load_chunk<T>(pl.cent, ((size_t)t * pl.K[pl.level] + own) * D, chunk_ok ? ch : 0);
        float cf[EPL];
        unpack<T>(craw, cf);
        if (pl.top && rg == 0 && chunk_ok)
            *reinterpret_cast<uint4*>(reinterpret_cast<T*>(pl.top) + (size_t)t * pl.out_stride * D +
                                      elem_index(pl.center_layout, D, (size_t)pl.node0 + p, ch * EPL)) = craw;
        T* const child = reinterpret_cast<T*>(pl.child) + (size_t)t * pl.child_stride * D;
        float r = -INFINITY;
        for (int j0 = 0; j0 < bf; j0 += U * groups) {  // (uniform trip count: the sums meet in shuffles)
            uint4 raw[U];
            int it[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {  // (a child that is none: row 0)
                const int j = j0 + u * groups + rg;
                it[u] = __shfl(mine, j & 63, 64);
                raw[u] = load_chunk<T>(pl.rows, ((size_t)t * pl.rows_stride + max(it[u], 0)) * D, chunk_ok ? ch : 0);
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int j = j0 + u * groups + rg;
                const bool have = j < bf && it[u] >= 0;
                if (j < bf && chunk_ok)
                    *reinterpret_cast<uint4*>(child + elem_index(pl.child_layout, D, (size_t)pl.slot0 + (size_t)p * bf + j, ch * EPL)) =
                        make_uint4(have ? raw[u].x : 0u, have ? raw[u].y : 0u, have ? raw[u].z : 0u, have ? raw[u].w : 0u);
                float f[EPL];
                unpack<T>(raw[u], f);
                float ss = 0.0f;
#pragma unroll
                for (int q = 0; q < EPL; ++q) {
                    const float df = f[q] - cf[q];
                    ss += df * df;
                }
                if (!chunk_ok) ss = 0.0f;
                ss = group_sum_of(ss, lpr);
                const float radius = __shfl(my_radius, j & 63, 64);
                if (have) {
                    float v = sqrtf(ss);
                    if (pl.child_radii) v += radius;
                    r = fmaxf(r, v);
                }
                if constexpr (ABSMAX) {
#pragma unroll
                    for (int q = 0; q < EPL; ++q) {
                        const float a = fabsf(f[q]);
                        big[q] = have && a < INFINITY && a > big[q] ? a : big[q];
                    }
                }
            }
        }
        if (pl.values) {
            const int lpr_v = pl.lpr_v, rg_v = lane / lpr_v, ch_v = lane % lpr_v, groups_v = 64 / lpr_v;
            T* const values = reinterpret_cast<T*>(pl.values);
            for (int c0 = 0; c0 * EPL < pl.vdim; c0 += lpr_v) {
                const int c = c0 + ch_v;
                const bool ok_v = c * EPL < pl.vdim;
                for (int j0 = 0; j0 < bf; j0 += U * groups_v) {
                    uint4 raw[U];
                    int it[U];
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        it[u] = __shfl(mine, (j0 + u * groups_v + rg_v) & 63, 64);
                        raw[u] = load_chunk<T>(pl.values_in, ((size_t)t * pl.rows_stride + max(it[u], 0)) * pl.vdim, ok_v ? c : 0);
                    }
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        const int j = j0 + u * groups_v + rg_v;
                        const bool have = it[u] >= 0;
                        if (j < bf && ok_v)
                            store_once(values + (s0 + j) * pl.vdim + c * EPL, have ? raw[u] : make_uint4(0, 0, 0, 0));
                    }
                }
            }
        }
        r = cross_group(r, lpr, OpMax{});
        if (lane == 0) {
            // a few ulp of head room: the bound must survive fp32 rounding of this sum
            if (r > 0.0f) r = r * (1.0f + 4.0f * 1.1920929e-7f) + 1e-30f;
            pl.radii[(size_t)t * pl.out_stride + pl.node0 + p] = r;
            pl.counts[(size_t)t * pl.out_stride + pl.node0 + p] = __popcll(live);
        }
    }
    if constexpr (ABSMAX) {
        // integer maxima: the bits of non-negative floats order like unsigned integers, and a maximum does not
        // depend on the order of arrival.  (Into kAbsCopies places in turn: workgroups of a tree that all join
        // the same 128 numbers wait for each other, 236 us for this launch instead of 214.)
        const int wave = threadIdx.x >> 6;
#pragma unroll
        for (int q = 0; q < EPL; ++q) {
            float m = big[q];
            m = cross_group(m, lpr, OpMax{});
            if (rg == 0 && chunk_ok) s_abs[wave][ch * EPL + q] = m;
        }
        __syncthreads();
        for (int j = threadIdx.x; j < D; j += kNodeThreads) {
            float m = s_abs[0][j];
#pragma unroll
            for (int w = 1; w < kNodeThreads / 64; ++w) m = fmaxf(m, s_abs[w][j]);
            atomicMax(reinterpret_cast<unsigned*>(pl.absmax) + ((size_t)t * kAbsCopies + tree_block() % kAbsCopies) * D + j, __float_as_uint(m));
        }
    }
}

// An index of one level: keys and values as they came, perm the numbers in order; a thread per 16-byte chunk
// of a row (a chunk is contiguous in either layout).
template <typename T>
__global__ void k_copy_rows(const void* src, int size, int D, void* dst, size_t dst_tree_stride, int dst_layout, int32_t* perm) {
    constexpr int EPL = Elem<T>::kPerChunk;
    const int t = blockIdx.x, chunks = D / EPL;
    const size_t i = (size_t)tree_block() * blockDim.x + threadIdx.x;
    if (i >= (size_t)size * chunks) return;
    const int s = (int)(i / chunks), c = (int)(i % chunks);
    *reinterpret_cast<uint4*>(reinterpret_cast<T*>(dst) + (size_t)t * dst_tree_stride * D + elem_index(dst_layout, D, (size_t)s, c * EPL)) =
        load_chunk<T>(src, ((size_t)t * size + s) * D, c);
    if (perm && c == 0) perm[(size_t)t * dst_tree_stride + s] = s;
}

// dst[t][s] = src[t][perm[t][s]] (zero row for -1), a thread per element: value rows whose length is not a
// multiple of 16 bytes
template <typename T>
__global__ void k_gather_elems(const void* src, size_t src_tree_stride, const int32_t* perm,
                               int size, int D, void* dst, size_t dst_tree_stride) {
    const int t = blockIdx.x;
    const size_t i = (size_t)tree_block() * blockDim.x + threadIdx.x;
    if (i >= (size_t)size * D) return;
    const int s = (int)(i / D), j = (int)(i % D);
    const int o = perm[(size_t)t * dst_tree_stride + s];
    float v = 0.0f;
    if (o >= 0) v = load_elem<T>(src, ((size_t)t * src_tree_stride + o) * D + j);
    store_elem<T>(dst, ((size_t)t * dst_tree_stride + s) * D + j, v);
}

// ------------------------------------------------------------------------------------
// host orchestration
// ------------------------------------------------------------------------------------
struct Carver {
    char* base;
    size_t used;
    template <typename U>
    U* take(size_t n) {
        used = (used + 255) & ~(size_t)255;
        U* p = base ? reinterpret_cast<U*>(base + used) : nullptr;
        used += n * sizeof(U);
        return p;
    }
};

struct BuildWs {
    float* cent_f32;
    CentroidTiles ct;    // centroids as operand tiles (matrix cores), or NULL
    CentroidTiles open;  // the same for the centroids with room, side by side (later packing rounds)
    int32_t *open_ids, *open_count;
    int32_t *members, *big, *unsure, *lost;
    float *dists, *more_dist;
    int2* more;
    int32_t* list[2];     // the items of a packing round, and those of the round after it
    int32_t* counters;    // (kBuildCounters, T), kCounterStride apart
    int32_t *counts, *fill;
    int32_t* slots[HIRA_MAX_LEVELS];
    void* cent_t[HIRA_MAX_LEVELS];
    float* absmax;  // (T, kAbsCopies, D), zero: an index with an 8-bit shadow; else NULL
    size_t total;
};

static int ceil_div(int a, int b) { return (a + b - 1) / b; }

// whether the matrix cores take the assignment of a level of K centroids (the exact kernel or the
// approximate one)
static bool assign_on_mfma(const HiraTree* t, int K) {
    return assign_exact_on_mfma(t->dtype, t->dim) || assign_approx_pays(t->dtype, t->dim, K);
}

// cluster counts per level: K[0] = n, K[l] = ceil(K[l-1] / bf)
static void cluster_counts(int n, int bf, int L, int* K) {
    K[0] = n;
    for (int l = 1; l < L; ++l) K[l] = K[l - 1] <= 0 ? 0 : (ceil_div(K[l - 1], bf) > 0 ? ceil_div(K[l - 1], bf) : 1);
}

// Whether a workgroup a tree takes this level, and with it all above (small_levels.hip).  It spends on a
// round what its items take one compute unit, the launches what launches take.  Trees x items x centroids (128
// columns), launches / one workgroup a tree, of a build of that level alone: 8 x 1024 x 32 164 / 126 us,
// 64 x 1024 x 32 203 / 141, 8 x 512 x 16 139 / 69, 8 x 1024 x 16 183 / 105.  With more centroids a wave
// takes them in turns (8 x 512 x 64: 134 / 147); rows of 256 columns, whose
// operands are twice as many: up to 512 x 16.
static bool level_is_small(const HiraTree* t, int n_c, int K) {
    return assign_exact_on_mfma(t->dtype, t->dim) && n_c <= kSmallItems && K <= kSmallCentroids &&
           n_c * K <= small_pairs(t->dim);
}

static void carve(const HiraTree* t, int n, void* ws, BuildWs* b) {
    const int L = t->num_levels, T = t->num_trees, D = t->dim, bf = t->bf;
    const size_t esize = t->dtype == HIRA_F32 ? 4 : 2;
    int K[HIRA_MAX_LEVELS];
    cluster_counts(n, bf, L, K);
    Carver c{reinterpret_cast<char*>(ws), 0};
    const size_t k1 = L >= 2 ? (size_t)K[1] : 1;
    b->cent_f32 = c.take<float>((size_t)T * k1 * D);
    b->ct = b->open = CentroidTiles{nullptr, nullptr, nullptr};
    b->open_ids = b->open_count = nullptr;
    if (assign_on_mfma(t, (int)k1)) {
        const size_t kpad = (size_t)assign_tiles((int)k1) * 16;
        const size_t chunks = kpad * assign_ks(t->dtype, D) * 8;  // hi and lo halves
        for (CentroidTiles* ct : {&b->ct, &b->open}) {
            ct->tiles = c.take<uint4>((size_t)T * chunks);
            ct->n2 = c.take<float>((size_t)T * kpad);
            ct->lo = c.take<float>((size_t)T * kpad);
        }
        b->open_ids = c.take<int32_t>((size_t)T * k1);
        b->open_count = c.take<int32_t>((size_t)T);
    }
    b->members = c.take<int32_t>((size_t)T * k1 << bucket_places_log2(bf));
    b->dists = c.take<float>((size_t)T * k1 << bucket_places_log2(bf));
    b->big = c.take<int32_t>((size_t)T * k1);
    b->more = c.take<int2>((size_t)T * n);
    b->more_dist = c.take<float>((size_t)T * n);
    b->lost = c.take<int32_t>((size_t)T * n);
    b->unsure = c.take<int32_t>((size_t)T * n);
    b->list[0] = c.take<int32_t>((size_t)T * n);
    b->list[1] = c.take<int32_t>((size_t)T * n);
    b->counters = c.take<int32_t>((size_t)T * kBuildCounters * kCounterStride);
    b->counts = c.take<int32_t>((size_t)T * k1 << bucket_count_log2(bf));
    b->fill = c.take<int32_t>((size_t)T * k1);
    for (int l = 0; l < HIRA_MAX_LEVELS; ++l) {
        b->slots[l] = nullptr;
        b->cent_t[l] = nullptr;
    }
    for (int l = 1; l < L; ++l) {
        b->slots[l] = c.take<int32_t>((size_t)T * K[l] * bf);
        b->cent_t[l] = c.take<char>((size_t)T * K[l] * D * esize);
    }
    b->absmax = t->layout == HIRA_TILE16_Q8 ? c.take<float>((size_t)T * kAbsCopies * D) : nullptr;
    b->total = (c.used + 255) & ~(size_t)255;
}

template <typename T>
static int launch_assign_simple(const AssignJob& job, const int32_t* fill, int bf, hipStream_t s) {
    int lpr = 2;
    while (lpr * Elem<T>::kPerChunk < job.D) lpr <<= 1;
    // (as many workgroups as a list of all items has sets, if all waves share them)
    const dim3 grid(job.num_trees, min(ceil_div(job.n_c, 64 / lpr * kPPG), max(kSimpleBlocks / job.num_trees, 16)));
#define HIRA_ASSIGN_CASE(N)                                                                            \
    case N:                                                                                            \
        hipLaunchKernelGGL((k_assign_simple<T, N>), grid, dim3(kSimpleThreads), 0, s, fill, bf, job);  \
        break;
    switch (lpr) {
        HIRA_ASSIGN_CASE(2)
        HIRA_ASSIGN_CASE(4)
        HIRA_ASSIGN_CASE(8)
        HIRA_ASSIGN_CASE(16)
        HIRA_ASSIGN_CASE(32)
        HIRA_ASSIGN_CASE(64)
        default:
            return fail(HIRA_EINVAL, "unsupported row width");
    }
#undef HIRA_ASSIGN_CASE
    return HIRA_OK;
}

static void fill_i32(int32_t* p, size_t n, int32_t v, hipStream_t s) {
    if (n == 0) return;
    hipLaunchKernelGGL(k_fill_i32, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, p, n, v);
}

static int lanes_per_row(int dtype, int D) {  // a power of two, 16 bytes a lane
    int lpr = 2;
    while (lpr * (dtype == HIRA_F32 ? 4 : 8) < D) lpr <<= 1;
    return lpr;
}

// Levels 1 .. L - 1: slots and block centres of every cluster, to the workspace.
// small_ragged: two levels of trees with key counts may go through small_levels.hip too (a subtree: 105 us for 8 x
// 1024 x 32, the launches 164; a build with counts stays with the launches, whatever its sizes).
template <typename T>
static int cluster_levels(const HiraTree* t, const void* keys_in, int n, const int32_t* n_live, int niter,
                          int pack_rounds, uint64_t seed, const BuildWs& w, bool small_ragged, hipStream_t s) {
    const int L = t->num_levels, NT = t->num_trees, D = t->dim, bf = t->bf, lpr = lanes_per_row(t->dtype, D);
    int K[HIRA_MAX_LEVELS];
    cluster_counts(n, bf, L, K);

    const size_t ct = (size_t)NT * kCounterStride;
    int32_t* const list_count = w.counters;           // (2, T)
    int32_t* const more_count = w.counters + 2 * ct;  // (2, T)
    int32_t* const unsure_count = w.counters + 4 * ct;
    int32_t* const lost_count = w.counters + 5 * ct;
    int32_t* const big_count = w.counters + 6 * ct;   // (2, T)
    const int KS = assign_ks(t->dtype, D);
    for (int l = 1; l < L; ++l) {
        if (level_is_small(t, K[l - 1], K[l]) && (n_live == nullptr || (small_ragged && L == 2))) {  // this one and all above it in one launch
            if (l == 1 && w.absmax != nullptr) fill_i32(reinterpret_cast<int32_t*>(w.absmax), (size_t)NT * kAbsCopies * D, 0, s);
            SmallLevels p{};
            p.x = l == 1 ? keys_in : w.cent_t[l - 1];
            p.n_live = n_live;
            p.first = l;
            p.last = L;
            for (int i = l - 1; i < L; ++i) {
                p.K[i] = K[i];
                p.slots[i] = w.slots[i];
                p.cent_t[i] = w.cent_t[i];
            }
            p.cent = w.cent_f32;
            p.seed = seed;
            p.niter = niter;
            p.pack_rounds = pack_rounds;
            p.bf = bf;
            if (const int rc = launch_small_levels(p, D, NT, s)) return rc;
            HIRA_CHECK_LAUNCH("build, small levels");
            break;
        }
        const void* x = l == 1 ? keys_in : w.cent_t[l - 1];
        const int n_c = K[l - 1];
        const size_t xs = (size_t)n_c;  // rows per tree in x
        const int Kl = K[l];
        const bool on_mfma = assign_on_mfma(t, Kl), approx = assign_approx_pays(t->dtype, D, Kl);
        const int Kt = on_mfma ? assign_tiles(Kl) : 0;
        const CentroidTiles tiles = on_mfma ? w.ct : CentroidTiles{nullptr, nullptr, nullptr};
        const long long all_items = (long long)n_c * NT;
        int round = 0;  // of the level, Lloyd and packing together
        const int large = large_blocks(Kl);
        const dim3 g_bucket = tree_grid(large + ceil_div(Kl, kWaves), NT);

        // Trees with fewer items than rows (n_live): the rounds over all items are over the first
        // ones of every tree.
        const bool ragged = n_live != nullptr && l == 1;
        int lanes = 1;
        while (lanes * 8 < D || (on_mfma && lanes < KS * 4)) lanes <<= 1;
        hipLaunchKernelGGL((k_level_init<T>), node_grid(ceil_div(Kl, 64 / lanes), NT), dim3(kNodeThreads), 0, s, x, n_c, xs, Kl, bf, D,
                           seed + 7919ull * (uint64_t)l, w.cent_f32, ragged ? n_live : nullptr, w.fill, w.slots[l], w.counts, w.counters,
                           l == 1 ? w.absmax : nullptr, Kt, tiles, KS, lanes, bucket_count_log2(bf));
        // a round: the assignment (which also puts the items into buckets), then what the round does
        // with every bucket.  A Lloyd round asks for no distances.
        auto buckets = [&]() {
            const int now = round & 1, next = now ^ 1;
            return Buckets{w.counts, w.members, w.dists, w.big, big_count + now * ct, w.more, more_count + now * ct,
                           w.more_dist, big_count + next * ct, more_count + next * ct, unsure_count, bucket_places_log2(bf), bucket_count_log2(bf)};
        };
        auto assign_round = [&](const int32_t* list, const int32_t* lcnt, const int32_t* fill, bool packing,
                                int32_t* zero, bool only_open, long long expected) -> int {
            AssignJob job{};
            job.x = x;
            job.n_c = n_c;
            job.n_live = ragged ? n_live : nullptr;
            job.x_tree_stride = xs;
            job.dtype = t->dtype;
            job.D = D;
            job.num_trees = NT;
            job.ct = tiles;
            job.cent = w.cent_f32;
            job.K = Kl;
            job.list = list;
            job.list_count = lcnt;
            job.counting = AssignCounting{w.counts, w.members, packing ? w.dists : nullptr, w.big,
                                          big_count + (round & 1) * ct, w.more, more_count + (round & 1) * ct, w.more_dist, w.lost, lost_count, zero,
                                          bucket_places_log2(bf), bucket_count_log2(bf)};
            job.unsure = w.unsure;
            job.unsure_count = unsure_count;
            int rc = HIRA_OK;
            if (on_mfma && only_open) {
                rc = launch_open_centroids(KS, w.ct, w.fill, bf, Kl, NT, w.open_ids, w.open_count, w.open, s);
                job.ct = w.open;
                job.open = AssignOpen{w.open_count, w.open_ids};
            }
            const bool exact_mfma = assign_exact_on_mfma(t->dtype, D);
            // (the lists of the packing about halve from round to round: the later ones are none of
            // the approximate pass's, and spared its launch)
            if (rc == HIRA_OK && approx && (!exact_mfma || expected > kApproxListItems)) {
                rc = launch_assign_approx(job, s);
                job.after_approx = 1;
            }
            if (rc != HIRA_OK) return rc;
            if (exact_mfma) return launch_assign_mfma(job, s);
            if (job.after_approx) {
                job.list = w.unsure;
                job.list_count = unsure_count;
            }
            return launch_assign_simple<T>(job, fill, bf, s);
        };
        for (int it = 0; it < niter; ++it, ++round) {
            const int rc = assign_round(nullptr, nullptr, ragged ? w.fill : nullptr, false, nullptr, false, all_items);
            if (rc != HIRA_OK) return rc;
            hipLaunchKernelGGL((k_bucket_mean<T>), g_bucket, dim3(kBucketThreads), 0, s, x, xs, n_c, Kl, D, buckets(),
                               ragged ? w.fill : nullptr, bf, w.cent_f32, Kt, tiles, KS, large);
        }
        // capacity packing: the first round is over all items, round r over list r % 2; it leaves those
        // it could not place on the other list
        for (int r = 0; r < pack_rounds; ++r, ++round) {
            const int32_t* list = r == 0 ? nullptr : w.list[r & 1];
            const int32_t* lcnt = r == 0 ? nullptr : list_count + (r & 1) * ct;
            int32_t* next_cnt = list_count + ((r + 1) & 1) * ct;
            // (from the second round on most blocks are full: the assignment then sees only the
            // centroids with room, side by side; worth its launch from 32 tiles on, and where rows are of 64 columns, whose products
            // with the full ones take half as long and leave the registers to twice the waves, only where the list may be long:
            // builds of 64 columns with the launch in all rounds / by this rule: 2 x 9600 keys at a fan-out of 16 247 / 229 us,
            // 2 x 16001 274 / 258, 1 x 24000 304 / 296, 8 x 16001 365 / 358, 8 x 30000 at 32 412 / 404; without it in all rounds
            // 8 x 30000 412, 8 x 60000 762 -> 816, 2 x 60011 at 16 575 -> 585 without it in the last four; of 128 columns
            // 8 x 32768 without it from the fifth round on 572 -> 575)
            const bool side_by_side = r >= 1 && Kl >= 512 && (KS > 2 || Kl > 2048 || (all_items >> r) * Kl > 25ll * 1000 * 1000);
            const int rc = assign_round(list, lcnt, w.fill, true, next_cnt, side_by_side, all_items >> r);
            if (rc != HIRA_OK) return rc;
            hipLaunchKernelGGL(k_bucket_accept, g_bucket, dim3(kBucketThreads), 0, s, buckets(), n_c, Kl, bf,
                               w.fill, w.slots[l], w.list[(r + 1) & 1], next_cnt, Kt, tiles.n2, large);
        }
        hipLaunchKernelGGL(k_leftover, dim3(NT), dim3(kLeftThreads), 0, s, w.list[pack_rounds & 1],
                           list_count + (pack_rounds & 1) * ct, w.lost, lost_count, n_c, Kl, bf, w.fill,
                           w.unsure, w.slots[l]);
        // block centre = mean of what is in the block, rounded to the storage type
        hipLaunchKernelGGL((k_block_mean<T>), node_grid(Kl, NT), dim3(kNodeThreads), 0, s, x, xs, Kl, D, w.slots[l], bf,
                           lpr, w.cent_f32, w.cent_t[l]);
        HIRA_CHECK_LAUNCH("build level");
    }

    return HIRA_OK;
}

template <typename T>
static int build_impl(const HiraTree* t, const void* keys_in, const void* values_in, int n,
                      const int32_t* n_live, int niter, int pack_rounds, uint64_t seed,
                      const BuildWs& w, hipStream_t s) {
    const int L = t->num_levels, NT = t->num_trees, D = t->dim, bf = t->bf, lpr = lanes_per_row(t->dtype, D);
    constexpr int EPL = Elem<T>::kPerChunk;
    int K[HIRA_MAX_LEVELS];
    cluster_counts(n, bf, L, K);
    if (const int rc = cluster_levels<T>(t, keys_in, n, n_live, niter, pack_rounds, seed, w, false, s)) return rc;

    // layout and radii, bottom-up
    const bool whole_v = t->vdim % EPL == 0, have_v = values_in && t->values;
    if (L == 1) {
        const size_t tot = (size_t)n * (D / EPL);
        hipLaunchKernelGGL((k_copy_rows<T>), tree_grid((long long)((tot + 255) / 256), NT), dim3(256), 0, s, keys_in, n, D,
                           t->keys, (size_t)t->cap[0], key_layout_of(t->layout), t->perm);
        if (have_v && whole_v) {
            const size_t totv = (size_t)n * (t->vdim / EPL);
            hipLaunchKernelGGL((k_copy_rows<T>), tree_grid((long long)((totv + 255) / 256), NT), dim3(256), 0, s, values_in,
                               n, t->vdim, t->values, (size_t)t->cap[0], (int)HIRA_ROW_MAJOR, nullptr);
        }
    }
    for (int l = 1; l < L; ++l) {
        PlaceLevel p{};
        p.rows = l == 1 ? keys_in : w.cent_t[l - 1];
        p.rows_stride = (size_t)K[l - 1];
        for (int i = l; i < L; ++i) {
            p.slots[i] = w.slots[i];
            p.K[i] = K[i];
        }
        p.num_levels = L;
        p.level = l;
        p.size = t->size[l];
        p.bf = bf;
        p.D = D;
        p.lpr = lpr;
        p.child = l == 1 ? t->keys : t->centers[l - 1];
        p.child_stride = (size_t)t->cap[l - 1];
        p.child_layout = l == 1 ? key_layout_of(t->layout) : center_layout_of(t->layout);
        p.center_layout = center_layout_of(t->layout);
        p.child_radii = l == 1 ? nullptr : t->radii[l - 1];
        p.cent = w.cent_t[l];
        p.top = l == L - 1 ? t->centers[l] : nullptr;
        p.radii = t->radii[l];
        p.counts = t->counts[l];
        p.out_stride = (size_t)t->cap[l];
        if (l == 1) {
            p.perm = t->perm;
            if (have_v && whole_v) {
                p.values_in = values_in;
                p.values = t->values;
                p.vdim = t->vdim;
                p.lpr_v = 2;
                while (p.lpr_v < 64 && p.lpr_v * EPL < t->vdim) p.lpr_v <<= 1;
            }
            p.absmax = w.absmax;
        }
        if (l == 1 && w.absmax != nullptr)
            hipLaunchKernelGGL((k_place<T, true>), node_grid(t->size[l], NT), dim3(kNodeThreads), 0, s, p);
        else
            hipLaunchKernelGGL((k_place<T, false>), node_grid(t->size[l], NT), dim3(kNodeThreads), 0, s, p);
    }
    if (have_v && !whole_v) {
        const size_t totv = (size_t)t->size[0] * t->vdim;
        hipLaunchKernelGGL((k_gather_elems<T>), tree_grid((long long)((totv + 255) / 256), NT), dim3(256), 0, s, values_in,
                           (size_t)n, t->perm, t->size[0], t->vdim, t->values, (size_t)t->cap[0]);
    }
    HIRA_CHECK_LAUNCH("build layout");
    if (w.absmax != nullptr) return quantize_with(t, w.absmax, kAbsCopies, s);  // the 8-bit shadow, its steps from all keys
    return HIRA_OK;
}

static int check_build_args(const HiraTree* t, int n) {
    HIRA_CHECK_ARG(t != nullptr, "tree is NULL");
    HIRA_CHECK_ARG(t->dtype == HIRA_F32 || t->dtype == HIRA_BF16, "dtype %d", t->dtype);
    HIRA_CHECK_ARG(t->num_trees >= 1 && t->num_trees <= 65535, "num_trees %d", t->num_trees);
    HIRA_CHECK_ARG(t->num_levels >= 1 && t->num_levels <= HIRA_MAX_LEVELS, "num_levels %d",
                   t->num_levels);
    HIRA_CHECK_ARG(t->bf >= 1 && t->bf <= 64, "branching factor %d not in 1..64", t->bf);
    const int epl = t->dtype == HIRA_F32 ? 4 : 8;
    HIRA_CHECK_ARG(t->dim >= epl && t->dim % epl == 0 && t->dim <= 64 * epl,
                   "dim %d: rows must be a multiple of 16 bytes", t->dim);
    HIRA_CHECK_ARG(n >= 1, "need at least one key, got %d", n);
    HIRA_CHECK_ARG(t->layout == HIRA_ROW_MAJOR || t->layout == HIRA_TILE16 ||
                       t->layout == HIRA_TILE16_Q8, "layout %d", t->layout);
    if (t->layout == HIRA_TILE16_Q8)
        HIRA_CHECK_ARG((t->dim == 64 || t->dim == 128) && t->num_levels >= 2 && t->keys8 &&
                           t->kscale && t->keps,
                       "the layout with an 8-bit shadow needs rows of 64 or 128 columns, at least "
                       "two levels, and the keys8 / kscale / keps arrays");
    if (t->layout != HIRA_ROW_MAJOR) {
        HIRA_CHECK_ARG(t->dtype == HIRA_BF16 && t->dim % 32 == 0,
                       "the tiled layout needs bf16 rows of a multiple of 32 columns");
        for (int l = 0; l < t->num_levels; ++l)
            HIRA_CHECK_ARG(t->cap[l] % 16 == 0, "tiled layout: cap[%d]=%d not a multiple of 16", l,
                           t->cap[l]);
    }
    int K[HIRA_MAX_LEVELS];
    cluster_counts(n, t->bf, t->num_levels, K);
    // padded sizes the layout needs
    long long want = t->num_levels == 1 ? n : K[t->num_levels - 1];
    for (int l = t->num_levels - 1; l >= 0; --l) {
        HIRA_CHECK_ARG(t->size[l] == want, "size[%d] = %d, the layout of %d keys needs %lld", l,
                       t->size[l], n, want);
        HIRA_CHECK_ARG(t->cap[l] >= t->size[l], "cap[%d] = %d < size %d", l, t->cap[l], t->size[l]);
        want *= t->bf;
    }
    return HIRA_OK;
}

}  // namespace hira

using namespace hira;

extern "C" size_t hira_build_workspace_bytes(const HiraTree* tree, int32_t n) {
    if (check_build_args(tree, n) != HIRA_OK) return 0;
    BuildWs b;
    carve(tree, n, nullptr, &b);
    return b.total;
}

extern "C" int hira_build(const HiraTree* tree, const void* keys_in, const void* values_in,
                          int32_t n, int32_t niter, int32_t pack_rounds, uint64_t seed,
                          void* workspace, size_t workspace_bytes, void* stream) {
    return hira_build_ragged(tree, keys_in, values_in, n, nullptr, niter, pack_rounds, seed,
                             workspace, workspace_bytes, stream);
}

/* see include/hira_hip.h */
extern "C" int hira_build_ragged(const HiraTree* tree, const void* keys_in, const void* values_in,
                                 int32_t n, const int32_t* n_live, int32_t niter,
                                 int32_t pack_rounds, uint64_t seed, void* workspace,
                                 size_t workspace_bytes, void* stream) {
    int rc = check_build_args(tree, n);
    if (rc != HIRA_OK) return rc;
    HIRA_CHECK_ARG(n_live == nullptr || tree->num_levels == 2,
                   "per-tree key counts are taken for trees of two levels only (got %d)",
                   tree->num_levels);
    HIRA_CHECK_ARG(keys_in != nullptr && tree->keys != nullptr && tree->perm != nullptr,
                   "keys / perm missing");
    HIRA_CHECK_ARG(niter >= 0 && pack_rounds >= 1, "niter %d, pack_rounds %d", niter, pack_rounds);
    for (int l = 1; l < tree->num_levels; ++l)
        HIRA_CHECK_ARG(tree->centers[l] && tree->radii[l] && tree->counts[l],
                       "level %d arrays missing", l);
    BuildWs b;
    carve(tree, n, workspace, &b);
    if (workspace == nullptr || workspace_bytes < b.total)
        return fail(HIRA_EWORKSPACE, "workspace %zu bytes, need %zu", workspace_bytes, b.total);
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    return tree->dtype == HIRA_F32
               ? build_impl<float>(tree, keys_in, values_in, n, n_live, niter, pack_rounds, seed, b, s)
               : build_impl<bf16_t>(tree, keys_in, values_in, n, n_live, niter, pack_rounds, seed, b, s);
}

// ---- one level-2 subtree of every tree clustered anew -----------------------------------------
// Four launches: the subtree's rows to the front of a workspace, the two levels over them, the nodes with keys
// into their places, the radii above.  8 trees x 1024 rows of 128 columns, keys and values, bf16: 11 + 105 + 9 + 9 us
// on the GPU, 21 on the host.  (As gathers, sorts and copies of a tensor library around a build of its own some fifty
// launches: 557 us of the host, which the GPU waited for.)  The clustering bounds it, a chain of rounds.
namespace hira {

constexpr int kTakeSlots = 64;

// The subtree's rows of every tree, those in use first, in slot order: rows (T, nsub, D) row-major, values, the
// insertion positions (-1: no key), how many a tree holds.  A workgroup per 64 slots; each counts for
// itself how many are in use ahead of its own.
template <typename T>
__global__ __launch_bounds__(256) void k_subtree_take(const HiraTree tree, int slot0, int nsub, T* rows, T* vals, int32_t* pos,
                                                      int32_t* counts) {
    constexpr int EPL = Elem<T>::kPerChunk;
    __shared__ int s_before[4], s_total[4], s_dst[kTakeSlots];
    const int t = blockIdx.x, first = tree_block() * kTakeSlots, tid = threadIdx.x, lane = tid & 63;
    const size_t cap0 = (size_t)tree.cap[0];
    const int32_t* perm = tree.perm + (size_t)t * cap0 + slot0;
    int before = 0, total = 0;
    for (int i = tid; i < nsub; i += 256) {
        const int live = perm[i] >= 0 ? 1 : 0;
        total += live;
        before += i < first ? live : 0;
    }
    before = lanes_fold<1, 64>(before, OpSum{});
    total = lanes_fold<1, 64>(total, OpSum{});
    if (lane == 0) {
        s_before[tid >> 6] = before;
        s_total[tid >> 6] = total;
    }
    __syncthreads();
    if (tid < kTakeSlots) {
        before = s_before[0] + s_before[1] + s_before[2] + s_before[3];
        total = s_total[0] + s_total[1] + s_total[2] + s_total[3];
        const int slot = first + tid, at = slot < nsub ? perm[slot] : -1;
        const unsigned long long live = __ballot(at >= 0);
        const int ahead = before + __popcll(live & ((1ull << tid) - 1ull));
        const int dst = at >= 0 ? ahead : total + slot - ahead;
        s_dst[tid] = dst;
        if (slot < nsub) pos[(size_t)t * nsub + dst] = at;
        if (first == 0 && tid == 0) counts[t] = total;
    }
    __syncthreads();
    const int kc = tree.dim / EPL, vc = vals ? tree.vdim / EPL : 0, per = kc + vc, here = min(kTakeSlots, nsub - first);
    const int layout = key_layout_of(tree.layout);
    for (int e = tid; e < here * per; e += 256) {
        const int r = e / per, c = e % per;
        const size_t slot = (size_t)slot0 + first + r, dst = (size_t)t * nsub + s_dst[r];
        if (c < kc)
            *reinterpret_cast<uint4*>(rows + dst * tree.dim + c * EPL) =
                load_row_chunk<T>(tree.keys, layout, tree.dim, (size_t)t * cap0, slot, c);
        else
            *reinterpret_cast<uint4*>(vals + dst * tree.vdim + (c - kc) * EPL) =
                load_chunk<T>(tree.values, ((size_t)t * cap0 + slot) * tree.vdim, c - kc);
    }
}

// The level-2 node keeps its centre and gets the radius its new children need; its ancestors cover it where it grew
// (with a little head room: fp32 norms).  A number that is none stays one.  A workgroup per tree.
template <typename T>
__global__ __launch_bounds__(256) void k_subtree_up(const HiraTree tree, int node, int32_t* state) {
    __shared__ float s_r[4], s_d[HIRA_MAX_LEVELS];
    const int t = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int D = tree.dim, bf = tree.bf, L = tree.num_levels, n0 = node * bf, layout = center_layout_of(tree.layout);
    auto at = [&](int l, size_t p, int j) {
        return load_elem<T>(tree.centers[l], (size_t)t * tree.cap[l] * D + elem_index(layout, D, p, j));
    };
    auto distance = [&](int l, size_t p, size_t q) {  // of node p of level l - 1 and node q of level l (one wave)
        float ss = 0.0f;
        for (int j = lane; j < D; j += 64) {
            const float df = at(l - 1, p, j) - at(l, q, j);
            ss += df * df;
        }
        ss = wave_sum(ss);
        return sqrtf(ss);
    };
    auto larger = [](float a, float b) { return b > a || b != b ? b : a; };
    float r = -INFINITY;
    for (int p = wave; p < bf; p += 4)
        r = larger(r, distance(2, (size_t)n0 + p, (size_t)node) + tree.radii[1][(size_t)t * tree.cap[1] + n0 + p]);
    if (lane == 0) s_r[wave] = r;
    size_t child = (size_t)node;
    for (int l = 3; l < L; ++l, child /= (size_t)bf)
        if ((l & 3) == wave) {
            const float d = distance(l, child, child / (size_t)bf);
            if (lane == 0) s_d[l] = d;
        }
    __syncthreads();
    const unsigned long long full = __ballot(lane < bf && tree.counts[1][(size_t)t * tree.cap[1] + n0 + min(lane, bf - 1)] > 0);
    if (tid != 0) return;
    constexpr float kRoom = 1.0f + 1e-6f;
    r = larger(larger(larger(s_r[0], s_r[1]), s_r[2]), s_r[3]) * kRoom;
    tree.radii[2][(size_t)t * tree.cap[2] + node] = r;
    tree.counts[2][(size_t)t * tree.cap[2] + node] = __popcll(full);
    child = (size_t)node;
    for (int l = 3; l < L; ++l) {
        child /= (size_t)bf;
        float* out = tree.radii[l] + (size_t)t * tree.cap[l] + child;
        r = larger(*out, (s_d[l] + r) * kRoom);
        *out = r;
    }
    if (state) state[(size_t)t * (HIRA_MAX_LEVELS + 2)] = 0;  // (the rebuilt nodes may have room again)
}

struct RebuildWs {
    BuildWs build;
    HiraTree sub;
    void *rows, *vals;
    int32_t *pos, *counts;
    size_t total;
};

static int carve_rebuild(const HiraTree* t, void* ws, RebuildWs* b) {
    HIRA_CHECK_ARG(t != nullptr && t->num_trees >= 1 && t->num_levels >= 3 && t->num_levels <= HIRA_MAX_LEVELS,
                   "a subtree of level 2 needs at least three levels");
    HIRA_CHECK_ARG(t->bf >= 1 && t->bf <= 64, "branching factor %d not in 1..64", t->bf);
    HIRA_CHECK_ARG(t->layout == HIRA_ROW_MAJOR || t->bf % 16 == 0, "tiled layout: fan-out %d, a subtree must start on a tile", t->bf);
    const int nsub = t->bf * t->bf;
    HiraTree& sub = b->sub;
    memset(&sub, 0, sizeof(sub));
    sub.num_trees = t->num_trees;
    sub.num_levels = 2;
    sub.bf = t->bf;
    sub.dim = t->dim;
    sub.vdim = t->vdim;
    sub.dtype = t->dtype;
    sub.layout = HIRA_ROW_MAJOR;
    sub.size[0] = sub.cap[0] = nsub;
    sub.size[1] = sub.cap[1] = t->bf;
    if (const int rc = check_build_args(&sub, nsub)) return rc;
    const size_t esize = t->dtype == HIRA_F32 ? 4 : 2, T = (size_t)t->num_trees;
    Carver c{reinterpret_cast<char*>(ws), 0};
    b->rows = c.take<char>(T * nsub * t->dim * esize);
    b->vals = t->values ? c.take<char>(T * nsub * t->vdim * esize) : nullptr;
    b->pos = c.take<int32_t>(T * nsub);
    b->counts = c.take<int32_t>(T);
    const size_t own = (c.used + 255) & ~(size_t)255;
    carve(&sub, nsub, ws ? reinterpret_cast<char*>(ws) + own : nullptr, &b->build);
    b->total = own + b->build.total;
    return HIRA_OK;
}

template <typename T>
static int rebuild_impl(const HiraTree* t, int node, int niter, int pack_rounds, uint64_t seed, int32_t* state, const RebuildWs& w,
                        hipStream_t s) {
    const int bf = t->bf, nsub = bf * bf, NT = t->num_trees;
    hipLaunchKernelGGL((k_subtree_take<T>), tree_grid((nsub + kTakeSlots - 1) / kTakeSlots, NT), dim3(256), 0, s, *t, node * nsub,
                       nsub, reinterpret_cast<T*>(w.rows), reinterpret_cast<T*>(w.vals), w.pos, w.counts);
    if (const int rc = cluster_levels<T>(&w.sub, w.rows, nsub, w.counts, niter, pack_rounds, seed, w.build, true, s)) return rc;
    PlaceLevel p{};
    p.rows = w.rows;
    p.rows_stride = (size_t)nsub;
    p.slots[1] = w.build.slots[1];
    p.K[1] = bf;
    p.num_levels = 2;
    p.level = 1;
    p.size = bf;
    p.bf = bf;
    p.D = t->dim;
    p.lpr = lanes_per_row(t->dtype, t->dim);
    p.child = t->keys;
    p.child_stride = (size_t)t->cap[0];
    p.child_layout = key_layout_of(t->layout);
    p.center_layout = center_layout_of(t->layout);
    p.cent = w.build.cent_t[1];
    p.top = t->centers[1];
    p.radii = t->radii[1];
    p.counts = t->counts[1];
    p.out_stride = (size_t)t->cap[1];
    p.perm = t->perm;
    if (w.vals) {
        p.values_in = w.vals;
        p.values = t->values;
        p.vdim = t->vdim;
        p.lpr_v = min(lanes_per_row(t->dtype, t->vdim), 64);
    }
    p.pos = w.pos;
    p.slot0 = node * nsub;
    p.node0 = node * bf;
    hipLaunchKernelGGL((k_place<T, false>), node_grid(bf, NT), dim3(kNodeThreads), 0, s, p);
    hipLaunchKernelGGL((k_subtree_up<T>), dim3(NT), dim3(256), 0, s, *t, node, state);
    HIRA_CHECK_LAUNCH("subtree rebuild");
    return t->layout == HIRA_TILE16_Q8 ? hira_quantize(t, node * nsub, nsub, 0, s) : HIRA_OK;
}

}  // namespace hira

/* see include/hira_hip.h */
extern "C" size_t hira_rebuild_workspace_bytes(const HiraTree* tree) {
    RebuildWs w;
    return carve_rebuild(tree, nullptr, &w) == HIRA_OK ? w.total : 0;
}

/* see include/hira_hip.h */
extern "C" int hira_rebuild_subtree(const HiraTree* tree, int32_t node, int32_t niter, int32_t pack_rounds, uint64_t seed,
                                    int32_t* state, void* workspace, size_t workspace_bytes, void* stream) {
    RebuildWs w;
    if (const int rc = carve_rebuild(tree, workspace, &w)) return rc;
    if (workspace == nullptr || workspace_bytes < w.total)
        return fail(HIRA_EWORKSPACE, "workspace %zu bytes, need %zu", workspace_bytes, w.total);
    const long long bf = tree->bf;
    HIRA_CHECK_ARG(node >= 0 && node < tree->cap[2] && (node + 1) * bf <= tree->cap[1] && (node + 1) * bf * bf <= tree->cap[0],
                   "level-2 node %d: its slots lie beyond the capacity of the index", node);
    HIRA_CHECK_ARG(tree->keys && tree->perm, "keys / perm missing");
    HIRA_CHECK_ARG(niter >= 0 && pack_rounds >= 1, "niter %d, pack_rounds %d", niter, pack_rounds);
    for (int l = 1; l < tree->num_levels; ++l)
        HIRA_CHECK_ARG(tree->centers[l] && tree->radii[l] && tree->counts[l], "level %d arrays missing", l);
    HIRA_CHECK_ARG(!tree->values || tree->vdim % (tree->dtype == HIRA_F32 ? 4 : 8) == 0, "vdim %d: rows must be a multiple of 16 bytes",
                   tree->vdim);
    if (tree->layout == HIRA_TILE16_Q8)
        HIRA_CHECK_ARG(tree->keys8 && tree->kscale && tree->keps, "keys8 / kscale / keps missing");
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    return tree->dtype == HIRA_F32 ? rebuild_impl<float>(tree, node, niter, pack_rounds, seed, state, w, s)
                                   : rebuild_impl<bf16_t>(tree, node, niter, pack_rounds, seed, state, w, s);
}

// ---- nearest centre as a call of its own -------------------------------------------------
namespace hira {

__global__ void k_valid_to_fill(const int32_t* valid, size_t n, int32_t* fill) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) fill[i] = valid[i] != 0 ? 0 : 1;  // "full" (>= 1 of 1 slots) = not usable
}

struct NearestWs {
    void* tiles;
    float* n2;
    int32_t* fill;
    size_t total;
};

static void carve_nearest(int dtype, int T, int m, int D, bool masked, void* ws, NearestWs* b) {
    Carver c{reinterpret_cast<char*>(ws), 0};
    b->tiles = nullptr;
    b->n2 = nullptr;
    if (assign_exact_on_mfma(dtype, D)) {
        const size_t kpad = (size_t)assign_tiles(m) * 16;
        b->tiles = c.take<char>((size_t)T * kpad * D * 4);
        b->n2 = c.take<float>((size_t)T * kpad);
    }
    b->fill = masked ? c.take<int32_t>((size_t)T * m) : nullptr;
    b->total = (c.used + 255) & ~(size_t)255;
}

static int check_nearest_args(int dtype, int T, int n, int m, int D) {
    HIRA_CHECK_ARG(dtype == HIRA_F32 || dtype == HIRA_BF16, "dtype %d", dtype);
    const int epl = dtype == HIRA_F32 ? 4 : 8;
    HIRA_CHECK_ARG(T >= 1 && T <= 65535, "num_trees %d", T);
    HIRA_CHECK_ARG(n >= 1 && m >= 1, "n = %d rows, m = %d centres", n, m);
    HIRA_CHECK_ARG(D >= epl && D % epl == 0 && D <= 64 * epl,
                   "dim %d: rows must be a multiple of 16 bytes", D);
    return HIRA_OK;
}

}  // namespace hira

extern "C" size_t hira_nearest_workspace_bytes(int32_t dtype, int32_t num_trees, int32_t m,
                                               int32_t dim) {
    if (check_nearest_args(dtype, num_trees, 1, m, dim) != HIRA_OK) return 0;
    NearestWs b;
    carve_nearest(dtype, num_trees, m, dim, true, nullptr, &b);
    return b.total > 0 ? b.total : 256;
}

extern "C" int hira_nearest(const void* x, int32_t dtype, int32_t num_trees, int32_t n,
                            const float* centers, int32_t m, int32_t dim, const int32_t* valid,
                            int32_t* idx, float* dist2, void* workspace, size_t workspace_bytes,
                            void* stream) {
    int rc = check_nearest_args(dtype, num_trees, n, m, dim);
    if (rc != HIRA_OK) return rc;
    HIRA_CHECK_ARG(x && centers && idx && dist2, "x / centers / idx / dist2 missing");
    NearestWs b;
    carve_nearest(dtype, num_trees, m, dim, valid != nullptr, workspace, &b);
    if (b.total > 0 && (workspace == nullptr || workspace_bytes < b.total))
        return fail(HIRA_EWORKSPACE, "workspace %zu bytes, need %zu", workspace_bytes, b.total);
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    const size_t nm = (size_t)num_trees * m;
    if (valid != nullptr)
        hipLaunchKernelGGL(k_valid_to_fill, dim3((unsigned)((nm + 255) / 256)), dim3(256), 0, s,
                           valid, nm, b.fill);
    // a row without any usable centre keeps idx -1 and an infinite distance
    fill_i32(idx, (size_t)num_trees * n, -1, s);
    fill_i32(reinterpret_cast<int32_t*>(dist2), (size_t)num_trees * n, 0x7f800000, s);
    AssignJob job{};
    job.x = x;
    job.n_c = n;
    job.x_tree_stride = (size_t)n;
    job.dtype = dtype;
    job.D = dim;
    job.num_trees = num_trees;
    job.cent = centers;
    job.K = m;
    job.assign = idx;
    job.dist = dist2;
    if (b.tiles != nullptr) {
        rc = launch_cent_prep(dim, centers, m, num_trees, b.fill, 1, b.tiles, b.n2, s);
        job.ct = CentroidTiles{reinterpret_cast<uint4*>(b.tiles), b.n2, nullptr};
        if (rc == HIRA_OK) rc = launch_assign_mfma(job, s);
    } else {
        rc = dtype == HIRA_F32 ? launch_assign_simple<float>(job, b.fill, 1, s)
                               : launch_assign_simple<bf16_t>(job, b.fill, 1, s);
    }
    if (rc != HIRA_OK) return rc;
    HIRA_CHECK_LAUNCH("nearest-centre kernel");
    return HIRA_OK;
}
