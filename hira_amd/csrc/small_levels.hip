// Whole small levels of an index build in one launch.
//
// A level of the build is some twenty launches: centroids, assignments, means, eight packing rounds of an
// assignment and an acceptance each, what is left over, block centres.  Where a level has a few
// hundred items none of them has work for the chip, and each costs its 4-14 us (the end of the launch
// before, first touch of its arguments, a chain of dependent trips to memory).  Here a workgroup of 16
// waves has a tree to itself and takes it through such a level, and through the levels above, from one
// barrier to the next.  The centroids do not move while blocks are packed, so the scores of all items and
// centroids are made once and stay in LDS (128 KiB for 1024 items and 32 centroids), and so do the centroids'
// operand tiles, the lists and the slots: a round of packing touches no memory.  Sixteen waves on one compute unit are bound
// by their instructions, and by trips to the level-2 cache for the rows, which are gathered four times (first
// assignment, means, scores, block centres; the first and the third are asked for ahead, under the first centroids and the means).
// A launch, 8 trees of 128 columns: 1024 items and 32 centroids 64 us, 256 and 8 21, 126 and 4 16.5; 2 x 112 x 12 of 64 columns
// and the two levels above 28.7 (95, 33, 27.5 and 49 with the items asked for where they were used, buckets looked for among
// all items, a wave a centroid at the start and a block at a time at the end; 74, 26.6, 21.5 and 40 with all that and numbers
// rounded to bf16 by shifts and additions).
//
// The numbers are those of the launches, bit for bit: the same products in the same order, means and
// block centres by the same functions (cluster.h), and rules that do not depend on the order of
// arrival there either (the closest first, then the lowest id).
#include "small_levels.h"

namespace hira {

typedef __attribute__((ext_vector_type(8))) __bf16 sbf16x8_t;
typedef __attribute__((ext_vector_type(4))) float sf32x4_t;

constexpr int kSmallThreads = 1024;
constexpr int kSmallWaves = kSmallThreads / 64;
static_assert(kSmallThreads >= kSmallItems, "the packing gives every item a thread");
constexpr int kPlaced = -2;
constexpr int kSmallBig = kSmallItems / 65 + 1;

// RI, below: item tiles a wave holds at a time, every sixteenth of the tree's: all of its own at the launch's first level, up
// to four; one of rows of 256 columns, which take twice the registers (a wave has 128).  (Chosen inside the launch, the two sets
// of registers met in spills: 8 x 1024 x 32 74 -> 112 us; four whatever the items: 128 x 4 25 -> 37.  Four tiles of 128 columns
// spill too, 41 registers a lane, the others three to five.)
// Steps of a bucket's rows on their way.  (One wave has a bucket, however many items it has.  Four waves for each of more than
// 128 items, or four steps of it: what both take from the registers costs every other level more than they gain.  Launches of
// 8 x 1024 x 32 keys of 128 columns as a build by itself, one wave / four waves / four steps: drawn from a normal distribution 90 / 94 / 90 us, six
// of seven close to one another 117 / 120 / 117, seven of eight the same row 276 / 274 / 274; 8 x 256 25 / 27 / 30.  Before one wave had
// them and items were asked for ahead 113, 130, 268 and 37; 8 x 512 x 16 of 256 columns, seven of eight the same row, 133 -> 144.)
constexpr int kSmallMean = 2;
constexpr int kSmallPlaces = 64;  // of a bucket, for items in order of arrival: what a wave ranks in registers

// (whole item tiles, and the four rows that a tile's four lane groups write at a time in different banks)
constexpr int small_stride(int n_c) { return (n_c + 15) / 16 * 16 + 4; }

template <int KS>
struct SmallLds {
    static constexpr int kTileChunks = 2 * KS * 64;
    int16_t near[kSmallItems];     // of every item the centroid; -1: none, kPlaced: the item has its slot
    int32_t fill[kSmallCentroids], count[kSmallCentroids];
    float n2[kSmallCentroids];     // squared norms of the centroids
    int32_t big[kSmallBig], big_at[kSmallBig];  // packing: buckets of more than kSmallPlaces items, the whole workgroup's
    int32_t n_big, n_keys, n_left;
    float x2[kSmallItems];         // squared norm of every item
    float dist[kSmallItems];       // of every item to its nearest centroid
    union {
        uint4 tiles[kSmallCentroids / 16 * kTileChunks];  // the centroids' operand tiles, until the scores are there
        struct {
            uint64_t keys[kSmallItems];  // proposers of the large buckets: (distance, id)
            union {
                uint16_t pack_places[kSmallCentroids * kSmallPlaces];
                uint16_t list[kSmallItems];  // what is left, by id
            };
            int16_t slots[kSmallCentroids * 64];  // (K, bf)
        };
    };
    union {
        struct {  // Lloyd
            float piece[kSmallWaves][kWaveMeanPiece<bf16_t>];
            uint16_t places[kSmallCentroids * kSmallPlaces];
            uint16_t members[kSmallItems];  // of the large buckets, end to end, each by id
        };
        // packing: the score ||c||^2 - 2 x.c of item i and centroid k at k * small_stride + i
        float score[small_pairs(32 * KS) + 20 * kSmallCentroids];
    };
};
static_assert(sizeof(SmallLds<2>) <= 160 * 1024 && sizeof(SmallLds<4>) <= 160 * 1024 && sizeof(SmallLds<8>) <= 160 * 1024, "LDS");

// emit_columns into the tiles here: columns 8 j .. 8 j + 7 of centroid k; `lanes` consecutive lanes hold a centroid
template <int KS>
__device__ __forceinline__ void small_emit(SmallLds<KS>& s, const float (&v)[8], int j, int lanes, bool have, int k, bool usable) {
    float ss = 0.0f;
    if (have && j < KS * 4) {
        uint4 hi, lo;
        float ls = 0.0f;
        split_bf16(v, hi, lo, ss, ls);
        uint4* out = s.tiles + (k >> 4) * SmallLds<KS>::kTileChunks + (j >> 2) * 64 + (j & 3) * 16 + (k & 15);
        out[0] = hi;
        out[KS * 64] = lo;
    }
    ss = group_sum_of(ss, lanes);
    if (have && j == 0) s.n2[k] = usable ? ss : INFINITY;
}
// the same with the centroid's D fp32 numbers at c (one wave)
template <int KS>
__device__ __forceinline__ void small_emit(SmallLds<KS>& s, const float* c, int k) {
    const int j = threadIdx.x & 63;
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = j < KS * 4 ? c[j * 8 + e] : 0.0f;
    small_emit<KS>(s, v, j, 32, true, k, true);
}

// The operands of a wave's next item tiles, from its tile number q0 on (tile q of wave w: items (16 q + w) * 16 ..): asked
// for well ahead of small_assign, which takes them.
template <int KS, int RI>
__device__ __forceinline__ void small_items(const void* x, size_t row0, int n_items, int q0, uint4 (&x_op)[RI][KS]) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n = lane & 15, kb = lane >> 4;
#pragma unroll
    for (int ri = 0; ri < RI; ++ri) {
        const int p0 = ((q0 + ri) * kSmallWaves + wave) * 16;
#pragma unroll
        for (int c = 0; c < KS; ++c)  // (whatever the tile: a load under a condition is waited for where that ends)
            x_op[ri][c] = *reinterpret_cast<const uint4*>(reinterpret_cast<const uint16_t*>(x) +
                                                          (row0 + max(min(p0 + n, n_items - 1), 0)) * (32 * KS) + c * 32 + kb * 8);
    }
}

// SCORES: the scores of all items and centroids; else the nearest centroid of every item, the buckets' counts and the
// first kSmallPlaces items of each.  x_op: small_items of the first tiles.
template <int KS, int RI, bool SCORES>
__device__ __forceinline__ void small_assign(SmallLds<KS>& s, const void* x, size_t row0, int K, int n_items, uint4 (&x_op)[RI][KS]) {
    constexpr int TILE_CHUNKS = 2 * KS * 64;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n = lane & 15, kb = lane >> 4, tiles = (K + 15) / 16, stride = small_stride(n_items);
    for (int q0 = 0; (q0 * kSmallWaves + wave) * 16 < n_items; q0 += RI) {  // uniform in the wave
        if (q0 > 0) small_items<KS, RI>(x, row0, n_items, q0, x_op);
        auto first = [&](int ri) { return ((q0 + ri) * kSmallWaves + wave) * 16; };
        float best[RI];
        int arg[RI];
        if constexpr (SCORES) {
#pragma unroll
            for (int ri = 0; ri < RI; ++ri) {
                float ss = 0.0f;
#pragma unroll
                for (int c = 0; c < KS; ++c) {
                    float f[8];
                    unpack<bf16_t>(x_op[ri][c], f);
#pragma unroll
                    for (int e = 0; e < 8; ++e) ss += f[e] * f[e];
                }
                ss = cross_group_sum<16>(ss);
                if (kb == 0 && first(ri) + n < n_items) s.x2[first(ri) + n] = ss;
            }
        } else {
#pragma unroll
            for (int ri = 0; ri < RI; ++ri) {
                best[ri] = INFINITY;
                arg[ri] = -1;
            }
        }
        for (int tile = 0; tile < tiles; ++tile) {
            const uint4* src = s.tiles + tile * TILE_CHUNKS + lane;
            const float4 n2 = *reinterpret_cast<const float4*>(s.n2 + tile * 16 + 4 * kb);
            sf32x4_t acc[RI];
#pragma unroll
            for (int ri = 0; ri < RI; ++ri) acc[ri] = sf32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int c = 0; c < KS; ++c) {
#pragma unroll
                for (int half = 0; half < 2; ++half) {
                    const sbf16x8_t c_op = __builtin_bit_cast(sbf16x8_t, src[(half * KS + c) * 64]);
#pragma unroll
                    for (int ri = 0; ri < RI; ++ri)
                        acc[ri] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(c_op, __builtin_bit_cast(sbf16x8_t, x_op[ri][c]), acc[ri], 0, 0, 0);
                }
                __builtin_amdgcn_sched_barrier(0);  // (a tile's operands all at once are more than there are registers for)
            }
            const float nn[4] = {n2.x, n2.y, n2.z, n2.w};
#pragma unroll
            for (int j = 0; j < 4; ++j) {  // (increasing: ties keep the lower one)
                const int k = tile * 16 + 4 * kb + j;
#pragma unroll
                for (int ri = 0; ri < RI; ++ri) {
                    const float v = nn[j] - 2.0f * acc[ri][j];
                    if constexpr (SCORES) {
                        if (k < K && first(ri) < n_items) s.score[k * stride + first(ri) + n] = v;
                    } else if (k < K && v < best[ri]) {  // (behind the last one a tile holds anything)
                        best[ri] = v;
                        arg[ri] = k;
                    }
                }
            }
        }
        if constexpr (!SCORES) {
            int mine = -1, item = n_items;  // lane (kb, n): item n of tile kb (lane groups from RI on: none)
#pragma unroll
            for (int ri = 0; ri < RI; ++ri) {
                auto nearer = [&](auto v, auto k) {  // of the two lanes that a swap has paired, in both of them
                    const float v0 = __uint_as_float((uint32_t)v[0]), v1 = __uint_as_float((uint32_t)v[1]);
                    const int k0 = (int)k[0], k1 = (int)k[1];
                    const bool second = k1 >= 0 && (k0 < 0 || v1 < v0 || (v1 == v0 && k1 < k0));
                    best[ri] = second ? v1 : v0;
                    arg[ri] = second ? k1 : k0;
                };
                nearer(__builtin_amdgcn_permlane16_swap(__float_as_uint(best[ri]), __float_as_uint(best[ri]), false, false),
                       __builtin_amdgcn_permlane16_swap((uint32_t)arg[ri], (uint32_t)arg[ri], false, false));
                nearer(__builtin_amdgcn_permlane32_swap(__float_as_uint(best[ri]), __float_as_uint(best[ri]), false, false),
                       __builtin_amdgcn_permlane32_swap((uint32_t)arg[ri], (uint32_t)arg[ri], false, false));
                if (kb == ri) {
                    mine = arg[ri];
                    item = first(ri) + n;
                }
            }
            if (item < n_items) {
                s.near[item] = (int16_t)mine;
                if (mine >= 0) {
                    const int at = atomicAdd(&s.count[mine], 1);
                    if (at < kSmallPlaces) s.places[mine * kSmallPlaces + at] = (uint16_t)item;
                }
            }
        }
    }
}

// f(place, item) for the m items of bucket k, places by id (one wave)
template <int KS, typename F>
__device__ __forceinline__ void small_members(const SmallLds<KS>& s, int k, int m, int n_items, F f) {
    const int lane = threadIdx.x & 63;
    int found = 0;
    for (int p0 = 0; p0 < n_items && found < m; p0 += 4 * 64) {  // uniform
        bool in[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int it = p0 + u * 64 + lane;
            in[u] = it < n_items && s.near[min(it, n_items - 1)] == k;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const unsigned long long bal = __ballot(in[u]);
            if (in[u]) f(found + __popcll(bal & ((1ull << lane) - 1ull)), p0 + u * 64 + lane);
            found += __popcll(bal);
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

// items that have no slot yet, by id, to list; returns how many (one wave)
template <int KS>
__device__ __forceinline__ int small_left(SmallLds<KS>& s, int n) {
    const int lane = threadIdx.x & 63;
    int at = 0;
    for (int p0 = 0; p0 < n; p0 += 64) {  // uniform
        const int it = p0 + lane;
        const bool in = it < n && s.near[min(it, n - 1)] != kPlaced;
        const unsigned long long bal = __ballot(in);
        if (in) s.list[at + __popcll(bal & ((1ull << lane) - 1ull))] = (uint16_t)it;
        at += __popcll(bal);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    return at;
}

template <int KS, int RI>
__global__ __launch_bounds__(kSmallThreads) void k_small_levels(const SmallLevels p) {
    constexpr int D = 32 * KS;
    extern __shared__ uint64_t s_raw[];
    SmallLds<KS>& s = *reinterpret_cast<SmallLds<KS>*>(s_raw);
    const int t = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int bf = p.bf;
    for (int l = p.first; l < p.last; ++l) {  // uniform, and so are the loops over rounds
        const int K = p.K[l];
        // (a tree with fewer items uses its first K_t centroids only: the others count as full)
        const int n_c = p.n_live == nullptr ? p.K[l - 1] : min(max(p.n_live[t], 0), p.K[l - 1]);
        const int K_t = p.n_live == nullptr ? K : min(max((n_c + bf - 1) / bf, 1), K);
        const void* x = l == p.first ? p.x : p.cent_t[l - 1];
        const size_t row0 = (size_t)t * p.K[l - 1];
        int32_t* slots = p.slots[l] + (size_t)t * K * bf;
        float* cent = p.cent + (size_t)t * K * D;
        float* piece = s.piece[wave];

        // ---- empty blocks, first centroids (all of them at once, KS * 4 lanes each), the items' operands --------
        for (int i = tid; i < K; i += kSmallThreads) {
            s.fill[i] = i >= K_t ? bf : 0;
            s.count[i] = 0;
        }
        if (tid == 0) s.n_big = s.n_keys = 0;
        uint4 x_op[RI][KS];
        {
            constexpr int LANES = KS * 4;
            static_assert(kSmallThreads / LANES >= kSmallCentroids, "a pass for all centroids");
            const int k = tid / LANES, j = lane % LANES, own = min(k, K - 1);
            const size_t src = (row0 + (size_t)first_centroid(p.seed + 7919ull * (uint64_t)l, t, own, max(n_c, 1), K_t)) * D;
            const uint4 raw = load_chunk<bf16_t>(x, src, j);
            small_items<KS, RI>(x, row0, n_c, 0, x_op);
            float v[8];
            unpack<bf16_t>(raw, v);
            if (k < K) {
                float4* dst = reinterpret_cast<float4*>(cent + (size_t)k * D + j * 8);
                dst[0] = make_float4(v[0], v[1], v[2], v[3]);
                dst[1] = make_float4(v[4], v[5], v[6], v[7]);
            }
            small_emit<KS>(s, v, j, LANES, k < K, own, own < K_t);
        }
        __syncthreads();

        // ---- Lloyd rounds ------------------------------------------------------------------------
        for (int r = 0; r < p.niter; ++r) {
            small_assign<KS, RI, false>(s, x, row0, K, n_c, x_op);
            __syncthreads();
            for (int k = wave; k < K; k += kSmallWaves) {
                const int m = __builtin_amdgcn_readfirstlane(s.count[k]);
                if (m == 0) continue;
                uint16_t* ids = s.places + k * kSmallPlaces;
                if (m <= kSmallPlaces) {  // by id
                    const uint32_t id = lane < m ? ids[lane] : 0xffffffffu;
                    const int rank = wave_rank(id, m);
                    if (lane < m) ids[rank] = (uint16_t)id;
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                } else {
                    int at = 0;
                    if (lane == 0) at = atomicAdd(&s.n_keys, m);
                    ids = s.members + __builtin_amdgcn_readfirstlane(at);
                    small_members(s, k, m, n_c, [&](int e, int it) { ids[e] = (uint16_t)it; });
                }
                wave_mean<bf16_t, kSmallMean>(x, row0, [&](int e) { return (uint32_t)ids[e]; }, m, D, piece, cent + (size_t)k * D);
                small_emit<KS>(s, piece, k);
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                if (lane == 0) s.count[k] = 0;
            }
            small_items<KS, RI>(x, row0, n_c, 0, x_op);  // (for what comes next)
            __syncthreads();
            if (tid == 0) s.n_keys = 0;
        }

        // ---- capacity packing: the closest proposers of a bucket (by distance, then id) take the free
        // slots of the block in that order, the others try again.  The centroids stay what they are, so
        // the scores are made once, and a round is a look at those of the centroids with room, a thread an item.
        small_assign<KS, RI, true>(s, x, row0, K, n_c, x_op);
        if (tid < n_c) s.near[tid] = -1;
        if (tid == 0) s.n_left = n_c;
        __syncthreads();
        for (int i = tid; i < K * bf; i += kSmallThreads) s.slots[i] = -1;  // (where the tiles were)
        const int stride = small_stride(n_c);
        const float x2 = tid < n_c ? s.x2[tid] : 0.0f;
        auto key_of = [&](uint32_t it) { return ((uint64_t)__float_as_uint(s.dist[it]) << 32) | it; };
        for (int r = 0; r < p.pack_rounds; ++r) {
            if (tid == 0) s.n_keys = 0;
            const unsigned long long with_room = __ballot(lane < K && s.fill[min(lane, K - 1)] < bf);  // (of all lanes: placed items' too)
            if (tid < n_c && s.near[tid] != kPlaced) {
                float best = INFINITY;
                int arg = -1;
                for (unsigned long long open = with_room; open != 0ull; open &= open - 1ull) {  // uniform
                    const int k = __ffsll((long long)open) - 1;
                    const float v = s.score[k * stride + tid];
                    if (v < best) {  // (increasing: ties keep the lower one)
                        best = v;
                        arg = k;
                    }
                }
                s.near[tid] = (int16_t)arg;
                s.dist[tid] = fmaxf(best + x2, 0.0f);
                if (arg >= 0) {
                    const int at = atomicAdd(&s.count[arg], 1);
                    if (at < kSmallPlaces) s.pack_places[arg * kSmallPlaces + at] = (uint16_t)tid;
                }
            }
            __syncthreads();
            auto filled = [&](int k, int f, int take) {  // (one thread)
                s.count[k] = 0;
                s.fill[k] = f + take;
                atomicSub(&s.n_left, take);
            };
            for (int k = wave; k < K; k += kSmallWaves) {
                const int m = __builtin_amdgcn_readfirstlane(s.count[k]);
                if (m == 0) continue;
                const int f = __builtin_amdgcn_readfirstlane(s.fill[k]), take = max(min(m, bf - f), 0);
                if (m > kSmallPlaces) {
                    int at = 0;
                    if (lane == 0) at = atomicAdd(&s.n_keys, m);
                    at = __builtin_amdgcn_readfirstlane(at);
                    small_members(s, k, m, n_c, [&](int e, int it) { s.keys[at + e] = key_of((uint32_t)it); });
                    if (lane == 0) {
                        const int b = atomicAdd(&s.n_big, 1);
                        s.big[b] = k;
                        s.big_at[b] = at;
                    }
                    continue;
                }
                const uint64_t mine = lane < m ? key_of(s.pack_places[k * kSmallPlaces + lane]) : ~0ull;
                const int rank = wave_rank(mine, m);
                if (lane < m && rank < take) {
                    s.slots[k * bf + f + rank] = (int16_t)(uint32_t)mine;
                    s.near[(uint32_t)mine] = kPlaced;
                }
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                if (lane == 0) filled(k, f, take);
            }
            __syncthreads();
            const int n_big = __builtin_amdgcn_readfirstlane(s.n_big);
            if (n_big > 0) {  // uniform
                if (tid < s.n_keys) {  // (no more than items: a proposer a thread, of all these buckets)
                    int b = 0;
                    while (tid < s.big_at[b] || tid >= s.big_at[b] + s.count[s.big[b]]) ++b;
                    const int k = s.big[b], m = s.count[k], f = s.fill[k];
                    const uint64_t mine = s.keys[tid];
                    const uint64_t* all = s.keys + s.big_at[b];
                    int rank = 0, j = 0;
                    for (; j + 8 <= m; j += 8)
#pragma unroll
                        for (int u = 0; u < 8; ++u) rank += all[j + u] < mine ? 1 : 0;
                    for (; j < m; ++j) rank += all[j] < mine ? 1 : 0;
                    if (rank < max(min(m, bf - f), 0)) {
                        s.slots[k * bf + f + rank] = (int16_t)(uint32_t)mine;
                        s.near[(uint32_t)mine] = kPlaced;
                    }
                }
                __syncthreads();
                if (tid < n_big) {
                    const int k = s.big[tid], f = s.fill[k];
                    filled(k, f, max(min(s.count[k], bf - f), 0));
                }
                __syncthreads();
            }
            if (tid == 0) s.n_big = 0;
            if (__builtin_amdgcn_readfirstlane(s.n_left) == 0) break;  // uniform: nobody writes it until the next barrier
        }
        __syncthreads();

        // ---- what is left, and items that are no numbers, to the free slots in order ------------------
        if (wave == 0 && s.n_left != 0) {
            const int total = small_left(s, n_c);
            int before = 0;
            for (int k0 = 0; k0 < K && before < total; k0 += 64) {  // uniform
                const int k = k0 + lane, f = k < K ? s.fill[k] : bf, room = max(bf - f, 0);
                int inc = room;
#pragma unroll
                for (int off = 1; off < 64; off <<= 1) {
                    const int o = __shfl_up(inc, off, 64);
                    if (lane >= off) inc += o;
                }
                const int at = before + inc - room;
                for (int j = 0; j < room && at + j < total; ++j) s.slots[k * bf + f + j] = (int16_t)s.list[at + j];
                before += __shfl(inc, 63, 64);
            }
        }
        __syncthreads();
        // ---- block centres ----------------------------------------------------------------------------
        for (int i = tid; i < K * bf; i += kSmallThreads) slots[i] = s.slots[i];
        for (int k = wave; k < K; k += 2 * kSmallWaves) {  // uniform; two at a time
            int slot[2];
            size_t out[2];
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                const int own = min(k + b * kSmallWaves, K - 1);
                slot[b] = lane < bf && k + b * kSmallWaves < K ? s.slots[own * bf + lane] : -1;
                out[b] = ((size_t)t * K + own) * D;
            }
            wave_block_means<bf16_t, 4, 2>(x, row0, D, slot, k + kSmallWaves < K ? 2 : 1, bf, KS * 4, out, p.cent, p.cent_t[l]);
        }
        __syncthreads();  // (the next level reads them)
    }
}

template <int KS, int RI>
static int launch_small(const SmallLevels& p, int num_trees, hipStream_t s) {
    static int asked[kMaxDevices];
    if (const int rc = ask_for_lds(reinterpret_cast<const void*>(&k_small_levels<KS, RI>), sizeof(SmallLds<KS>), asked, current_device()))
        return rc;
    hipLaunchKernelGGL((k_small_levels<KS, RI>), dim3(num_trees), dim3(kSmallThreads), sizeof(SmallLds<KS>), s, p);
    return HIRA_OK;
}

template <int KS>
static int launch_small_of(const SmallLevels& p, int num_trees, hipStream_t s) {
    const int tiles = (p.K[p.first - 1] + 16 * kSmallWaves - 1) / (16 * kSmallWaves);  // of a wave
    if constexpr (KS <= 4) {
        if (tiles > 2) return launch_small<KS, 4>(p, num_trees, s);
        if (tiles > 1) return launch_small<KS, 2>(p, num_trees, s);
    }
    return launch_small<KS, 1>(p, num_trees, s);
}

int launch_small_levels(const SmallLevels& p, int D, int num_trees, hipStream_t s) {
    switch (D) {
        case 64: return launch_small_of<2>(p, num_trees, s);
        case 128: return launch_small_of<4>(p, num_trees, s);
        case 256: return launch_small_of<8>(p, num_trees, s);
        default: return fail(HIRA_EINVAL, "small levels: %d columns", D);
    }
}

}  // namespace hira
