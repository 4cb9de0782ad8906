// Whole small levels of an index build in one launch.
//
// A level of the build is some twenty launches: centroids, assignments, means, eight packing rounds of an
// assignment and an acceptance each, what is left over, block centres.  Where a level has a few
// hundred items none of them has work for the chip, and each costs its 4-14 us (the end of the launch
// before, first touch of its arguments, a chain of dependent trips to memory).  Here a workgroup of 16
// waves has a tree to itself and takes it through such a level, and through the levels above, from one
// barrier to the next.  The centroids do not move while blocks are packed, so the scores of all items and
// centroids are made once and stay in LDS (128 KiB for 1024 items and 32 centroids), and so do the centroids'
// operand tiles, the lists and the slots: a round of packing touches no memory.  What bounds it is the chain of
// barriers and, for the first assignment, the means, the scores and the block centres, trips to the level-2 cache.
// A level of 8 trees: 1024 items and 32 centroids 94 us (rounds 3-14), 128 and 4 20 us (rounds 1.5; with tiles and
// scores in memory, made anew every round, 32).  Builds, launches / with that / this: 2 x 1111 keys of 64 columns, five
// levels, fan-out 10: 426 / 207 / 181 us; 8 x 500, three levels, fan-out 32: 228 / 116 / 81; 8 x 8192, three levels,
// fan-out 32, the second level here: - / 395 / 365.
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

// items of a wave's stretch: the registers of a wave (128 with sixteen waves a workgroup) hold their
// operands and those of a centroid tile
constexpr int small_ri(int KS) { return KS <= 4 ? 2 : 1; }

// (whole item tiles, and the four rows that a tile's four lane groups write at a time in different banks)
constexpr int small_stride(int n_c) { return (n_c + 15) / 16 * 16 + 4; }

template <int KS>
struct SmallLds {
    static constexpr int kTileChunks = 2 * KS * 64;
    int16_t near[kSmallItems];     // of every item the centroid; -1: none, kPlaced: the item has its slot
    uint16_t members[kSmallItems]; // Lloyd: of the buckets, end to end, by id; packing: 64 a wave
    int32_t fill[kSmallCentroids], count[kSmallCentroids], first[kSmallCentroids];
    float n2[kSmallCentroids];     // squared norms of the centroids
    int32_t big[kSmallBig], big_at[kSmallBig];  // buckets of more than 64 items: the whole workgroup's
    int32_t n_big, n_keys, n_left;
    float x2[kSmallItems];         // squared norm of every item
    float dist[kSmallItems];       // of every item to its nearest centroid
    union {
        uint4 tiles[kSmallCentroids / 16 * kTileChunks];  // the centroids' operand tiles, until the scores are there
        struct {
            uint64_t keys[kSmallItems];  // proposers of the large buckets: (distance, id)
            uint16_t list[kSmallItems];  // what is left, by id
            int16_t slots[kSmallCentroids * 64];  // (K, bf)
        };
    };
    union {
        float piece[kSmallWaves][kWaveMeanPiece<bf16_t>];   // Lloyd
        // packing: the score ||c||^2 - 2 x.c of item i and centroid k at k * small_stride + i
        float score[small_pairs(32 * KS) + 20 * kSmallCentroids];
    };
};
static_assert(sizeof(SmallLds<2>) <= 160 * 1024 && sizeof(SmallLds<4>) <= 160 * 1024 && sizeof(SmallLds<8>) <= 160 * 1024, "LDS");

// emit_centroid into the tiles here: centroid k, D fp32 numbers at c (one wave)
template <int KS>
__device__ __forceinline__ void small_emit(SmallLds<KS>& s, const float* c, int k) {
    const int j = threadIdx.x & 63;
    float ss = 0.0f;
    if (j < KS * 4) {
        float hi[8], lo[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float v = c[j * 8 + e];
            hi[e] = bf16_bits_to_f32(f32_to_bf16_bits(v));
            lo[e] = bf16_bits_to_f32(f32_to_bf16_bits(v - hi[e]));
            const float w = hi[e] + lo[e];
            ss += w * w;
        }
        uint4* out = s.tiles + (k >> 4) * SmallLds<KS>::kTileChunks + (j >> 2) * 64 + (j & 3) * 16 + (k & 15);
        out[0] = make_uint4(pack_bf16(hi[0], hi[1]), pack_bf16(hi[2], hi[3]), pack_bf16(hi[4], hi[5]), pack_bf16(hi[6], hi[7]));
        out[KS * 64] = make_uint4(pack_bf16(lo[0], lo[1]), pack_bf16(lo[2], lo[3]), pack_bf16(lo[4], lo[5]), pack_bf16(lo[6], lo[7]));
    }
    ss = group_sum<32>(ss);
    if (j == 0) s.n2[k] = ss;
}

// SCORES: the scores of all items and centroids; else the nearest centroid of every item and the buckets' counts
template <int KS, bool SCORES>
__device__ __forceinline__ void small_assign(SmallLds<KS>& s, const void* x, size_t row0, int K, int n_items) {
    constexpr int D = 32 * KS, RI = small_ri(KS), ITEMS = RI * 16, TILE_CHUNKS = 2 * KS * 64;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n = lane & 15, kb = lane >> 4, tiles = (K + 15) / 16, stride = small_stride(n_items);
    for (int p0 = wave * ITEMS; p0 < n_items; p0 += kSmallWaves * ITEMS) {  // uniform in the wave
        uint4 x_op[RI][KS];
        float x2[RI], best[RI];
        int arg[RI];
#pragma unroll
        for (int ri = 0; ri < RI; ++ri)
#pragma unroll
            for (int c = 0; c < KS; ++c)
                x_op[ri][c] = *reinterpret_cast<const uint4*>(reinterpret_cast<const uint16_t*>(x) +
                                                              (row0 + min(p0 + ri * 16 + n, n_items - 1)) * D + c * 32 + kb * 8);
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
                x2[ri] = ss;
            }
        }
#pragma unroll
        for (int ri = 0; ri < RI; ++ri) {
            best[ri] = INFINITY;
            arg[ri] = -1;
        }
        for (int tile = 0; tile < tiles; ++tile) {
            const uint4* src = s.tiles + tile * TILE_CHUNKS + lane;
            uint4 c_op[2 * KS];
#pragma unroll
            for (int c = 0; c < 2 * KS; ++c) c_op[c] = src[c * 64];
            const float4 n2 = *reinterpret_cast<const float4*>(s.n2 + tile * 16 + 4 * kb);
            sf32x4_t acc[RI];
#pragma unroll
            for (int ri = 0; ri < RI; ++ri) acc[ri] = sf32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int c = 0; c < KS; ++c)
#pragma unroll
                for (int half = 0; half < 2; ++half)
#pragma unroll
                    for (int ri = 0; ri < RI; ++ri)
                        acc[ri] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(sbf16x8_t, c_op[half * KS + c]),
                                                                          __builtin_bit_cast(sbf16x8_t, x_op[ri][c]), acc[ri], 0, 0, 0);
            const float nn[4] = {n2.x, n2.y, n2.z, n2.w};
#pragma unroll
            for (int j = 0; j < 4; ++j) {  // (increasing: ties keep the lower one)
                const int k = tile * 16 + 4 * kb + j;
#pragma unroll
                for (int ri = 0; ri < RI; ++ri) {
                    const float v = nn[j] - 2.0f * acc[ri][j];
                    if constexpr (SCORES) {
                        if (k < K && p0 + ri * 16 < n_items) s.score[k * stride + p0 + ri * 16 + n] = v;
                    } else if (k < K && v < best[ri]) {  // (behind the last one a tile holds anything)
                        best[ri] = v;
                        arg[ri] = k;
                    }
                }
            }
        }
#pragma unroll
        for (int ri = 0; ri < RI; ++ri) {
            const int item = p0 + ri * 16 + n;
            if constexpr (SCORES) {
                if (kb == 0 && item < n_items) s.x2[item] = x2[ri];
            } else {
#pragma unroll
                for (int off = 16; off < 64; off <<= 1) {
                    const float ob = __shfl_xor(best[ri], off, 64);
                    const int og = __shfl_xor(arg[ri], off, 64);
                    if (og >= 0 && (arg[ri] < 0 || ob < best[ri] || (ob == best[ri] && og < arg[ri]))) {
                        best[ri] = ob;
                        arg[ri] = og;
                    }
                }
                if (kb == 0 && item < n_items) {
                    s.near[item] = (int16_t)arg[ri];
                    if (arg[ri] >= 0) atomicAdd(&s.count[arg[ri]], 1);
                }
            }
        }
    }
}

// where the bucket of every centroid begins (K <= kSmallCentroids; one wave)
template <int KS>
__device__ __forceinline__ void small_offsets(SmallLds<KS>& s, int K) {
    const int lane = threadIdx.x & 63;
    int before = 0;
    for (int k0 = 0; k0 < K; k0 += 64) {
        const int mine = k0 + lane < K ? s.count[k0 + lane] : 0;
        int inc = mine;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int o = __shfl_up(inc, off, 64);
            if (lane >= off) inc += o;
        }
        if (k0 + lane < K) s.first[k0 + lane] = before + inc - mine;
        before += __shfl(inc, 63, 64);
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

// wave_mean over 256 threads: their sums over the m rows members[at ..), R rows of D numbers, to part
template <int KS>
__device__ __forceinline__ void small_big_sums(const SmallLds<KS>& s, const void* x, size_t row0, int at, int m, float* part) {
    constexpr int D = 32 * KS, EPL = 8, CPR = D / EPL, R = 256 / CPR, U = 4;  // (U rows on their way)
    const int i = threadIdx.x & 255, r = i / CPR, c = i % CPR;
    float acc[EPL];
#pragma unroll
    for (int q = 0; q < EPL; ++q) acc[q] = 0.0f;
    for (int e = r; e < m; e += U * R) {
        uint4 raw[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            raw[u] = make_uint4(0, 0, 0, 0);  // (a row that is none adds zeros)
            if (e + u * R < m) raw[u] = load_chunk<bf16_t>(x, (row0 + s.members[at + e + u * R]) * D, c);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            float f[EPL];
            unpack<bf16_t>(raw[u], f);
#pragma unroll
            for (int q = 0; q < EPL; ++q) acc[q] += f[q];
        }
    }
#pragma unroll
    for (int q = 0; q < EPL; ++q) part[r * D + c * EPL + q] = acc[q];
}
// the sums added in order; the mean's D numbers to cent_row and to part[0 .. D) (a thread's column is
// nobody else's)
template <int KS>
__device__ __forceinline__ void small_big_mean(float* part, int m, float* cent_row) {
    constexpr int D = 32 * KS, R = 256 / (D / 8);
    const int j = threadIdx.x & 255, rows = min(R, m);
    if (j >= D) return;
    float sum = 0.0f;
    for (int q = 0; q < rows; ++q) sum += part[q * D + j];
    const float v = sum / (float)m;
    cent_row[j] = v;
    part[j] = v;
}

template <int KS>
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

        // ---- empty blocks, first centroids -------------------------------------------------------
        for (int i = tid; i < K; i += kSmallThreads) {
            s.fill[i] = i >= K_t ? bf : 0;
            s.count[i] = 0;
        }
        if (tid == 0) s.n_big = 0;
        constexpr int kMine = (kSmallCentroids + kSmallWaves - 1) / kSmallWaves, NJ = D / 64;
        float first[kMine][NJ];  // (a wave's centroids, asked for together)
#pragma unroll
        for (int i = 0; i < kMine; ++i) {
            const int k = min(wave + i * kSmallWaves, K - 1);
            const size_t src = (row0 + (size_t)first_centroid(p.seed + 7919ull * (uint64_t)l, t, k, max(n_c, 1), K_t)) * D;
#pragma unroll
            for (int j = 0; j < NJ; ++j) first[i][j] = load_elem<bf16_t>(x, src + j * 64 + lane);
        }
#pragma unroll
        for (int i = 0; i < kMine; ++i) {
            const int k = wave + i * kSmallWaves;
            if (k >= K) break;  // uniform
#pragma unroll
            for (int j = 0; j < NJ; ++j) cent[(size_t)k * D + j * 64 + lane] = piece[j * 64 + lane] = first[i][j];
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            small_emit<KS>(s, piece, k);
            if (lane == 0 && k >= K_t) s.n2[k] = INFINITY;
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        }
        __syncthreads();

        // ---- Lloyd rounds ------------------------------------------------------------------------
        for (int r = 0; r < p.niter; ++r) {
            small_assign<KS, false>(s, x, row0, K, n_c);
            __syncthreads();
            if (wave == 0) small_offsets(s, K);
            __syncthreads();
            for (int k = wave; k < K; k += kSmallWaves) {
                const int m = __builtin_amdgcn_readfirstlane(s.count[k]), at = __builtin_amdgcn_readfirstlane(s.first[k]);
                if (m == 0) continue;
                small_members(s, k, m, n_c, [&](int e, int it) { s.members[at + e] = (uint16_t)it; });
                if (m > 64) {
                    if (lane == 0) s.big[atomicAdd(&s.n_big, 1)] = k;
                    continue;
                }
                wave_mean<bf16_t, 1>(x, row0, [&](int e) { return (uint32_t)s.members[at + e]; }, m, D, piece,
                                     cent + (size_t)k * D);
                small_emit<KS>(s, piece, k);
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                if (lane == 0) s.count[k] = 0;
            }
            __syncthreads();
            // the large ones, four at a time: 256 threads each, with the sums of wave_mean
            const int n_big = __builtin_amdgcn_readfirstlane(s.n_big);
            float* part = s.piece[wave & ~3];
            for (int b0 = 0; b0 < n_big; b0 += kSmallWaves / 4) {  // uniform
                const int b = b0 + (wave >> 2), k = b < n_big ? s.big[b] : 0;
                const int m = b < n_big ? s.count[k] : 0, at = s.first[k];
                small_big_sums<KS>(s, x, row0, at, m, part);
                __syncthreads();
                if (b < n_big) small_big_mean<KS>(part, m, cent + (size_t)k * D);
                __syncthreads();
                if (b < n_big && (wave & 3) == 0) {
                    small_emit<KS>(s, part, k);
                    if (lane == 0) s.count[k] = 0;
                }
                __syncthreads();
            }
            if (tid == 0) s.n_big = 0;  // (read by everybody ahead of a barrier: none was passed if there were none)
        }

        // ---- capacity packing: the closest proposers of a bucket (by distance, then id) take the free
        // slots of the block in that order, the others try again.  The centroids stay what they are, so
        // the scores are made once, and a round is a look at those of the centroids with room, a thread an item.
        __syncthreads();  // (the last centroids' tiles are written)
        small_assign<KS, true>(s, x, row0, K, n_c);
        if (tid < n_c) s.near[tid] = -1;
        if (tid == 0) s.n_left = n_c;
        __syncthreads();
        for (int i = tid; i < K * bf; i += kSmallThreads) s.slots[i] = -1;  // (where the tiles were)
        const int stride = small_stride(n_c);
        const float x2 = tid < n_c ? s.x2[tid] : 0.0f;
        uint16_t* const mem = s.members + wave * 64;
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
                if (arg >= 0) atomicAdd(&s.count[arg], 1);
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
                if (m > 64) {
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
                small_members(s, k, m, n_c, [&](int e, int it) { mem[e] = (uint16_t)it; });
                const uint64_t mine = lane < m ? key_of(mem[lane]) : ~0ull;
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
        if (wave == 0) {
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
        for (int k = wave; k < K; k += kSmallWaves)
            wave_block_mean<bf16_t, 4>(x, row0, D, lane < bf ? s.slots[k * bf + lane] : -1, bf, p.lpr, ((size_t)t * K + k) * D, p.cent,
                                       p.cent_t[l]);
        __syncthreads();  // (the next level reads them)
    }
}

template <int KS>
static int launch_small(const SmallLevels& p, int num_trees, hipStream_t s) {
    static int asked[kMaxDevices];
    if (const int rc = ask_for_lds(reinterpret_cast<const void*>(&k_small_levels<KS>), sizeof(SmallLds<KS>), asked, current_device()))
        return rc;
    hipLaunchKernelGGL((k_small_levels<KS>), dim3(num_trees), dim3(kSmallThreads), sizeof(SmallLds<KS>), s, p);
    return HIRA_OK;
}

int launch_small_levels(const SmallLevels& p, int D, int num_trees, hipStream_t s) {
    switch (D) {
        case 64: return launch_small<2>(p, num_trees, s);
        case 128: return launch_small<4>(p, num_trees, s);
        case 256: return launch_small<8>(p, num_trees, s);
        default: return fail(HIRA_EINVAL, "small levels: %d columns", D);
    }
}

}  // namespace hira
