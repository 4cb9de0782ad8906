// Whole small levels of an index build in one launch.
//
// A level of the build is some twenty launches: centroids, assignments, means, eight packing rounds of an
// assignment and an acceptance each, what is left over, block centres.  Where a level has a few
// hundred items none of them has work for the chip, and each costs its 4-14 us (the end of the launch
// before, first touch of its arguments, a chain of dependent trips to memory).  Here a workgroup of 16
// waves has a tree to itself and takes it through such a level, and through the levels above, from one
// barrier to the next; what a round leaves for the one after it (nearest centroid and distance of every
// item, members of the buckets, the list) stays in LDS.  What bounds it is the chain of a round, 5-6 us of
// barriers and trips to the level-2 cache.  Builds, launches -> this: 2 x 1111 keys of 64 columns, five
// levels, fan-out 10: 426 -> 208 us; 8 x 500, three levels, fan-out 32: 228 -> 142; 8 x 256, two levels:
// 122 -> 80; the third level of 8 x 131072 keys (128 items): about 110 -> 53.
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
constexpr int kPlaced = -2;
constexpr int kSmallBig = kSmallItems / 65 + 1;

// items of a wave's stretch: the registers of a wave (128 with sixteen waves a workgroup) hold their
// operands and those of a centroid tile
constexpr int small_ri(int KS) { return KS <= 4 ? 2 : 1; }

struct SmallLds {
    float dist[kSmallItems];       // of every item to its nearest centroid
    int16_t near[kSmallItems];     // the centroid; -1: none, kPlaced: the item has its slot
    uint16_t list[kSmallItems];    // items of the round, by id
    uint16_t members[kSmallItems]; // of the buckets, end to end, by id
    int32_t fill[kSmallCentroids], count[kSmallCentroids], first[kSmallCentroids];
    int32_t big[kSmallBig];        // buckets of more than 64 items: the whole workgroup's
    int32_t n_big, n_list;
    uint64_t keys[kSmallItems];    // of a round's proposers: (distance, id), as `members`
    float piece[kSmallWaves][kWaveMeanPiece<bf16_t>];
};

// nearest usable centroid of items list[0 .. n_items) (all: of items 0 .. n_items)
template <int KS>
__device__ __forceinline__ void small_assign(SmallLds& s, const void* x, size_t row0, const uint4* tt, const float* n2t,
                                             int tiles, bool all, int n_items) {
    constexpr int D = 32 * KS, RI = small_ri(KS), ITEMS = RI * 16, TILE_CHUNKS = 2 * KS * 64;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n = lane & 15, kb = lane >> 4;
    for (int p0 = wave * ITEMS; p0 < n_items; p0 += kSmallWaves * ITEMS) {  // uniform in the wave
        int item[RI];
        uint4 x_op[RI][KS];
        float x2[RI], best[RI];
        int arg[RI];
#pragma unroll
        for (int ri = 0; ri < RI; ++ri) {
            const int pos = p0 + ri * 16 + n;
            item[ri] = pos < n_items ? (all ? pos : (int)s.list[pos]) : -1;
        }
#pragma unroll
        for (int ri = 0; ri < RI; ++ri)
#pragma unroll
            for (int c = 0; c < KS; ++c)
                x_op[ri][c] = *reinterpret_cast<const uint4*>(reinterpret_cast<const uint16_t*>(x) +
                                                              (row0 + max(item[ri], 0)) * D + c * 32 + kb * 8);
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
            ss += __shfl_xor(ss, 16, 64);
            ss += __shfl_xor(ss, 32, 64);
            x2[ri] = ss;
            best[ri] = INFINITY;
            arg[ri] = -1;
        }
        for (int tile = 0; tile < tiles; ++tile) {
            const uint4* src = tt + (size_t)tile * TILE_CHUNKS + lane;
            uint4 c_op[2 * KS];
#pragma unroll
            for (int c = 0; c < 2 * KS; ++c) c_op[c] = src[c * 64];
            const float4 n2 = *reinterpret_cast<const float4*>(n2t + tile * 16 + 4 * kb);
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
            for (int j = 0; j < 4; ++j)  // (increasing: ties keep the lower one)
#pragma unroll
                for (int ri = 0; ri < RI; ++ri) {
                    const float v = nn[j] - 2.0f * acc[ri][j];
                    if (v < best[ri]) {
                        best[ri] = v;
                        arg[ri] = tile * 16 + 4 * kb + j;
                    }
                }
        }
#pragma unroll
        for (int ri = 0; ri < RI; ++ri) {
#pragma unroll
            for (int off = 16; off < 64; off <<= 1) {
                const float ob = __shfl_xor(best[ri], off, 64);
                const int og = __shfl_xor(arg[ri], off, 64);
                if (og >= 0 && (arg[ri] < 0 || ob < best[ri] || (ob == best[ri] && og < arg[ri]))) {
                    best[ri] = ob;
                    arg[ri] = og;
                }
            }
            if (kb == 0 && item[ri] >= 0) {
                s.near[item[ri]] = (int16_t)arg[ri];
                s.dist[item[ri]] = fmaxf(best[ri] + x2[ri], 0.0f);
                if (arg[ri] >= 0) atomicAdd(&s.count[arg[ri]], 1);
            }
        }
    }
}

// where the bucket of every centroid begins (K <= kSmallCentroids; one wave)
__device__ __forceinline__ void small_offsets(SmallLds& s, int K) {
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

// the items of bucket k by id, to members[first ..) (one wave)
__device__ __forceinline__ void small_members(SmallLds& s, int k, int first, int m, bool all, int n_items) {
    const int lane = threadIdx.x & 63;
    int found = 0;
    for (int p0 = 0; p0 < n_items && found < m; p0 += 4 * 64) {  // uniform
        int it[4];
        bool in[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int pos = p0 + u * 64 + lane;
            it[u] = pos < n_items ? (all ? pos : (int)s.list[pos]) : -1;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) in[u] = it[u] >= 0 && s.near[max(it[u], 0)] == k;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const unsigned long long bal = __ballot(in[u]);
            if (in[u]) s.members[first + found + __popcll(bal & ((1ull << lane) - 1ull))] = (uint16_t)it[u];
            found += __popcll(bal);
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

// entries of a sequence of n items that satisfy `keep`, in order, to list; returns how many (one wave;
// the sequence may be the list itself)
template <typename Seq, typename Keep>
__device__ __forceinline__ int small_compact(SmallLds& s, int n, Seq seq, Keep keep) {
    const int lane = threadIdx.x & 63;
    int at = 0;
    for (int p0 = 0; p0 < n; p0 += 64) {  // uniform
        const int it = p0 + lane < n ? seq(p0 + lane) : -1;
        const bool in = it >= 0 && keep(max(it, 0));
        const unsigned long long bal = __ballot(in);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        if (in) s.list[at + __popcll(bal & ((1ull << lane) - 1ull))] = (uint16_t)it;
        at += __popcll(bal);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    return at;
}

// wave_mean over 256 threads: their sums over the m rows members[at ..), R rows of D numbers, to part
template <int KS>
__device__ __forceinline__ void small_big_sums(const SmallLds& s, const void* x, size_t row0, int at, int m, float* part) {
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
    constexpr int D = 32 * KS, TILE_CHUNKS = 2 * KS * 64;
    __shared__ SmallLds s;
    const int t = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int bf = p.bf;
    for (int l = p.first; l < p.last; ++l) {  // uniform, and so are the loops over rounds
        const int n_c = p.K[l - 1], K = p.K[l], Kt = p.Kt[l], tiles = (K + 15) / 16;
        const void* x = l == p.first ? p.x : p.cent_t[l - 1];
        const size_t row0 = (size_t)t * n_c;
        int32_t* slots = p.slots[l] + (size_t)t * K * bf;
        const uint4* tt = p.ct.tiles + (size_t)t * Kt * TILE_CHUNKS;
        float* n2t = p.ct.n2 + (size_t)t * Kt * 16;
        float* cent = p.cent + (size_t)t * K * D;
        float* piece = s.piece[wave];

        // ---- empty blocks, first centroids -------------------------------------------------------
        for (int i = tid; i < K * bf; i += kSmallThreads) slots[i] = -1;
        for (int i = tid; i < K; i += kSmallThreads) s.fill[i] = s.count[i] = 0;
        if (tid == 0) s.n_big = 0;
        for (int i = K + tid; i < tiles * 16; i += kSmallThreads) n2t[i] = INFINITY;
        for (int k = wave; k < K; k += kSmallWaves) {
            const size_t src = (row0 + (size_t)first_centroid(p.seed + 7919ull * (uint64_t)l, t, k, n_c, K)) * D;
            for (int j = lane; j < D; j += 64) {
                const float v = load_elem<bf16_t>(x, src + j);
                cent[(size_t)k * D + j] = v;
                piece[j] = v;
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            emit_centroid(piece, D, KS, Kt, t, k, true, p.ct);
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        }
        __syncthreads();

        // ---- Lloyd rounds ------------------------------------------------------------------------
        for (int r = 0; r < p.niter; ++r) {
            small_assign<KS>(s, x, row0, tt, n2t, tiles, true, n_c);
            __syncthreads();
            if (wave == 0) small_offsets(s, K);
            __syncthreads();
            for (int k = wave; k < K; k += kSmallWaves) {
                const int m = __builtin_amdgcn_readfirstlane(s.count[k]), at = __builtin_amdgcn_readfirstlane(s.first[k]);
                if (m == 0) continue;
                small_members(s, k, at, m, true, n_c);
                if (m > 64) {
                    if (lane == 0) s.big[atomicAdd(&s.n_big, 1)] = k;
                    continue;
                }
                wave_mean<bf16_t, 1>(x, row0, [&](int e) { return (uint32_t)s.members[at + e]; }, m, D, piece,
                                     cent + (size_t)k * D);
                emit_centroid(piece, D, KS, Kt, t, k, true, p.ct);
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
                    emit_centroid(part, D, KS, Kt, t, k, true, p.ct);
                    if (lane == 0) s.count[k] = 0;
                }
                __syncthreads();
            }
            if (tid == 0) s.n_big = 0;  // (read by everybody ahead of a barrier: none was passed if there were none)
        }

        // ---- capacity packing: the closest proposers of a bucket (by distance, then id) take the free
        // slots of the block in that order, the others try again ---------------------------------
        auto key_of = [&](uint32_t it) { return ((uint64_t)__float_as_uint(s.dist[it]) << 32) | it; };
        auto filled = [&](int k, int f) {  // (one thread)
            s.count[k] = 0;
            s.fill[k] = f;
            if (f >= bf) n2t[k] = INFINITY;
        };
        int n_items = n_c;
        for (int r = 0; r < p.pack_rounds && n_items > 0; ++r) {
            const bool all = r == 0;
            small_assign<KS>(s, x, row0, tt, n2t, tiles, all, n_items);
            __syncthreads();
            if (wave == 0) small_offsets(s, K);
            __syncthreads();
            for (int k = wave; k < K; k += kSmallWaves) {
                const int m = __builtin_amdgcn_readfirstlane(s.count[k]), at = __builtin_amdgcn_readfirstlane(s.first[k]);
                if (m == 0) continue;
                small_members(s, k, at, m, all, n_items);
                const int f = __builtin_amdgcn_readfirstlane(s.fill[k]), take = max(min(m, bf - f), 0);
                if (m > 64) {
                    for (int e = lane; e < m; e += 64) s.keys[at + e] = key_of(s.members[at + e]);
                    if (lane == 0) s.big[atomicAdd(&s.n_big, 1)] = k;
                    continue;
                }
                const uint64_t mine = lane < m ? key_of(s.members[at + lane]) : ~0ull;
                const int rank = wave_rank(mine, m);
                if (lane < m && rank < take) {
                    slots[k * bf + f + rank] = (int)(uint32_t)mine;
                    s.near[(uint32_t)mine] = kPlaced;
                }
                if (lane == 0) filled(k, f + take);
            }
            __syncthreads();
            const int n_big = __builtin_amdgcn_readfirstlane(s.n_big);
            for (int b = 0; b < n_big; ++b) {  // uniform
                const int k = s.big[b], m = s.count[k], at = s.first[k], f = s.fill[k], take = max(min(m, bf - f), 0);
                for (int e = tid; e < m; e += kSmallThreads) {
                    const uint64_t mine = s.keys[at + e];
                    int rank = 0, j = 0;
                    for (; j + 8 <= m; j += 8)
#pragma unroll
                        for (int u = 0; u < 8; ++u) rank += s.keys[at + j + u] < mine ? 1 : 0;
                    for (; j < m; ++j) rank += s.keys[at + j] < mine ? 1 : 0;
                    if (rank < take) {
                        slots[k * bf + f + rank] = (int)(uint32_t)mine;
                        s.near[(uint32_t)mine] = kPlaced;
                    }
                }
                __syncthreads();
                if (tid == 0) filled(k, f + take);
            }
            if (n_big > 0) __syncthreads();  // uniform
            if (tid == 0) s.n_big = 0;
            if (wave == 0) {
                const int n = small_compact(s, n_items, [&](int i) { return all ? i : (int)s.list[i]; },
                                            [&](int it) { return s.near[it] >= 0; });
                if (lane == 0) s.n_list = n;
            }
            __syncthreads();
            n_items = __builtin_amdgcn_readfirstlane(s.n_list);
        }

        // ---- what is left, and items that are no numbers, to the free slots in order ------------------
        if (wave == 0) {
            const int total = small_compact(s, n_c, [](int i) { return i; }, [&](int it) { return s.near[it] != kPlaced; });
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
                for (int j = 0; j < room && at + j < total; ++j) slots[k * bf + f + j] = s.list[at + j];
                before += __shfl(inc, 63, 64);
            }
        }
        __syncthreads();
        // ---- block centres ----------------------------------------------------------------------------
        for (int k = wave; k < K; k += kSmallWaves)
            wave_block_mean<bf16_t, 2>(x, row0, D, slots + (size_t)k * bf, bf, p.lpr, ((size_t)t * K + k) * D, p.cent, p.cent_t[l]);
        __syncthreads();  // (the next level reads them)
    }
}

int launch_small_levels(const SmallLevels& p, int D, int num_trees, hipStream_t s) {
    switch (D) {
        case 64: hipLaunchKernelGGL((k_small_levels<2>), dim3(num_trees), dim3(kSmallThreads), 0, s, p); break;
        case 128: hipLaunchKernelGGL((k_small_levels<4>), dim3(num_trees), dim3(kSmallThreads), 0, s, p); break;
        case 256: hipLaunchKernelGGL((k_small_levels<8>), dim3(num_trees), dim3(kSmallThreads), 0, s, p); break;
        default: return fail(HIRA_EINVAL, "small levels: %d columns", D);
    }
    return HIRA_OK;
}

}  // namespace hira
