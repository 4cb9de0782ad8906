// What the kernels of the index build share where a level is clustered: the per-bucket kernels of
// build.hip and the one that takes whole small levels (small_levels.hip).  Both have to come to the
// same numbers, bit for bit, whichever of them a level goes through.
#pragma once

#include "rows.h"

namespace hira {

// quantize.hip: the 8-bit shadow of all keys, its steps from the largest magnitudes per channel,
// (T, copies, D)
int quantize_with(const HiraTree* tree, const float* absmax, int copies, hipStream_t s);
constexpr int kAbsCopies = 32;

__device__ __forceinline__ uint64_t mix64(uint64_t z) {
    z += 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

// the item that centroid k of tree t starts from: floor((k + u) * n_t / K_t), u in [0, 1) from the seed;
// a tree uses the first K_t centroids, the others start from an item of the last one's
__device__ __forceinline__ long long first_centroid(uint64_t seed, int t, int k, int n_t, int K_t) {
    const uint64_t h = mix64(seed ^ mix64((uint64_t)t * 0x100000001b3ull + (uint64_t)k));
    const double u = (double)(h >> 11) * (1.0 / 9007199254740992.0);
    const long long idx = (long long)(((double)min(k, K_t - 1) + u) * (double)n_t / (double)K_t);
    return idx >= n_t ? n_t - 1 : idx;
}

// rank of this lane's value among those of lanes 0 .. m - 1 (distinct; the other lanes hold the
// largest number; m uniform in the wave).  Lane numbers are constants: a step is three or four
// instructions.
template <typename Key>
__device__ __forceinline__ int wave_rank(Key mine, int m) {
    int rank = 0;
#pragma unroll
    for (int j0 = 0; j0 < 64; j0 += 8) {
        if (j0 >= m) break;
#pragma unroll
        for (int j = j0; j < j0 + 8; ++j) {
            Key o;
            if constexpr (sizeof(Key) == 8)
                o = ((Key)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(mine >> 32), j) << 32) |
                    (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)mine, j);
            else
                o = (Key)__builtin_amdgcn_readlane((int)mine, j);
            rank += o < mine ? 1 : 0;
        }
    }
    return rank;
}

// Mean of the m > 0 rows row0 + ids(e) of x, by one wave: row e is summed by row group e % R, the R sums
// added in order (a row is CPR = D / EPL threads of 16 bytes, R = 256 / CPR rows at a time: a wave
// stands for 256 threads).  H steps of R rows are in flight.  piece: kWaveMeanPiece numbers of LDS of
// the wave's own, the mean's D numbers lie there at the end; cent_row: where they go.
template <typename T>
constexpr int kWaveMeanPiece = 64 * Elem<T>::kPerChunk;

template <typename T, int H, typename Ids>
__device__ __forceinline__ void wave_mean(const void* x, size_t row0, Ids ids, int m, int D, float* piece,
                                          float* cent_row) {
    constexpr int EPL = Elem<T>::kPerChunk;
    constexpr int kPiece = kWaveMeanPiece<T>;
    const int lane = threadIdx.x & 63;
    const int CPR = D / EPL, R = 256 / CPR;
    float acc[4][EPL];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int q = 0; q < EPL; ++q) acc[i][q] = 0.0f;
    for (int e0 = 0; e0 < m; e0 += H * R) {  // uniform
        uint4 raw[H][4];
#pragma unroll
        for (int h = 0; h < H; ++h)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int v = lane + 64 * i, e = e0 + h * R + v / CPR;
                raw[h][i] = make_uint4(0, 0, 0, 0);
                if (v < R * CPR && e < m)
                    raw[h][i] = load_chunk<T>(x, (row0 + ids(e)) * D, v % CPR);
            }
#pragma unroll
        for (int h = 0; h < H; ++h)
#pragma unroll
            for (int i = 0; i < 4; ++i) {  // (a row that is none adds zeros)
                float f[EPL];
                unpack<T>(raw[h][i], f);
#pragma unroll
                for (int q = 0; q < EPL; ++q) acc[i][q] += f[q];
            }
    }
    // the partial sums as one row of R * D numbers pass through LDS a quarter at a time; a lane
    // adds up its columns
    const int rows = min(R, m);
    if (const int nc = D / 64; D % 64 == 0 && (nc == 1 || nc == 2 || nc == 4)) {  // uniform
        // (64 lanes are whole columns: what a lane reads of a quarter is all on its way together.  Partial sums of
        // rows that are none are zeros, and a sum that began as +0 stays what it is when a zero is added.)
        float sum[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
            for (int q = 0; q < EPL; ++q) piece[lane * EPL + q] = acc[i][q];
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            float v[EPL];
#pragma unroll
            for (int q = 0; q < EPL; ++q) v[q] = piece[lane + 64 * q];
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            if (nc == 1) {
#pragma unroll
                for (int q = 0; q < EPL; ++q) sum[0] += v[q];
            } else if (nc == 2) {
#pragma unroll
                for (int q = 0; q < EPL; ++q) sum[q % 2] += v[q];
            } else {
#pragma unroll
                for (int q = 0; q < EPL; ++q) sum[q % 4] += v[q];
            }
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (u < nc) {
                const float v = sum[u] / (float)m;
                cent_row[lane + 64 * u] = v;
                piece[lane + 64 * u] = v;
            }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        return;
    }
    float sum[8];
    int at[8];  // where the column's next partial sum lies
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        sum[u] = 0.0f;
        at[u] = lane + 64 * u;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int q = 0; q < EPL; ++q) piece[lane * EPL + q] = acc[i][q];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        const int end = min((i + 1) * kPiece, rows * D);
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (64 * u < D)  // uniform
                for (; at[u] < end; at[u] += D) sum[u] += piece[at[u] - i * kPiece];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        const int j = lane + 64 * u;
        if (j < D) {
            const float v = sum[u] / (float)m;
            cent_row[j] = v;
            piece[j] = v;
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

// block centre = mean of the items in the bf slots of the block, rounded to the
// storage type.  One wave: `lpr` lanes (a power of two) hold a row in 16-byte chunks,
// the 64 / lpr lane groups take every (64 / lpr)-th slot, and their sums are added pairwise in a
// fixed order.  An empty block's is its centroid.
// (slot: what lies in slot `lane` of the block, -1 from bf on; U rows a lane group in flight: bf <= 64; B blocks at a
// time, of which there are `have`)
template <typename T, int U, int B>
__device__ __forceinline__ void wave_block_means(const void* x, size_t row0, int D, const int (&slot)[B], int have, int bf,
                                                 int lpr, const size_t (&out)[B], const float* cent, void* out_t) {
    constexpr int EPL = Elem<T>::kPerChunk;
    const int lane = threadIdx.x & 63;
    const int rg = lane / lpr, ch = lane % lpr, groups = 64 / lpr;
    const bool chunk_ok = ch * EPL < D;
    float acc[B][EPL];
    int cnt[B];
#pragma unroll
    for (int b = 0; b < B; ++b) {
        cnt[b] = 0;
#pragma unroll
        for (int q = 0; q < EPL; ++q) acc[b][q] = 0.0f;
    }
    for (int e0 = 0; e0 < bf; e0 += U * groups) {  // uniform: the slots come by shuffles
        int it[B][U];
        uint4 raw[B][U];
#pragma unroll
        for (int b = 0; b < B; ++b)
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int e = e0 + u * groups + rg;
                it[b][u] = __shfl(slot[b], e & 63, 64);
                if (e >= bf) it[b][u] = -1;
                raw[b][u] = load_chunk<T>(x, (row0 + max(it[b][u], 0)) * D, chunk_ok ? ch : 0);
            }
#pragma unroll
        for (int b = 0; b < B; ++b)
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (it[b][u] >= 0) {
                    ++cnt[b];
                    float f[EPL];
                    unpack<T>(raw[b][u], f);
#pragma unroll
                    for (int q = 0; q < EPL; ++q) acc[b][q] += f[q];
                }
    }
#pragma unroll
    for (int b = 0; b < B; ++b) {
        if (b >= have) break;  // uniform
        cnt[b] = cross_group(cnt[b], lpr, OpSum{});
#pragma unroll
        for (int q = 0; q < EPL; ++q) acc[b][q] = cross_group(acc[b][q], lpr, OpSum{});
        if (rg == 0 && chunk_ok) {
            const size_t o = out[b] + ch * EPL;
            if (cnt[b] == 0) {
#pragma unroll
                for (int q = 0; q < EPL; ++q) acc[b][q] = cent[o + q];
            } else {
#pragma unroll
                for (int q = 0; q < EPL; ++q) acc[b][q] = acc[b][q] / (float)cnt[b];
            }
            store_chunk<T>(out_t, o, acc[b]);
        }
    }
}
template <typename T, int U>
__device__ __forceinline__ void wave_block_mean(const void* x, size_t row0, int D, int slot, int bf, int lpr, size_t out,
                                                const float* cent, void* out_t) {
    const int slots[1] = {slot};
    const size_t outs[1] = {out};
    wave_block_means<T, U, 1>(x, row0, D, slots, 1, bf, lpr, outs, cent, out_t);
}

}  // namespace hira
