// Nearest-centroid assignment of the index build on the matrix cores (bf16 rows).
//
// Replaces the distance step of the reference's k-means (faiss.Kmeans.train / index.search,
// indexer/cpu.py:239-250) and of its capacity packing (indexer/cuda.py:247-334):
//   argmin_k ||x_i - c_k||^2 = argmin_k (||c_k||^2 - 2 x_i.c_k),
// with X.C^T on v_mfma_f32_16x16x32_bf16 and the argmin fused into the epilogue, so the
// n x K distance matrix is never written.  Items are bf16 (exact operands).  Centroids are
// fp32 means: each is split into two bf16 numbers, c = hi + lo (16 bits of mantissa), and
// both halves are multiplied, so the distances are as good as fp32 ones for choosing the
// nearest centroid.
//
// k_cent_prep   centroids (T, K, D) fp32 -> operand tiles (assign.h), for hira_nearest; the build's
//               kernels write the tile of a centroid where they make the centroid.
// k_assign_mfma every product with both halves: a workgroup of 4 waves owns 256 items (64 a wave: 4
//               operand tiles kept in registers) and walks all centroid tiles; four tiles at a
//               time are staged once per workgroup in LDS (double buffered, one barrier a stage).
//               Lane (n, kb) of a wave sees the products of its centroid column n with rows 4*kb + j,
//               keeps the best (value, index) per row, and the 16 columns are merged at the end
//               (lowest index on ties).  Over a list of items it can spread them 64 a workgroup,
//               and it can walk the centroids with room only, put side by side by k_open_gather
//               (AssignOpen).
// k_assign_approx  the same choice for a fraction of the products and of the comparisons: all
//               centroids by their `hi` halves alone, then the few that could still be the nearest by
//               the arithmetic of the exact kernel (k_assign_mfma's for its shapes, k_assign_simple's
//               for any other type and width up to 256 columns).
#include "assign.h"

namespace hira {

typedef __attribute__((ext_vector_type(8))) __bf16 abf16x8_t;
typedef __attribute__((ext_vector_type(4))) float af32x4_t;
typedef __attribute__((ext_vector_type(8))) float af32x8_t;

constexpr int kAssignRI = 4;       // operand tiles of 16 items per wave
constexpr int kAssignThreads = 256;
__device__ __forceinline__ bool approx_takes(int n_items, int num_trees) {
    return (long long)n_items * num_trees > kApproxListItems;
}
constexpr int kAssignStage = 4;    // centroid tiles staged together: the time they keep the
                                   // matrix cores busy covers the latency of fetching the next
                                   // four (two for D = 256, whose tiles are twice as large)
constexpr int assign_stage(int KS) { return KS <= 4 ? kAssignStage : kAssignStage / 2; }
// centroids from which on the approximate pass is worth its second launch
constexpr int kApproxMinMfma = 256;
constexpr int kApproxMinSimple = 48;

template <int KS>
__global__ __launch_bounds__(64) void k_cent_prep(const float* cent, int K, const int32_t* fill,
                                                  int bf, uint4* tiles, float* cn2, int Kt) {
    // (Kt counts whole stages of kAssignStage tiles: the tiles past K are zeros with norm +inf)
    constexpr int D = 32 * KS;
    const int lane = threadIdx.x & 63, i = lane & 15, kb = lane >> 4;
    const int tile = blockIdx.x, t = blockIdx.y;
    const int k = tile * 16 + i;
    uint4* out = tiles + ((size_t)t * Kt + tile) * (size_t)(2 * KS * 64);
    float ss = 0.0f;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
        float c[8], ls = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; ++e) c[e] = k < K ? cent[((size_t)t * K + k) * D + s * 32 + kb * 8 + e] : 0.0f;
        uint4 hi, lo;
        split_bf16(c, hi, lo, ss, ls);
        out[s * 64 + kb * 16 + i] = hi;
        out[KS * 64 + s * 64 + kb * 16 + i] = lo;
    }
    ss = cross_group_sum<16>(ss);
    if (kb == 0) {
        const bool usable = k < K && !(fill != nullptr && fill[(size_t)t * K + k] >= bf);
        cn2[((size_t)t * Kt + tile) * 16 + i] = usable ? ss : INFINITY;
    }
}

// ---- every product with both halves, many items: 256 a workgroup --------------------------------
template <int KS>
__global__ __launch_bounds__(kAssignThreads, 2) void k_assign_mfma(const AssignJob job, const int Kt) {
    constexpr int RI = kAssignRI;
    constexpr int D = 32 * KS;
    constexpr int TILE_CHUNKS = 2 * KS * 64;                 // hi and lo halves of 16 centroids
    constexpr int TPS = assign_stage(KS);
    constexpr int STAGE_CHUNKS = TPS * TILE_CHUNKS;
    constexpr int CPT = STAGE_CHUNKS / kAssignThreads;       // chunks a thread stages per stage
    static_assert(STAGE_CHUNKS % kAssignThreads == 0, "stage does not split over the workgroup");
    extern __shared__ uint4 s_dyn[];                         // two stages of tiles, then their norms
    uint4* s_c0 = s_dyn;
    uint4* s_c1 = s_dyn + STAGE_CHUNKS;
    float* s_n2 = reinterpret_cast<float*>(s_dyn + 2 * STAGE_CHUNKS);  // (2, TPS * 16)

    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int n = lane & 15, kb = lane >> 4;  // operand row / centroid column, column block
    const int t = blockIdx.y, n_items = items_of(job, t);
    const int first = (blockIdx.x * (kAssignThreads / 64) + wave) * (RI * 16);
    if (job.counting.zero != nullptr && blockIdx.x == 0 && threadIdx.x == 0) job.counting.zero[t * kCounterStride] = 0;

    // ---- my items: operand tiles in registers, ||x||^2 of row lane % 16 ------------------
    int item[RI];
    uint4 a[RI][KS];
    float x2[RI];
#pragma unroll
    for (int ri = 0; ri < RI; ++ri) {
        const int pos = first + ri * 16 + n;
        item[ri] = pos < n_items ? pos : -1;
        float ss = 0.0f;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            a[ri][s] = make_uint4(0, 0, 0, 0);
            if (item[ri] >= 0)
                a[ri][s] = *reinterpret_cast<const uint4*>(
                    reinterpret_cast<const uint16_t*>(job.x) +
                    ((size_t)t * job.x_tree_stride + item[ri]) * D + s * 32 + kb * 8);
            float f[8];
            unpack<bf16_t>(a[ri][s], f);
#pragma unroll
            for (int e = 0; e < 8; ++e) ss += f[e] * f[e];
        }
        ss = cross_group_sum<16>(ss);
        x2[ri] = ss;
    }
    float best[RI][4];
    int arg[RI][4];
#pragma unroll
    for (int ri = 0; ri < RI; ++ri)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            best[ri][j] = INFINITY;
            arg[ri][j] = -1;
        }

    // ---- all centroid tiles, staged through LDS TPS at a time (the last stage may hold fewer;
    // the arrays are padded to whole stages, their norms with +inf) ---------------------------
    const int Ks = (Kt + TPS - 1) / TPS;
    const uint4* tt = job.ct.tiles + (size_t)t * Ks * STAGE_CHUNKS;
    const float* n2t = job.ct.n2 + (size_t)t * Ks * (TPS * 16);
    uint4 stage[CPT];
    float stage_n2 = 0.0f;
#pragma unroll
    for (int c = 0; c < CPT; ++c) s_c0[threadIdx.x + c * kAssignThreads] = tt[threadIdx.x + c * kAssignThreads];
    if (threadIdx.x < TPS * 16) s_n2[threadIdx.x] = n2t[threadIdx.x];
    __syncthreads();
    for (int st = 0; st < Ks; ++st) {
        const uint4* cbuf = (st & 1) ? s_c1 : s_c0;
        uint4* nbuf = (st & 1) ? s_c0 : s_c1;
        const float* n2buf = s_n2 + (st & 1) * (TPS * 16);
        // the next stage is on its way while this one is used (after the last stage: the last
        // one again, unused; straight-line code keeps `stage` in registers)
        const int nst = min(st + 1, Ks - 1);  // (Ks >= 1 inside the loop)
#pragma unroll
        for (int c = 0; c < CPT; ++c)
            stage[c] = tt[(size_t)nst * STAGE_CHUNKS + threadIdx.x + c * kAssignThreads];
        stage_n2 = n2t[nst * (TPS * 16) + (threadIdx.x & (TPS * 16 - 1))];
#pragma unroll
        for (int ti = 0; ti < TPS; ++ti) {
            abf16x8_t bh[KS], bl[KS];
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                bh[s] = __builtin_bit_cast(abf16x8_t, cbuf[ti * TILE_CHUNKS + s * 64 + lane]);
                bl[s] = __builtin_bit_cast(abf16x8_t, cbuf[ti * TILE_CHUNKS + KS * 64 + s * 64 + lane]);
            }
            const float n2 = n2buf[ti * 16 + n];
            const int kcol = (st * TPS + ti) * 16 + n;
            // four independent accumulator chains: a product never waits for the one before it
            af32x4_t acc[RI];
#pragma unroll
            for (int ri = 0; ri < RI; ++ri) acc[ri] = af32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < KS; ++s) {
#pragma unroll
                for (int ri = 0; ri < RI; ++ri)
                    acc[ri] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        __builtin_bit_cast(abf16x8_t, a[ri][s]), bh[s], acc[ri], 0, 0, 0);
#pragma unroll
                for (int ri = 0; ri < RI; ++ri)
                    acc[ri] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        __builtin_bit_cast(abf16x8_t, a[ri][s]), bl[s], acc[ri], 0, 0, 0);
            }
#pragma unroll
            for (int ri = 0; ri < RI; ++ri)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float v = n2 - 2.0f * acc[ri][j];
                    if (v < best[ri][j]) {  // tiles come in increasing order: ties keep the lower k
                        best[ri][j] = v;
                        arg[ri][j] = kcol;
                    }
                }
        }
#pragma unroll
        for (int c = 0; c < CPT; ++c) nbuf[threadIdx.x + c * kAssignThreads] = stage[c];
        if (threadIdx.x < TPS * 16) s_n2[((st + 1) & 1) * (TPS * 16) + threadIdx.x] = stage_n2;
        __syncthreads();
    }

    // ---- merge the 16 centroid columns of a row group; the wave's 64 results pass through LDS
    // (free behind the loop's last barrier) so that every lane ends up with one item: one store
    // instruction, and one counting instruction, for the whole wave -----------------------------
    static_assert(RI == 4, "a result per lane");
    int* s_g = reinterpret_cast<int*>(s_dyn) + wave * 128;
    float* s_b = reinterpret_cast<float*>(s_g + 64);
#pragma unroll
    for (int ri = 0; ri < RI; ++ri)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            float b = best[ri][j];
            int g = arg[ri][j];
#pragma unroll
            for (int off = 1; off < 16; off <<= 1) {
                const float ob = __shfl_xor(b, off, 64);
                const int og = __shfl_xor(g, off, 64);
                if (og >= 0 && (g < 0 || ob < b || (ob == b && og < g))) {
                    b = ob;
                    g = og;
                }
            }
            if (n == 0) {  // row 4*kb + j of operand tile ri
                s_g[ri * 16 + 4 * kb + j] = g;
                s_b[ri * 16 + 4 * kb + j] = b;
            }
        }
    __builtin_amdgcn_wave_barrier();
    {
        // lane (kb, n) takes row n of operand tile kb: its item and ||x||^2 are its own
        const int g = s_g[lane];
        int it = item[0];
        float xx = x2[0];
#pragma unroll
        for (int ri = 1; ri < RI; ++ri)
            if (kb == ri) {
                it = item[ri];
                xx = x2[ri];
            }
        if (it >= 0) {
            put_result(job, t, it, g, fmaxf(s_b[lane] + xx, 0.0f));
        }
    }
}

// ---- every product with both halves, few items: 64 a wave, or a few waves -----------------------
// Lists (the packing's, or what the approximate pass leaves) and small levels leave most of the chip
// idle if 256 items go together.  Here a wave holds 64 items and walks the tiles straight from memory to
// registers, the next one on its way while one is used; `share` waves of the workgroup hold the same items
// and walk every share-th tile, as many as there are waves for on the chip (split_share).  Centroids are the rows of a
// product, so a lane's results are four centroids of one item per item tile, and what is left at the
// end is a minimum over four lanes and `share` waves.
// What bounds it is the chain items, tiles, bucket, and for long lists the matrix cores.  Eight waves to 64 items
// whatever their number: a workgroup's items and its end were most of its time where lists are long and
// centroids few (8 x 7200 items, 330 centroids: 40 us, now 24; 8 x 8300, 330: 58, now 48); one wave to
// 64 items whatever their number: 8 x ~1000 items, 1024 centroids 52 us, now 9.
constexpr int kSplitThreads = 512;
// Workgroups of a tree, at most (they go through a list in strides): those of all trees fill the chip twice.  (128
// whatever the trees: builds of 1 x 100000 rows of 64 columns in three levels at a fan-out of 16 779 us, now 724, at 32 551 / 514.)
constexpr int split_blocks(int KS, int trees) {
    const int all = KS <= 2 ? 1024 : 512;
    return all / 16 < trees ? 16 : all / trees;
}
constexpr int kSplitWavesLog2 = 11;      // of the waves on the chip at a time: 256 compute units, 8 each
static_assert(kSplitThreads == 64 << 3, "split_share_log2");

constexpr int split_ri(int KS) { return KS <= 4 ? 4 : 2; }

// Waves that share a set of items, of which each of `trees` trees has `sets` (as a power of two): the number
// whose rounds of waves take least, a wave's items and its end as long as kSplitFixed tiles.
template <int KS>
__device__ __forceinline__ int split_share_log2(int sets, int trees, int tiles) {
    constexpr int kSplitFixed = 48 / KS, on_chip_log2 = KS <= 2 ? kSplitWavesLog2 + 1 : kSplitWavesLog2;
    int best = 0;
    long long least = 0;
#pragma unroll
    for (int s = 0; s <= 3; ++s) {
        const long long rounds = (((long long)sets * trees << s) + (1 << on_chip_log2) - 1) >> on_chip_log2;
        const long long cost = rounds * (kSplitFixed + ((tiles + (1 << s) - 1) >> s));
        if (s == 0 || cost < least) {
            best = s;
            least = cost;
        }
    }
    return best;
}

template <int KS>
__device__ __forceinline__ void split_items(const AssignJob& job, int Kt, int tiles, const int32_t* list, int n_items, int share_log2, int block) {
    constexpr int D = 32 * KS, RI = split_ri(KS), ITEMS = RI * 16, WAVES = kSplitThreads / 64;
    constexpr int TILE_CHUNKS = 2 * KS * 64;
    __shared__ float s_b[WAVES][ITEMS];
    __shared__ int s_g[WAVES][ITEMS];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n = lane & 15, kb = lane >> 4;
    const int t = blockIdx.x, n_c = job.n_c, K = job.K;

    // ---- the first tile of the wave, and the items ---------------------------------------------
    const uint4* tt = job.ct.tiles + (size_t)t * Kt * TILE_CHUNKS + lane;
    const float* n2t = job.ct.n2 + (size_t)t * Kt * 16 + 4 * kb;
    const int share = 1 << share_log2;
    const int set = block * (WAVES >> share_log2) + (wave >> share_log2), part = wave & (share - 1);
    uint4 c[2][2 * KS];
    float4 c2[2];
    auto fetch = [&](int tile, uint4 (&to)[2 * KS], float4& n2) {
        const uint4* src = tt + (size_t)tile * TILE_CHUNKS;
#pragma unroll
        for (int s = 0; s < 2 * KS; ++s) to[s] = src[s * 64];
        n2 = *reinterpret_cast<const float4*>(n2t + tile * 16);
        __builtin_amdgcn_sched_barrier(0);  // (asked for here, not where the first product wants it)
    };
    fetch(min(part, Kt - 1), c[0], c2[0]);
    int item[RI];
    uint4 x[RI][KS];
    float x2[RI];
#pragma unroll
    for (int ri = 0; ri < RI; ++ri) {
        const int pos = set * ITEMS + ri * 16 + n, at = min(pos, n_items - 1);  // (n_items > 0)
        item[ri] = list ? list[(size_t)t * n_c + at] : at;
        if (pos >= n_items) item[ri] = -1;
    }
#pragma unroll
    for (int ri = 0; ri < RI; ++ri)
#pragma unroll
        for (int s = 0; s < KS; ++s)
            x[ri][s] = *reinterpret_cast<const uint4*>(
                reinterpret_cast<const uint16_t*>(job.x) +
                ((size_t)t * job.x_tree_stride + max(item[ri], 0)) * D + s * 32 + kb * 8);
#pragma unroll
    for (int ri = 0; ri < RI; ++ri) {
        float ss = 0.0f;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            float f[8];
            unpack<bf16_t>(x[ri][s], f);
#pragma unroll
            for (int e = 0; e < 8; ++e) ss += f[e] * f[e];
        }
        ss = cross_group_sum<16>(ss);
        x2[ri] = ss;
    }
    float best[RI];
    int arg[RI];
#pragma unroll
    for (int ri = 0; ri < RI; ++ri) {
        best[ri] = INFINITY;
        arg[ri] = -1;
    }
    auto use = [&](int tile, const uint4 (&ct)[2 * KS], const float4& n2) {
        af32x4_t acc[RI];
#pragma unroll
        for (int ri = 0; ri < RI; ++ri) acc[ri] = af32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < KS; ++s)
#pragma unroll
            for (int half = 0; half < 2; ++half)
#pragma unroll
                for (int ri = 0; ri < RI; ++ri)
                    acc[ri] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(abf16x8_t, ct[half * KS + s]),
                                                                      __builtin_bit_cast(abf16x8_t, x[ri][s]), acc[ri], 0, 0, 0);
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
    };
    int tile = set * ITEMS < n_items ? part : tiles;  // (a wave without items walks none)
    for (; tile + share < tiles; tile += 2 * share) {  // uniform in the wave; no barrier inside
        fetch(tile + share, c[1], c2[1]);
        use(tile, c[0], c2[0]);
        fetch(min(tile + 2 * share, Kt - 1), c[0], c2[0]);
        use(tile + share, c[1], c2[1]);
    }
    if (tile < tiles) use(tile, c[0], c2[0]);

    // ---- one of the four lanes, then of the waves, of an item ------------------------------------
    auto better = [](float b, int g, float ob, int og) { return og >= 0 && (g < 0 || ob < b || (ob == b && og < g)); };
#pragma unroll
    for (int ri = 0; ri < RI; ++ri) {
        auto nearer = [&](auto v, auto k) {  // of the two lanes that a swap has paired, in both of them
            const float v0 = __uint_as_float((uint32_t)v[0]), v1 = __uint_as_float((uint32_t)v[1]);
            const int k0 = (int)k[0], k1 = (int)k[1];
            const bool second = better(v0, k0, v1, k1);
            best[ri] = second ? v1 : v0;
            arg[ri] = second ? k1 : k0;
        };
        nearer(__builtin_amdgcn_permlane16_swap(__float_as_uint(best[ri]), __float_as_uint(best[ri]), false, false),
               __builtin_amdgcn_permlane16_swap((uint32_t)arg[ri], (uint32_t)arg[ri], false, false));
        nearer(__builtin_amdgcn_permlane32_swap(__float_as_uint(best[ri]), __float_as_uint(best[ri]), false, false),
               __builtin_amdgcn_permlane32_swap((uint32_t)arg[ri], (uint32_t)arg[ri], false, false));
        if (kb == 0) {
            s_b[wave][ri * 16 + n] = best[ri];
            s_g[wave][ri * 16 + n] = arg[ri];
        }
    }
    __syncthreads();
    if (part != 0 || lane >= ITEMS) return;
    // lane (kb, n) takes item n of tile kb
    float b = s_b[wave][lane];
    int g = s_g[wave][lane];
    for (int w = wave + 1; w < wave + share; ++w)  // uniform
        if (better(b, g, s_b[w][lane], s_g[w][lane])) {
            b = s_b[w][lane];
            g = s_g[w][lane];
        }
    int it = item[0];
    float xx = x2[0];
#pragma unroll
    for (int ri = 1; ri < RI; ++ri)
        if (kb == ri) {
            it = item[ri];
            xx = x2[ri];
        }
    if (it < 0) return;
    if (job.open.ids != nullptr && g >= 0) g = job.open.ids[(size_t)t * K + g];  // column -> centroid
    put_result(job, t, it, g, fmaxf(b + xx, 0.0f));
}

// The kernel's arguments (the job, and Kt behind it) lie in five 64-byte lines of memory: all of them asked for at once (touch_kernel_arguments of search.h).
// Builds, with the lanes of an item meeting by swaps: 8 x 4001 keys 186.3 -> 183.8 us, 2 x 1111 x 64 in five levels 150.5 -> 148.2.
__device__ __forceinline__ void touch_job() {
    static_assert(sizeof(AssignJob) + sizeof(int) > 4 * 64 && sizeof(AssignJob) + sizeof(int) <= 5 * 64, "one load per 64-byte line of the arguments");
    auto ka = __builtin_amdgcn_kernarg_segment_ptr();
    uint32_t d0, d1, d2, d3, d4;
    asm volatile(
        "s_load_dword %0, %5, 0x0\n\t"
        "s_load_dword %1, %5, 0x40\n\t"
        "s_load_dword %2, %5, 0x80\n\t"
        "s_load_dword %3, %5, 0xc0\n\t"
        "s_load_dword %4, %5, 0x100\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&s"(d0), "=&s"(d1), "=&s"(d2), "=&s"(d3), "=&s"(d4)
        : "s"(ka)
        : "memory");
}
template <int KS>
__global__ __launch_bounds__(kSplitThreads, 2) void k_assign_split(const AssignJob job, const int Kt) {
    touch_job();
    const int t = blockIdx.x;
    const int32_t* list = job.list;
    int n_items = items_of(job, t);
    if (job.after_approx && (list == nullptr || approx_takes(n_items, gridDim.x))) {
        list = job.unsure;
        n_items = job.unsure_count[t * kCounterStride];
    }
    if (job.counting.zero != nullptr && blockIdx.y == 0 && threadIdx.x == 0) job.counting.zero[t * kCounterStride] = 0;
    constexpr int ITEMS = split_ri(KS) * 16;
    const int tiles = job.open.count ? min((job.open.count[t] + 15) / 16, Kt) : (job.K + 15) / 16;
    const int sets = (n_items + ITEMS - 1) / ITEMS, share_log2 = split_share_log2<KS>(sets, gridDim.x, tiles);
    for (int b = blockIdx.y; b * (kSplitThreads / 64 >> share_log2) < sets; b += gridDim.y) {  // uniform
        if (b != (int)blockIdx.y) __syncthreads();  // (the results of the stride before are out of LDS)
        split_items<KS>(job, Kt, tiles, list, n_items, share_log2, b);
    }
}

// ---- the approximate pass -------------------------------------------------------------------
// score_k = x.c_k - ||c_k||^2 / 2; the nearest centroid has the largest.  With x = xh + xl (bf16 and
// rest; xl = 0 for bf16 items) and c = hi + rest:
//   |x.c - xh.hi| <= ||x|| lo_k + ||xl|| ||c_k||      (lo_k: assign.h, rounding of the sums included)
// so the products with `hi` alone, started from  -||c_k||^2 / 2 + X lo_k + Xl ||c_k||  (X, Xl: the
// largest norms among the workgroup's items), are never below the exact score, and above it by at most
// twice that allowance.  A lane keeps its best and second best of them per item and
// class of tiles, the centroid's number in the low bits of the value (one instruction, against a comparison
// and two selections that a separate index takes; what the bits shift the value by counts as error).  Per item
// the lower bound of the largest decides who is still in the running: of the four lanes that share the item, and
// their bests, those that reach it.  One candidate: that is the nearest.  Several: each is scored by the
// exact kernel's own arithmetic, and the smallest distance wins, the lowest centroid on ties -- the exact kernel's
// result bit for bit.  Where a SECOND best is in the running too, a third could be as well, which
// nobody noted: such items (about 1 % on normal keys) go on a list that the exact kernel takes.
// Operands: centroids are the rows (A), items the columns (B): a lane's four results of a product are
// four centroids of ONE item, so best and second are one pair per item tile instead of four, and the
// start values are a 16-byte read from LDS.
// What bounds it is the matrix cores: 8 x 131072 items x 4096 centroids take 1690-1740 us with the
// exact kernel and 875 us with this one, 950 us where the distances are asked for; 8 x 32768 x 1024:
// 165 -> 80 / 89 us.  Of a workgroup's 102 / 111 us its walk of the tiles takes 90 (1.5 PFLOP/s; a large
// matrix product reaches 1.6 on this card), its items 6, its end 6 / 12.  (930 / 1060 us with a barrier every
// 64 products of a wave and an end that looked rows up in operand tiles.)
constexpr float kNoScore = -1e37f;  // start value of a centroid that takes no items
constexpr int kMaxTagBits = 14;     // centroid numbers inside a lane: Kt * 4 of them

// 16 bytes of every lane straight from memory to LDS: lane i's to dst + i (dst: the wave's)
__device__ __forceinline__ void load_to_lds(const uint4* src, uint4* dst) {
    __builtin_amdgcn_global_load_lds(reinterpret_cast<const __attribute__((address_space(1))) void*>(
                                         reinterpret_cast<uintptr_t>(src)),
                                     (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
}
// (ahead of the barrier behind which the others read them)
__device__ __forceinline__ void arrived_in_lds() {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
}

// columns [c0, c0 + 8) of a row: what `raw` holds of them (zeros where there is nothing) as an operand chunk,
// and the sums of squares of the row and of what bf16 drops
template <typename T>
__device__ __forceinline__ void approx_row(const uint4 (&raw)[8 / Elem<T>::kPerChunk], uint4& packed, float& x2, float& l2) {
    constexpr int EPL = Elem<T>::kPerChunk;
    float f[8];
#pragma unroll
    for (int h = 0; h < 8 / EPL; ++h) {
        float g[EPL];
        unpack<T>(raw[h], g);
#pragma unroll
        for (int e = 0; e < EPL; ++e) f[h * EPL + e] = g[e];
        if (EPL == 8) packed = raw[h];
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) x2 += f[e] * f[e];
    if (EPL == 4) {
        packed = make_uint4(pack_bf16(f[0], f[1]), pack_bf16(f[2], f[3]), pack_bf16(f[4], f[5]), pack_bf16(f[6], f[7]));
        float h[8];
        unpack<bf16_t>(packed, h);
#pragma unroll
        for (int e = 0; e < 8; ++e) l2 += (f[e] - h[e]) * (f[e] - h[e]);
    }
}

// a float as an unsigned number of the same order
__device__ __forceinline__ uint32_t ordered_bits(float v) {
    const uint32_t u = __float_as_uint(v);
    return u ^ ((u >> 31) ? 0xffffffffu : 0x80000000u);
}
__device__ __forceinline__ float from_ordered(uint32_t u) {
    return __uint_as_float(u ^ ((u >> 31) ? 0x80000000u : 0xffffffffu));
}

constexpr int kApproxThreads = 256;
// Tiles of a stage: two of the stages that the tiles are padded to.  (A barrier every 64 products of a wave
// had the matrix cores wait a third of the time; eight waves a workgroup instead of four were no better.)
constexpr int approx_stage(int KS) { return 2 * assign_stage(KS); }
// Classes of tiles (by number) that a lane keeps a best and a second best of: the more, the fewer items of which
// two candidates share a class.  (Two classes instead of four: twice the items the exact kernel has to take,
// 109 us for it instead of 58 after the packing's full pass over 8 x 131072 items.)
constexpr int kApproxClasses = 4;
constexpr int kApproxPairs = 64 * 4 * kApproxClasses;  // (item, candidate) pairs of a wave, at most

template <typename T, int KS, int RI, bool LISTED, bool EXACT_MFMA>
__device__ __forceinline__ void approx_items(const AssignJob& job, int Kt, int tag_bits, int n_items, int block) {
    constexpr int HALF = KS * 64;                       // chunks of the hi half of 16 centroids
    constexpr int TILE_CHUNKS = 2 * HALF;
    constexpr int TPS = approx_stage(KS);
    constexpr int STAGE = TPS * HALF;
    constexpr int CPT = STAGE / kApproxThreads;
    constexpr int ITEMS = RI * 16;                      // of a wave
    constexpr int WAVES = kApproxThreads / 64, CLS = kApproxClasses;
    constexpr bool SPLIT = sizeof(T) == 4;              // items lose something in bf16
    static_assert(STAGE % kApproxThreads == 0, "stage does not split over the workgroup");
    extern __shared__ uint4 s_dyn[];
    uint4* s_c = s_dyn;                                             // (2, STAGE)
    float* s_start = reinterpret_cast<float*>(s_dyn + 2 * STAGE);   // (2, TPS * 16)
    float* s_x = s_start + 2 * TPS * 16;                            // (2, waves): largest norms

    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wave_u = __builtin_amdgcn_readfirstlane(wave);
    const int n = lane & 15, kb = lane >> 4;
    const int t = blockIdx.x, n_c = job.n_c, K = job.K;
    const int first = (block * (kApproxThreads / 64) + wave) * ITEMS;

    // ---- the first stage of tiles: on its way while the items come ---------------------------------
    // (whole stages of assign_stage(KS) tiles are there; the walk's last stage may have no second half: it
    // takes a tile there is, whose centroids take no items)
    const int tiles = job.open.count ? min(((job.open.count[t] + 15) / 16 + TPS / 2 - 1) / (TPS / 2) * (TPS / 2), Kt) : Kt;
    const int Ks = (tiles + TPS - 1) / TPS;
    const uint4* tt = job.ct.tiles + (size_t)t * Kt * TILE_CHUNKS;
    const float* n2t = job.ct.n2 + (size_t)t * Kt * 16;
    const float* lot = job.ct.lo + (size_t)t * Kt * 16;
    const int q = threadIdx.x & (TPS * 16 - 1);
    // (of a tile only the hi half is fetched)
    auto fetch = [&](int st, int buf) {
        const int last = tiles - 1 - st * TPS;  // of the stage
#pragma unroll
        for (int c = 0; c < CPT; ++c) {
            constexpr int PER = HALF / kApproxThreads;  // steps of the workgroup a tile (0: several tiles a step)
            const int ci = c * kApproxThreads + (int)threadIdx.x;
            const int tile = PER > 0 ? c / max(PER, 1) : ci / HALF;
            const uint4* src = tt + (size_t)(st * TPS + min(tile, last)) * TILE_CHUNKS + ci % HALF;
            load_to_lds(src, s_c + buf * STAGE + c * kApproxThreads + wave_u * 64);
        }
    };
    auto norms_at = [&](int st) { return min(st * (TPS * 16) + q, tiles * 16 - 1); };
    float first_n2 = 0.0f, first_lo = 0.0f;
    if (Ks > 0) {
        fetch(0, 0);
        first_n2 = n2t[norms_at(0)];
        first_lo = lot[norms_at(0)];
    }
    // ---- my items ----------------------------------------------------------------------------
    int item[RI];
    uint4 b[RI][KS];
    float x2[RI];
    float X = 0.0f, Xl = 0.0f;
#pragma unroll
    for (int ri = 0; ri < RI; ++ri) {
        const int pos = first + ri * 16 + n;
        item[ri] = -1;
        const int at = min(pos, n_items - 1);  // (n_items > 0: the workgroup has work)
        item[ri] = LISTED ? job.list[(size_t)t * n_c + at] : at;
        if (pos >= n_items) item[ri] = -1;
    }
    constexpr int EPL = Elem<T>::kPerChunk;
    auto norms = [&](int ri, float ss, float ls) {  // (of this lane's columns)
        ss = cross_group_sum<16>(ss);
        x2[ri] = ss;
        X = fmaxf(X, ss);
        if (SPLIT) {
            ls = cross_group_sum<16>(ls);
            Xl = fmaxf(Xl, ls);
        }
    };
    if constexpr (EXACT_MFMA) {
        // whole operands: all rows on their way under no condition (a load under one is waited for where
        // the condition ends, one item tile after the other)
        uint4 raw[RI][KS][1];
#pragma unroll
        for (int ri = 0; ri < RI; ++ri)
#pragma unroll
            for (int s = 0; s < KS; ++s)
                raw[ri][s][0] = load_chunk<T>(job.x, ((size_t)t * job.x_tree_stride + max(item[ri], 0)) * (32 * KS), s * 4 + kb);
#pragma unroll
        for (int ri = 0; ri < RI; ++ri) {
            float ss = 0.0f, ls = 0.0f;
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                if (item[ri] < 0) raw[ri][s][0] = make_uint4(0, 0, 0, 0);
                approx_row<T>(raw[ri][s], b[ri][s], ss, ls);
            }
            norms(ri, ss, ls);
        }
    } else {
#pragma unroll
        for (int ri = 0; ri < RI; ++ri) {
            float ss = 0.0f, ls = 0.0f;
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                const int c0 = s * 32 + kb * 8;
                uint4 raw[8 / EPL];
#pragma unroll
                for (int h = 0; h < 8 / EPL; ++h) {
                    raw[h] = make_uint4(0, 0, 0, 0);
                    if (item[ri] >= 0 && c0 + h * EPL < job.D)
                        raw[h] = load_chunk<T>(job.x, ((size_t)t * job.x_tree_stride + item[ri]) * job.D, c0 / EPL + h);
                }
                approx_row<T>(raw, b[ri][s], ss, ls);
            }
            norms(ri, ss, ls);
        }
    }
    X = lanes_fold<1, 16>(X, OpMax{});
    if (SPLIT) Xl = lanes_fold<1, 16>(Xl, OpMax{});
    if (lane == 0) {
        s_x[wave] = X;
        s_x[WAVES + wave] = Xl;
    }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
        X = fmaxf(X, s_x[w]);
        if (SPLIT) Xl = fmaxf(Xl, s_x[WAVES + w]);
    }
    X = sqrtf(X) * 1.0001f;
    if (SPLIT) {
        Xl = sqrtf(Xl) * 1.0001f;
    }

    auto put_start = [&](int st, int buf, float n2, float lo) {
        // (1e-5 of the squared norm: what the rounding of the norm can be worth)
        float v = fmaf(X, lo, -0.5f * n2 + 1e-5f * n2);
        if (SPLIT) v = fmaf(Xl, sqrtf(n2), v);
        if (!(n2 < INFINITY) || st * TPS * 16 + q >= tiles * 16) v = kNoScore;
        s_start[buf * TPS * 16 + q] = v;  // (the same by every wave that has the column: no branch)
    };

    float best[CLS][RI], second[CLS][RI];  // of the tiles 0, CLS, 2 CLS, ..., of 1, CLS + 1, ..., ...
#pragma unroll
    for (int ri = 0; ri < RI; ++ri)
#pragma unroll
        for (int e = 0; e < CLS; ++e) best[e][ri] = second[e][ri] = -INFINITY;
    const uint32_t keep = ~((1u << tag_bits) - 1u);

    // ---- all centroid tiles --------------------------------------------------------------------
    if (Ks > 0) put_start(0, 0, first_n2, first_lo);
    arrived_in_lds();
    // The results of a tile are looked at while the next tile's products are made: a product keeps the
    // matrix cores busy for the time of four vector instructions, three of which deal with a result.
    // The order is the one written here (left to itself the compiler makes all products of a stage
    // first and looks at all results behind them: 1.3 ms instead of 0.9 at 8 x 131072 x 4096).
    af32x4_t acc[2][RI];
#pragma unroll
    for (int ri = 0; ri < RI; ++ri) acc[1][ri] = af32x4_t{-3e38f, -3e38f, -3e38f, -3e38f};
    uint32_t keep_v;  // (in a vector register: with `tag` in a scalar one the bits are one instruction)
    asm volatile("v_mov_b32 %0, %1" : "=v"(keep_v) : "s"(keep));
    // The four results of an item tile in LOOKS steps: tagged, then two at a time into best and second.  With
    // best >= second the two largest of {best, second, u, v} are max3(best, u, v) and
    // max(med3(best, u, v), second), and the maxima of `second` of both pairs are one instruction.
    // (Asm: fmaxf quiets its operands first, an instruction each.)
    constexpr int LOOKS = 8, PRODUCTS = KS * RI, RESULTS = LOOKS * RI;
    float m3[RI];
    auto look = [&](int of, int cls, uint32_t tag, int o) {
        const int ri = o / LOOKS, k = o % LOOKS;
        float(&r)[RI] = best[cls];
        auto tagged = [&](int j) { acc[of][ri][j] = __uint_as_float((__float_as_uint(acc[of][ri][j]) & keep_v) | (tag + j)); };
        auto max3 = [](float& a, float u, float v) { asm("v_max3_f32 %0, %0, %1, %2" : "+v"(a) : "v"(u), "v"(v)); };
        if (k == 0) tagged(0);
        if (k == 1) tagged(1);
        if (k == 2) m3[ri] = __builtin_amdgcn_fmed3f(r[ri], acc[of][ri][0], acc[of][ri][1]);
        if (k == 3) max3(r[ri], acc[of][ri][0], acc[of][ri][1]);
        if (k == 4) tagged(2);
        if (k == 5) tagged(3);
        if (k == 6) {
            const float m = __builtin_amdgcn_fmed3f(r[ri], acc[of][ri][2], acc[of][ri][3]);
            max3(second[cls][ri], m3[ri], m);
        }
        if (k == 7) max3(r[ri], acc[of][ri][2], acc[of][ri][3]);
    };
    for (int st = 0; st < Ks; ++st) {
        const int buf = st & 1;
        const uint4* cbuf = s_c + buf * STAGE + lane;
        const float* sbuf = s_start + buf * TPS * 16 + 4 * kb;
        const int nst = min(st + 1, Ks - 1);
        const float next_n2 = n2t[norms_at(nst)], next_lo = lot[norms_at(nst)];
        fetch(nst, buf ^ 1);
        abf16x8_t a[2][KS];
        af32x4_t start[2];
#pragma unroll
        for (int s = 0; s < KS; ++s) a[0][s] = __builtin_bit_cast(abf16x8_t, cbuf[s * 64]);
        start[0] = *reinterpret_cast<const af32x4_t*>(sbuf);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int ti = 0; ti < TPS; ++ti) {
            const int me = ti & 1;
            const uint32_t tag = (uint32_t)max(st * TPS + ti - 1, 0) * 4u;  // of the tile before
#pragma unroll
            for (int p = 0; p < PRODUCTS; ++p) {
                const int s = p / RI, ri = p % RI;
                acc[me][ri] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    a[me][s], __builtin_bit_cast(abf16x8_t, b[ri][s]), s == 0 ? start[me] : acc[me][ri], 0, 0, 0);
#pragma unroll
                for (int o = p * RESULTS / PRODUCTS; o < (p + 1) * RESULTS / PRODUCTS; ++o) look(me ^ 1, (ti + CLS - 1) % CLS, tag, o);
                if (p == 1 && ti + 1 < TPS) {  // the next tile's operands
#pragma unroll
                    for (int s2 = 0; s2 < KS; ++s2)
                        a[me ^ 1][s2] = __builtin_bit_cast(abf16x8_t, cbuf[(ti + 1) * HALF + s2 * 64]);
                    start[me ^ 1] = *reinterpret_cast<const af32x4_t*>(sbuf + (ti + 1) * 16);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        put_start(nst, buf ^ 1, next_n2, next_lo);
        arrived_in_lds();
    }
    if (Ks > 0) {
        static_assert(TPS % 2 == 0 && TPS % CLS == 0, "the last tile's results are in acc[1]");
#pragma unroll
        for (int o = 0; o < RESULTS; ++o) look(1, CLS - 1, (uint32_t)(Ks * TPS - 1) * 4u, o);
    }

    // ---- who is still in the running (LDS is free behind the loop's last barrier) -------------------
    const bool want_dist = job.counting.dists != nullptr;  // uniform: then every item's distance is needed
    constexpr int WAVE_BYTES = 64 * 8 + kApproxPairs * 8;
    char* mine = reinterpret_cast<char*>(s_dyn) + wave * WAVE_BYTES;
    unsigned long long* s_key = reinterpret_cast<unsigned long long*>(mine);  // (64) best (distance, column)
    int* s_item = reinterpret_cast<int*>(mine + 64 * 8);                      // pairs: item of the wave
    int* s_col = s_item + kApproxPairs;                                       //        column
    const float shift = ldexpf(1.0f, tag_bits - 23);
    s_key[lane] = ~0ull;
    int npairs = 0;      // uniform in the wave
    bool unsure[RI];
    int top[RI];         // the column with the largest value among the item's lanes
    bool scored[RI];     // its exact distance is needed, and those of the others in the running
    unsigned long long ask = 0;  // (uniform) not zero: some are
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    // The largest value among the item's lanes, less what it can be too large by, is what the exact score of
    // the nearest reaches at least.  (One lookup an item, for all item tiles at once: a lookup of every lane's
    // own two columns is 64 lines of memory a load, 4.4 us at the end of a workgroup's 106.)
    int col[CLS][RI];
    float top_v[RI], top_n2[RI], top_lo[RI];
#pragma unroll
    for (int ri = 0; ri < RI; ++ri) {
        float tv = -INFINITY;
        int tc = Kt * 16 - 1;
#pragma unroll
        for (int e = 0; e < CLS; ++e) {  // (a value that is no number holds any tag, and is none of the largest)
            const uint32_t tag = __float_as_uint(best[e][ri]) & ~keep;
            col[e][ri] = min((int)(tag >> 2) * 16 + 4 * kb + (int)(tag & 3u), Kt * 16 - 1);
            if (best[e][ri] > 0.5f * kNoScore && best[e][ri] > tv) {
                tv = best[e][ri];
                tc = col[e][ri];
            }
        }
#pragma unroll
        for (int off = 16; off < 64; off <<= 1) {
            const float ov = __shfl_xor(tv, off, 64);
            const int oc = __shfl_xor(tc, off, 64);
            if (ov > tv || (ov == tv && oc < tc)) {
                tv = ov;
                tc = oc;
            }
        }
        top_v[ri] = tv;
        top[ri] = tc;
        top_n2[ri] = n2t[tc];
        top_lo[ri] = lot[tc];
    }
#pragma unroll
    for (int ri = 0; ri < RI; ++ri) {
        const bool have = item[ri] >= 0 && top_v[ri] > 0.5f * kNoScore;
        float off = 2.0f * (X * top_lo[ri] + 1e-5f * top_n2[ri]);
        if (SPLIT) off += 2.0f * Xl * sqrtf(top_n2[ri]);
        if (!EXACT_MFMA) off += 1e-5f * X * X;  // (rounding of sums of squared differences)
        const float floor_of = top_v[ri] - off - fabsf(top_v[ri]) * shift;
        bool in[CLS];
        int un = 0, cands = 0;
#pragma unroll
        for (int e = 0; e < CLS; ++e) {
            const bool any = have && best[e][ri] > 0.5f * kNoScore;  // (not a number: no)
            in[e] = any && best[e][ri] + fabsf(best[e][ri]) * shift >= floor_of;
            // (a value next to zero does not hold its tag)
            un |= any && (!(second[e][ri] + fabsf(second[e][ri]) * shift < floor_of) || fabsf(best[e][ri]) < 1e-30f);
            cands += in[e];
        }
        un |= __shfl_xor(un, 16, 64);
        un |= __shfl_xor(un, 32, 64);
        cands += __shfl_xor(cands, 16, 64);
        cands += __shfl_xor(cands, 32, 64);
        un |= cands == 0;  // (rows with numbers that are none: as the exact kernel has it)
        unsure[ri] = un;
        scored[ri] = !un && (want_dist || cands > 1);
        ask |= __ballot(scored[ri]);
        if (!un && !scored[ri] && kb == 0) s_key[ri * 16 + n] = (unsigned long long)(uint32_t)top[ri];  // (the only one)
#pragma unroll
        for (int e = 0; e < CLS; ++e) {
            const bool score = in[e] && scored[ri] && !(EXACT_MFMA && col[e][ri] == top[ri]);
            const unsigned long long bal = __ballot(score);
            if (score) {
                const int at = npairs + __popcll(bal & ((1ull << lane) - 1ull));
                s_item[at] = ri * 16 + n;
                s_col[at] = col[e][ri];
            }
            npairs += __popcll(bal);
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");

    // ---- the candidates' exact distances ---------------------------------------------------------
    if constexpr (EXACT_MFMA) {
        // Row i of the A operand is a centroid, column i of B an item, the result on the diagonal; the
        // products in the exact kernel's order.  First the largest of every item, whose operands are still in
        // registers: the centroids' rows of all item tiles are asked for at once.  Then the others,
        // sixteen pairs at a time.  The rows come from the fp32 centroids and are split here as emit_centroid
        // splits them: sixteen lines of memory a load.  (Out of sixteen operand tiles they are 64, and the end of
        // a workgroup that asks for distances took 9.3 of its 125 us.)
        auto cent_row = [&](int c) {
            const int k = job.open.ids != nullptr ? job.open.ids[(size_t)t * K + c] : c;  // column -> centroid
            return reinterpret_cast<const uint4*>(job.cent + ((size_t)t * K + k) * (32 * KS) + kb * 8);
        };
        auto halves = [](const uint4& lo4, const uint4& hi4, abf16x8_t& h, abf16x8_t& l) {
            const af32x8_t v = {__uint_as_float(lo4.x), __uint_as_float(lo4.y), __uint_as_float(lo4.z), __uint_as_float(lo4.w),
                                __uint_as_float(hi4.x), __uint_as_float(hi4.y), __uint_as_float(hi4.z), __uint_as_float(hi4.w)};
            h = __builtin_convertvector(v, abf16x8_t);
            l = __builtin_convertvector(v - __builtin_convertvector(h, af32x8_t), abf16x8_t);
        };
        auto put_diagonal = [&](const af32x4_t& d4, float n2, int c, int it_local, bool have) {
            if (kb == (n >> 2) && have) {  // row n = 4 * kb + j of column n
                const int j = n & 3;
                const float d = j == 0 ? d4[0] : j == 1 ? d4[1] : j == 2 ? d4[2] : d4[3];
                const float v = n2 - 2.0f * d;
                atomicMin(&s_key[it_local], ((unsigned long long)ordered_bits(v) << 32) | (uint32_t)c);
            }
        };
        if (ask != 0) {  // uniform
            uint4 rows[RI][KS][2];
#pragma unroll
            for (int ri = 0; ri < RI; ++ri) {
                const uint4* row = cent_row(scored[ri] ? top[ri] : 0);  // (column 0: there is one)
#pragma unroll
                for (int s = 0; s < KS; ++s) {
                    rows[ri][s][0] = row[s * 8];
                    rows[ri][s][1] = row[s * 8 + 1];
                }
            }
#pragma unroll
            for (int ri = 0; ri < RI; ++ri) {
                af32x4_t d4 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int s = 0; s < KS; ++s) {
                    abf16x8_t h, l;
                    halves(rows[ri][s][0], rows[ri][s][1], h, l);
                    d4 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(h, __builtin_bit_cast(abf16x8_t, b[ri][s]), d4, 0, 0, 0);
                    d4 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(l, __builtin_bit_cast(abf16x8_t, b[ri][s]), d4, 0, 0, 0);
                }
                put_diagonal(d4, top_n2[ri], top[ri], ri * 16 + n, scored[ri]);
            }
        }
        for (int p0 = 0; p0 < npairs; p0 += 16) {  // uniform in the wave
            const int pi = min(p0 + n, npairs - 1);
            const int it_local = s_item[pi], col = s_col[pi];
            int it = 0;
#pragma unroll
            for (int ri = 0; ri < RI; ++ri) {
                const int o = __shfl(item[ri], it_local & 15, 64);
                if ((it_local >> 4) == ri) it = o;
            }
            const uint4* row = cent_row(col);
            const uint4* xt = reinterpret_cast<const uint4*>(reinterpret_cast<const uint16_t*>(job.x) +
                                                             ((size_t)t * job.x_tree_stride + it) * (32 * KS) + kb * 8);
            uint4 rows[KS][2], xr[KS];
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                rows[s][0] = row[s * 8];
                rows[s][1] = row[s * 8 + 1];
                xr[s] = xt[s * 4];
            }
            const float n2 = n2t[col];
            af32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                abf16x8_t h, l;
                halves(rows[s][0], rows[s][1], h, l);
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(h, __builtin_bit_cast(abf16x8_t, xr[s]), acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(l, __builtin_bit_cast(abf16x8_t, xr[s]), acc, 0, 0, 0);
            }
            put_diagonal(acc, n2, col, it_local, p0 + n < npairs);
        }
    } else {
        // LPR lanes a pair, as the vector-ALU kernel holds an item and a centroid
        constexpr int EPL = Elem<T>::kPerChunk;
        int lpr = 2;
        while (lpr * EPL < job.D) lpr <<= 1;
        const int rpw = 64 / lpr, rg = lane / lpr, ch = lane % lpr;
        const bool chunk_ok = ch * EPL < job.D;
        for (int p0 = 0; p0 < npairs; p0 += rpw) {  // uniform in the wave
            const int pi = min(p0 + rg, npairs - 1);
            const int it_local = s_item[pi], col = s_col[pi];
            int it = 0;
#pragma unroll
            for (int ri = 0; ri < RI; ++ri) {
                const int o = __shfl(item[ri], it_local & 15, 64);
                if ((it_local >> 4) == ri) it = o;
            }
            const int k = job.open.ids != nullptr ? job.open.ids[(size_t)t * K + col] : col;
            uint4 raw = make_uint4(0, 0, 0, 0);
            float c[EPL];
#pragma unroll
            for (int e = 0; e < EPL; ++e) c[e] = 0.0f;
            if (chunk_ok) {
                raw = load_chunk<T>(job.x, ((size_t)t * job.x_tree_stride + it) * job.D, ch);
                const float* cp = job.cent + ((size_t)t * K + k) * job.D + ch * EPL;
#pragma unroll
                for (int e = 0; e < EPL; e += 4) {
                    const float4 v = *reinterpret_cast<const float4*>(cp + e);
                    c[e] = v.x, c[e + 1] = v.y, c[e + 2] = v.z, c[e + 3] = v.w;
                }
            }
            float x[EPL];
            unpack<T>(raw, x);
            float ss = 0.0f;
#pragma unroll
            for (int e = 0; e < EPL; ++e) {
                const float df = x[e] - c[e];
                ss += df * df;
            }
            ss = group_sum_of(ss, lpr);
            if (ch == 0 && p0 + rg < npairs)
                atomicMin(&s_key[it_local], ((unsigned long long)ordered_bits(ss) << 32) | (uint32_t)col);
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    // ---- lane (kb, n) takes item n of tile kb ----------------------------------------------------
    int it = -1;
    float xx = 0.0f;
    bool un = false;
#pragma unroll
    for (int ri = 0; ri < RI; ++ri)
        if (kb == ri) {
            it = item[ri];
            xx = x2[ri];
            un = unsure[ri];
        }
    const bool listed_later = it >= 0 && un;
    if (__ballot(listed_later) != 0ull) {
        const unsigned long long bal = __ballot(listed_later);
        int base = 0;
        if (lane == __ffsll((long long)bal) - 1) base = atomicAdd(&job.unsure_count[t * kCounterStride], __popcll(bal));
        base = __shfl(base, __ffsll((long long)bal) - 1, 64);
        if (listed_later) job.unsure[(size_t)t * n_c + base + __popcll(bal & ((1ull << lane) - 1ull))] = it;
    }
    if (it >= 0 && !un) {
        const unsigned long long key = s_key[lane];
        int g = -1;
        float d = INFINITY;
        if (key != ~0ull) {
            g = (int)(uint32_t)key;
            if (job.open.ids != nullptr) g = job.open.ids[(size_t)t * K + g];  // column -> centroid
            const float v = from_ordered((uint32_t)(key >> 32));
            d = EXACT_MFMA ? fmaxf(v + xx, 0.0f) : v;
        }
        put_result(job, t, it, g, d);
    }
}

template <typename T, int KS, bool LISTED, bool EXACT_MFMA>
__global__ __launch_bounds__(kApproxThreads, 2) void k_assign_approx(const AssignJob job, const int Kt,
                                                                     const int tag_bits) {
    // (trees in the fast index: the workgroups of a tree run behind the same L2s, which hold its tiles)
    const int t = blockIdx.x;
    constexpr int RI = KS <= 4 ? 4 : 2;
    const int n_items = items_of(job, t);
    if (LISTED && EXACT_MFMA && !approx_takes(n_items, gridDim.x)) return;  // (k_assign_split's)
    const bool narrow = LISTED && !EXACT_MFMA && !approx_takes(n_items, gridDim.x);
    const int per_block = (kApproxThreads / 64) * 16 * (narrow ? 1 : RI);
    if (!EXACT_MFMA && job.counting.zero != nullptr && blockIdx.y == 0 && threadIdx.x == 0) job.counting.zero[t * kCounterStride] = 0;
    for (int b = blockIdx.y; b * per_block < n_items; b += gridDim.y) {  // uniform
        if (b != (int)blockIdx.y) __syncthreads();
        if (LISTED && !EXACT_MFMA && narrow) approx_items<T, KS, 1, LISTED, EXACT_MFMA>(job, Kt, tag_bits, n_items, b);
        else approx_items<T, KS, RI, LISTED, EXACT_MFMA>(job, Kt, tag_bits, n_items, b);
    }
}

// ---- the centroids with room, side by side ---------------------------------------------------
// A workgroup per four tiles of the side-by-side arrays: column i of tile c is the centroid that is the
// (16 c + i)-th not full; the columns behind the last one, up to the end of the stage, are zeros
// that take no items.  Every workgroup counts for itself which centroids those are (a walk over the
// tree's fill counts, 16 KiB at 4096 centroids, instead of a launch of its own ahead: 4.7 us).  That walk bounds it:
// 4096 counts in one trip to memory, 8.6 us a launch at 8 x 4096 centroids, 10.9 with a trip for every 1024.
template <int KS>
__global__ __launch_bounds__(256) void k_open_gather(const CentroidTiles ct, const int32_t* fill, int K,
                                                     int bf, int Kt, int32_t* ids, int32_t* count,
                                                     const CentroidTiles open) {
    constexpr int TILE_CHUNKS = 2 * KS * 64;
    constexpr int TPS = assign_stage(KS);
    __shared__ int s_ids[64];
    __shared__ uint64_t s_w[4];
    const int t = blockIdx.x, block = tree_block(), lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int first = block * 64;  // my columns: [first, first + 64)
    const int32_t* ft = fill + (size_t)t * K;
    if (threadIdx.x < 64) s_ids[threadIdx.x] = -1;
    int before = 0;  // open centroids ahead of the stretch
    for (int k0 = 0; k0 < K; k0 += 4096) {  // uniform; four runs of 1024, their counts in 16 bits of a sum each
        unsigned open_mask[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            open_mask[r] = 0;
            const int k = k0 + r * 1024 + (int)threadIdx.x * 4;
            if (k0 + r * 1024 >= K) continue;  // uniform
            if (K % 4 == 0) {  // uniform (rows of the trees begin on 16 bytes)
                const int4 f = *reinterpret_cast<const int4*>(ft + min(k, K - 4));
                if (k < K) open_mask[r] = (f.x < bf ? 1u : 0u) | (f.y < bf ? 2u : 0u) | (f.z < bf ? 4u : 0u) | (f.w < bf ? 8u : 0u);
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (k + j < K && ft[k + j] < bf) open_mask[r] |= 1u << j;
            }
        }
        // (a lane's place by ballots: 4 masks a run, where a scan over the lanes was six dependent steps through the LDS crossbar:
        // builds of 8 x 32768 keys, seven such launches, 569.3 -> 566.1 us, 8 x 20000 420.1 -> 417.8)
        uint64_t ahead = 0, sum = 0;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if (k0 + r * 1024 >= K) continue;  // uniform
            unsigned mine = 0, ours = 0;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint64_t m = __ballot((open_mask[r] >> j) & 1u);
                mine = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, mine));
                ours += (unsigned)__popcll(m);
            }
            ahead |= (uint64_t)mine << (16 * r);
            sum |= (uint64_t)ours << (16 * r);
        }
        if (lane == 0) s_w[wave] = sum;
        __syncthreads();
        for (int w = 0; w < wave; ++w) ahead += s_w[w];
        const uint64_t all = s_w[0] + s_w[1] + s_w[2] + s_w[3];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if (k0 + r * 1024 >= K) continue;  // uniform
            int at = before + (int)((ahead >> (16 * r)) & 0xffffu);
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if ((open_mask[r] >> j) & 1u) {
                    const int k = k0 + r * 1024 + (int)threadIdx.x * 4 + j;
                    if (block == 0) ids[(size_t)t * K + at] = k;
                    if (at >= first && at < first + 64) s_ids[at - first] = k;
                    ++at;
                }
            before += (int)((all >> (16 * r)) & 0xffffu);
        }
        __syncthreads();
    }
    if (block == 0 && threadIdx.x == 0) count[t] = before;
    const int need = min((((before + 15) / 16 + TPS - 1) / TPS) * TPS, Kt);  // tiles the assignment will walk
    const int tile = block * 4 + wave;
    if (tile >= need) return;
    const uint4* src = ct.tiles + (size_t)t * Kt * TILE_CHUNKS;
    uint4* dst = open.tiles + ((size_t)t * Kt + tile) * TILE_CHUNKS;
    const int i = lane & 15;
    const int k = s_ids[wave * 16 + i];
#pragma unroll
    for (int c0 = 0; c0 < TILE_CHUNKS; c0 += 64) {
        const int ci = c0 + lane;  // (ci % 16 == i: a lane always moves chunks of its own column)
        uint4 v = make_uint4(0, 0, 0, 0);
        if (k >= 0) v = src[(size_t)(k >> 4) * TILE_CHUNKS + (ci - i) + (k & 15)];
        dst[ci] = v;
    }
    if (lane < 16) {
        const size_t o = ((size_t)t * Kt + tile) * 16 + i, c = (size_t)t * Kt * 16 + max(k, 0);
        open.n2[o] = k >= 0 ? ct.n2[c] : INFINITY;
        open.lo[o] = k >= 0 ? ct.lo[c] : 0.0f;
    }
}

int launch_open_centroids(int KS, const CentroidTiles& ct, const int32_t* fill, int bf, int K,
                          int num_trees, int32_t* open_ids, int32_t* open_count,
                          const CentroidTiles& open, hipStream_t s) {
    const int Kt = assign_tiles(K);
    const dim3 grid = tree_grid((Kt + 3) / 4, num_trees);
    switch (KS) {
        case 2: hipLaunchKernelGGL((k_open_gather<2>), grid, dim3(256), 0, s, ct, fill, K, bf, Kt, open_ids, open_count, open); break;
        case 4: hipLaunchKernelGGL((k_open_gather<4>), grid, dim3(256), 0, s, ct, fill, K, bf, Kt, open_ids, open_count, open); break;
        case 8: hipLaunchKernelGGL((k_open_gather<8>), grid, dim3(256), 0, s, ct, fill, K, bf, Kt, open_ids, open_count, open); break;
        default: return fail(HIRA_EINVAL, "open centroids: KS %d", KS);
    }
    return HIRA_OK;
}

// centroid tiles per tree, in whole stages
int assign_tiles(int K) {
    const int kt = (K + 15) / 16;
    return (kt + kAssignStage - 1) / kAssignStage * kAssignStage;
}

int assign_ks(int dtype, int D) { return D <= 64 ? 2 : D <= 128 ? 4 : D <= 256 ? 8 : 0; }

// bf16 rows of 64, 128 or 256 columns have an exact kernel on the matrix cores
bool assign_exact_on_mfma(int dtype, int D) { return dtype == HIRA_BF16 && (D == 64 || D == 128 || D == 256); }

// hi/lo tiles and norms of the centroids of every tree
int launch_cent_prep(int dim, const float* cent, int K, int num_trees, const int32_t* fill, int bf,
                     void* tiles, float* cn2, hipStream_t s) {
    const int Kt = assign_tiles(K);
    const dim3 grid(Kt, num_trees);
    uint4* tl = reinterpret_cast<uint4*>(tiles);
    switch (dim) {
        case 64: hipLaunchKernelGGL((k_cent_prep<2>), grid, dim3(64), 0, s, cent, K, fill, bf, tl, cn2, Kt); break;
        case 128: hipLaunchKernelGGL((k_cent_prep<4>), grid, dim3(64), 0, s, cent, K, fill, bf, tl, cn2, Kt); break;
        case 256: hipLaunchKernelGGL((k_cent_prep<8>), grid, dim3(64), 0, s, cent, K, fill, bf, tl, cn2, Kt); break;
        default: return fail(HIRA_EINVAL, "MFMA assignment: dim %d", dim);
    }
    return HIRA_OK;
}

template <int KS>
static int launch_exact(const AssignJob& job, hipStream_t s) {
    const int Kt = assign_tiles(job.K);
    // Many items walk the centroids 256 a workgroup, every tile read once for all of them; lists, whose
    // length only the device knows, and few items, which would leave the chip idle, 64 a workgroup.
    if (job.list != nullptr || job.after_approx || (long long)job.n_c * job.num_trees <= kApproxListItems) {
        const int per_block = split_ri(KS) * 16, blocks = (job.n_c + per_block - 1) / per_block;
        hipLaunchKernelGGL((k_assign_split<KS>), dim3(job.num_trees, min(blocks, split_blocks(KS, job.num_trees))),
                           dim3(kSplitThreads), 0, s, job, Kt);
        return HIRA_OK;
    }
    static int asked[kMaxDevices];
    constexpr int TPS = assign_stage(KS);
    constexpr size_t smem = 2 * (size_t)TPS * (2 * KS * 64) * sizeof(uint4) + 2 * (size_t)TPS * 16 * sizeof(float);
    if (const int rc = ask_for_lds(reinterpret_cast<const void*>(&k_assign_mfma<KS>), smem, asked, current_device()))
        return rc;
    const int per_block = (kAssignThreads / 64) * kAssignRI * 16;
    hipLaunchKernelGGL((k_assign_mfma<KS>), dim3((job.n_c + per_block - 1) / per_block, job.num_trees),
                       dim3(kAssignThreads), smem, s, job, Kt);
    return HIRA_OK;
}

// nearest usable centroid of every item, or of the items list[0 .. *list_count) of each tree, or of those
// the approximate pass over either left
int launch_assign_mfma(const AssignJob& job, hipStream_t s) {
    switch (job.D) {
        case 64: return launch_exact<2>(job, s);
        case 128: return launch_exact<4>(job, s);
        case 256: return launch_exact<8>(job, s);
        default: return fail(HIRA_EINVAL, "MFMA assignment: dim %d", job.D);
    }
}

template <typename T, int KS, bool LISTED, bool EXACT_MFMA>
static int launch_approx(const AssignJob& job, hipStream_t s) {
    static int asked[kMaxDevices];
    constexpr int TPS = approx_stage(KS);
    // (the pairs lie where the tiles were)
    constexpr size_t tiles = 2 * (size_t)TPS * (KS * 64 * sizeof(uint4) + 16 * sizeof(float)) + 2 * (kApproxThreads / 64) * sizeof(float);
    constexpr size_t pairs = kApproxThreads / 64 * (64 * 8 + kApproxPairs * 8), smem = tiles > pairs ? tiles : pairs;
    if (const int rc = ask_for_lds(reinterpret_cast<const void*>(&k_assign_approx<T, KS, LISTED, EXACT_MFMA>), smem, asked,
                                   current_device()))
        return rc;
    constexpr int RI = KS <= 4 ? 4 : 2;
    const int per_block = (kApproxThreads / 64) * (LISTED && !EXACT_MFMA ? 1 : RI) * 16;
    const int blocks = min((job.n_c + per_block - 1) / per_block, 65535);  // (they go on in strides)
    const int Kt = assign_tiles(job.K);
    int tag_bits = 1;
    while ((1 << tag_bits) < Kt * 4) ++tag_bits;
    if (tag_bits > kMaxTagBits) return fail(HIRA_EINVAL, "approximate assignment: %d centroids", job.K);
    hipLaunchKernelGGL((k_assign_approx<T, KS, LISTED, EXACT_MFMA>), dim3(job.num_trees, blocks), dim3(kApproxThreads),
                       smem, s, job, Kt, tag_bits);
    return HIRA_OK;
}

template <typename T, int KS, bool EXACT_MFMA>
static int launch_approx_l(const AssignJob& job, hipStream_t s) {
    return job.list != nullptr ? launch_approx<T, KS, true, EXACT_MFMA>(job, s)
                               : launch_approx<T, KS, false, EXACT_MFMA>(job, s);
}

int launch_assign_approx(const AssignJob& job, hipStream_t s) {
    const int KS = assign_ks(job.dtype, job.D);
    if (assign_exact_on_mfma(job.dtype, job.D)) {
        if (KS == 2) return launch_approx_l<bf16_t, 2, true>(job, s);
        if (KS == 4) return launch_approx_l<bf16_t, 4, true>(job, s);
        return launch_approx_l<bf16_t, 8, true>(job, s);
    }
    if (job.dtype == HIRA_BF16) {
        if (KS == 2) return launch_approx_l<bf16_t, 2, false>(job, s);
        if (KS == 4) return launch_approx_l<bf16_t, 4, false>(job, s);
        if (KS == 8) return launch_approx_l<bf16_t, 8, false>(job, s);
    } else {
        if (KS == 2) return launch_approx_l<float, 2, false>(job, s);
        if (KS == 4) return launch_approx_l<float, 4, false>(job, s);
        if (KS == 8) return launch_approx_l<float, 8, false>(job, s);
    }
    return fail(HIRA_EINVAL, "approximate assignment: %d columns", job.D);
}

// whether the approximate pass can take a level of K centroids over rows of D columns, and pays: it
// costs a launch for the items it is unsure of, so the exact kernel must have something to lose
bool assign_approx_pays(int dtype, int D, int K) {
    if (assign_ks(dtype, D) == 0 || assign_tiles(K) * 4 > (1 << kMaxTagBits)) return false;
    return K >= (assign_exact_on_mfma(dtype, D) ? kApproxMinMfma : kApproxMinSimple);
}

}  // namespace hira
