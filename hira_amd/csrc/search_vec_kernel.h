// Halfspace range search over the fixed-fan-out ball tree, fused with sparse attention, on the
// vector units: any row width, fan-out, depth and type (the matrix-core kernel next door takes
// the bf16 shapes it is made for).
//
// One launch covers every tree and every query head.  A workgroup owns a run of consecutive
// level-1 nodes ("leaf parents") of one tree and takes them up to kBatch at a time, in three steps:
//   gates   all rows the batch needs -- its nodes and, once each, their ancestors at every level --
//           are asked for together and dealt out over the workgroup's lane groups; each leaves a
//           word in LDS saying for which heads it passes;
//   list    a node survives for the heads that it and all its ancestors pass for: one wave puts the
//           survivors side by side in LDS;
//   scan    the survivors' key slots, end to end, are dealt out over the waves in blocks of up to 64
//           rows; the values of a block's selected rows are asked for together.
// So a launch is a chain of four trips to memory (arguments, gates, keys, values) plus the hand-off
// of the partials, whatever the fan-out, and a pruned node costs nothing behind its gate.  (4 trees x
// 5003 rows of 80 fp32, three heads, as the work falls away: 15.25 us; with a key a head selected 13.4;
// with every node pruned 10.6; without the attention 8.8, 8.6 and 5.6.)  Small launches ask for gates and
// keys at once, in straight-line code (ONE, below): 12.4 us for that one.  No
// global frontier is exchanged between workgroups.  (Before, every wave walked nodes of its own:
// each gate repeated the ancestors' rows, and short nodes left most lanes without a row.)
//
// Lane layout: a row of D elements is 16-byte chunks; LPR lanes hold one row (lane % LPR =
// chunk), so a wave reads RPW = 64/LPR rows per 128-bit load instruction, fully coalesced.  The
// query heads that share the tree (GQA group) are scored against every chunk that is loaded: one
// HBM read of a centroid or key row serves the whole group.
//
// Semantics (reference: kernels/cpp/torch_ext_v3.cpp:172-242, with the conservative
// non-unit-query bound of searcher/cpu.py:61-63): keep a node when q.c + ||q||*r >= tau,
// select a key when q.k >= tau.
#pragma once
#include "search.h"
#include "threshold_kernel.h"

namespace hira {

constexpr int kVecThreads = 512;  // workgroup size, at most
constexpr int kBatch = 64;        // level-1 nodes a workgroup gates together
constexpr int kOneGateRows = 2;   // level-1 rows a lane group asks for where there is one batch (ONE, below)
// rows of a block that a wave scans at once: eight loads a lane (with eight heads a pass as many as
// the registers have room for: four, two of bf16), at most 64 rows
constexpr int vec_rows(int rpw, int gmax, int epl) {
    const int r = (gmax <= 4 ? 8 : 16 / epl) * rpw;
    return r < 64 ? r : 64;
}
// rows of a wave's block where it has only one (ONE, below), for `elems` elements a lane: a block is as much
// work whatever it holds, so the smaller one is taken where the workgroups then still fit
constexpr int kOneSmall = 16, kOneLarge = 32;
constexpr int vec_one_rows(int rpw, int epl, int elems) {
    const int r = elems / epl * rpw;
    return r < 64 ? r : 64;
}

// ---- sums over the LPR lanes of a row, many at once ------------------------------------------
// Every lane comes with NV partial sums (value u * GMAX + g: row u of the lane group's block, head
// g).  Summing each over the lanes by itself takes log2(LPR) steps a value; here a step over a lane
// bit also halves the values a lane goes on with (lanes with the bit clear keep the first half,
// the others the second), until a lane holds the sums of its own max(NV / LPR, 1) values: 77
// instructions for 32 values over 32 lanes instead of 192 and as many LDS permutes.
constexpr int vec_kept(int nv, int lpr) { return nv >= lpr ? nv / lpr : 1; }
// first value whose sum lane `j` of a lane group ends up with
constexpr int vec_value_of(int j, int nv, int lpr) {
    int v = 0, n = nv;
    for (int bit = lpr / 2; bit >= 1 && n > 1; bit /= 2) {
        n /= 2;
        if (j & bit) v += n;
    }
    return v;
}
// lanes of a group that hold a value nobody below them holds too (fewer values than lanes)
constexpr bool vec_is_owner(int j, int nv, int lpr) {
    for (int i = 0; i < j; ++i)
        if (vec_value_of(i, nv, lpr) == vec_value_of(j, nv, lpr)) return false;
    return true;
}
// lanes of the wave that hold a value of row u of their group's block
template <int GMAX, int NV, int LPR>
struct VecLanes {
    uint64_t row[NV / GMAX], any;
    constexpr VecLanes() : row{}, any(0) {
        for (int j = 0; j < LPR; ++j) {
            if (!vec_is_owner(j, NV, LPR)) continue;
            for (int v = vec_value_of(j, NV, LPR), n = 0; n < vec_kept(NV, LPR); ++v, ++n)
                for (int r = 0; r < 64 / LPR; ++r) row[v / GMAX] |= 1ull << (r * LPR + j);
        }
        for (int u = 0; u < NV / GMAX; ++u) any |= row[u];
    }
};

template <int N, int BIT>
__device__ __forceinline__ void reduce_step(float* v, int lane) {
    // partner: a lane that differs in BIT (and maybe in lower bits)
    constexpr int CTRL = BIT == 8 ? 0x140 : BIT == 4 ? 0x141 : BIT == 2 ? 0x1B : 0xB1;
    if constexpr (N > 1) {
        constexpr int H = N / 2;
#pragma unroll
        for (int i = 0; i < H; ++i) {
            if constexpr (BIT >= 16) {
                const auto r = BIT == 32 ? __builtin_amdgcn_permlane32_swap(__float_as_uint(v[i]), __float_as_uint(v[i + H]), false, false)
                                         : __builtin_amdgcn_permlane16_swap(__float_as_uint(v[i]), __float_as_uint(v[i + H]), false, false);
                v[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
            } else {
                const bool up = (lane & BIT) != 0;
                const float keep = up ? v[i + H] : v[i], send = up ? v[i] : v[i + H];
                v[i] = keep + dpp_move<CTRL>(send);
            }
        }
    } else if constexpr (BIT >= 16) {
        const auto r = BIT == 32 ? __builtin_amdgcn_permlane32_swap(__float_as_uint(v[0]), __float_as_uint(v[0]), false, false)
                                 : __builtin_amdgcn_permlane16_swap(__float_as_uint(v[0]), __float_as_uint(v[0]), false, false);
        v[0] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    } else {
        v[0] += dpp_move<CTRL>(v[0]);
    }
}
template <int N, int BIT>
__device__ __forceinline__ void reduce_scatter(float* v, int lane) {
    reduce_step<N, BIT>(v, lane);
    if constexpr (BIT > 1) reduce_scatter<(N > 1 ? N / 2 : 1), BIT / 2>(v, lane);
}

// The fold as the work of one workgroup per head (a launch of its own):
// out[o0 ..] = sum_p 2^(m_p - M) acc_p / sum_p 2^(m_p - M) l_p over the P partials of one head, by
// all threads of the workgroup (a multiple of 64, at least dvl).  Thread t owns four columns of
// the output (t % dvl) for the partials p = t / dvl (mod ng).  rows: (ng, Dv + 1) floats of
// LDS, red: one float per wave.  The partials are read with device-scope loads: they may have
// been written by workgroups behind another L2.
__device__ __forceinline__ void fold_partials(const float* pm, const float* pl, const float* pa,
                                              int P, int Dv, int dvl, void* out, int out_bf16,
                                              size_t o0, float* rows, float* red) {
    auto ld = [](const float* q) {
        return __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    const int t = threadIdx.x, nt = blockDim.x, nw = nt >> 6;
    float mx = -INFINITY;
    for (int i = t; i < P; i += nt) mx = fmaxf(mx, ld(pm + i));
    mx = wave_max(mx);
    if ((t & 63) == 0) red[t >> 6] = mx;
    __syncthreads();
    float M = red[0];
    for (int w = 1; w < nw; ++w) M = fmaxf(M, red[w]);
    if (M == -INFINITY) {  // nothing selected for this head (uniform)
        for (int e = t; e < Dv; e += nt) store_out(out, out_bf16, o0 + e, 0.0f);
        return;
    }
    const int ng = nt / dvl;
    const int gi = t / dvl, li = t % dvl;
    float a[4] = {0.f, 0.f, 0.f, 0.f};
    float lsum = 0.0f;
    const bool lane_ok = li * 4 < Dv;
    // (four partials in flight; nothing is asked for only after something else has arrived.  A
    // partial without a selected key may hold anything: it is masked, not multiplied)
    constexpr int U = 4;
    for (int i0 = gi; i0 < P; i0 += U * ng) {
        float m[U], l[U], v[U][4];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = min(i0 + u * ng, P - 1);
            m[u] = ld(pm + i);
            l[u] = ld(pl + i);
#pragma unroll
            for (int c = 0; c < 4; ++c) v[u][c] = lane_ok ? ld(pa + (size_t)i * Dv + li * 4 + c) : 0.0f;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (i0 + u * ng >= P || m[u] == -INFINITY) continue;
            const float w = exp2f(m[u] - M);
            lsum += w * l[u];
#pragma unroll
            for (int c = 0; c < 4; ++c) a[c] += w * v[u][c];
        }
    }
    float* row = rows + (size_t)gi * (Dv + 1);
    if (lane_ok) {
#pragma unroll
        for (int c = 0; c < 4; ++c) row[li * 4 + c] = a[c];
    }
    if (li == 0) row[Dv] = lsum;
    __syncthreads();
    float ltot = 0.0f;
    for (int g = 0; g < ng; ++g) ltot += rows[(size_t)g * (Dv + 1) + Dv];
    for (int e = t; e < Dv; e += nt) {
        float sum = 0.0f;
        for (int g = 0; g < ng; ++g) sum += rows[(size_t)g * (Dv + 1) + e];
        store_out(out, out_bf16, o0 + e, sum / ltot);
    }
}

// The fold by the last workgroup of a tree and pass to arrive: its G heads side by side, in two
// trips to memory.  A wave per head takes the partials' maxima and sums and lists those that hold
// anything with their weights; then a thread owns four output columns of a head and every
// n_grp-th listed partial, eight 16-byte loads in flight; the groups' sums meet in LDS.  (One head
// after the other, as the fold above would do it, took 7 us more at 4 heads x 64 partials than a
// second launch with a workgroup per head; side by side it takes less than that launch.)
//   lds: 2 G P floats, then blockDim.x * 4
constexpr int kVecFoldMax = 4096;  // G * P at most
__device__ __forceinline__ void fold_heads(const SearchParams& p, int hoff, int G, float* lds) {
    __shared__ float s_l[8];
    __shared__ int s_n[8];
    auto ld = [](const float* q) {
        return __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, nw = blockDim.x >> 6;
    const int P = p.num_parts, Dv = p.vdim;
    int* list = reinterpret_cast<int*>(lds);   // (G, P)
    float* wts = lds + (size_t)G * P;          // (G, P)
    float* red = lds + 2 * (size_t)G * P;      // (n_grp, G * Dv)
    for (int g = wave; g < G; g += nw) {  // uniform in the wave
        const int head = p.group_size > 0 ? hoff + g : p.tree_q_heads[hoff + g];
        const float* pm = p.part_m + (size_t)head * P;
        const float* pl = p.part_l + (size_t)head * P;
        // (the first 64 partials' in one trip: up to there nothing is asked for twice)
        const float m0 = lane < P ? ld(pm + lane) : -INFINITY, l0 = lane < P ? ld(pl + lane) : 0.0f;
        float mx = m0;
        for (int i = lane + 64; i < P; i += 64) mx = fmaxf(mx, ld(pm + i));
        mx = wave_max(mx);
        float ls = 0.0f;
        int n = 0;
        for (int i0 = 0; i0 < P; i0 += 64) {  // uniform
            const int i = i0 + lane;
            const float m = i0 == 0 ? m0 : (i < P ? ld(pm + i) : -INFINITY);
            const float l = i0 == 0 ? l0 : (i < P ? ld(pl + i) : 0.0f);
            const float w = m > -INFINITY ? exp2f(m - mx) : 0.0f;
            ls += w * l;
            // (whatever holds a selected key, however small its weight beside the others': zero times an
            // infinite sum is no zero)
            const bool nz = m > -INFINITY;
            const unsigned long long bal = __ballot(nz);
            if (nz) {
                const int k = n + __popcll(bal & ((1ull << lane) - 1ull));
                list[g * P + k] = i;
                wts[g * P + k] = w;
            }
            n += __popcll(bal);
        }
        ls = wave_sum(ls);
        if (lane == 0) {
            s_l[g] = ls;
            s_n[g] = n;
        }
    }
    __syncthreads();
    const int quads = Dv / 4, items = G * quads;
    // (quotients of small numbers as products with a reciprocal, exact for numbers of a few thousand: a division is
    // thirty instructions of a chain)
    const float inv_items = 1.0f / (float)items, inv_quads = 1.0f / (float)quads, inv_dv = 1.0f / (float)Dv;
    auto over = [](int x, float inv) { return (int)(((float)x + 0.5f) * inv); };
    const int n_grp = max(over((int)blockDim.x, inv_items), 1);
    for (int i0 = 0; i0 < items; i0 += blockDim.x) {  // uniform; once unless G * Dv > 4 threads
        const int grp = n_grp > 1 ? over(t, inv_items) : 0, item = n_grp > 1 ? t - grp * items : i0 + t;
        if (item < items && grp < n_grp) {
            const int g = over(item, inv_quads), qd = item - g * quads;
            const int head = p.group_size > 0 ? hoff + g : p.tree_q_heads[hoff + g];
            typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
            const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
                const_cast<float*>(p.part_acc), 0, 0x7fffffff, 0x00020000);
            const unsigned col0 = ((unsigned)head * (unsigned)P * (unsigned)Dv + 4u * (unsigned)qd) * 4u;
            const int n = s_n[g];
            float sx = 0.0f, sy = 0.0f, sz = 0.0f, sw = 0.0f;
            for (int k0 = grp; k0 < n; k0 += 8 * n_grp) {
                u32x4 v[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) {  // (16: the device-scope bit)
                    // (beyond the list: an address beyond the buffer, which reads as zero)
                    const unsigned at = col0 + (unsigned)list[g * P + min(k0 + u * n_grp, n - 1)] * (unsigned)(Dv * 4);
                    v[u] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, k0 + u * n_grp < n ? at : 0xfffffff0u, 0, 16);
                }
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const float w = k0 + u * n_grp < n ? wts[g * P + k0 + u * n_grp] : 0.0f;
                    sx += w * __uint_as_float(v[u].x);
                    sy += w * __uint_as_float(v[u].y);
                    sz += w * __uint_as_float(v[u].z);
                    sw += w * __uint_as_float(v[u].w);
                }
            }
            if (n_grp > 1) {
                float4* r = reinterpret_cast<float4*>(red + (size_t)grp * items * 4 + item * 4);
                *r = make_float4(sx, sy, sz, sw);
            } else {
                const float L = s_l[g];
                const float o[4] = {sx, sy, sz, sw};
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    store_out(p.attn_out, p.out_bf16, (size_t)head * Dv + qd * 4 + c, L == 0.0f ? 0.0f : o[c] / L);
            }
        }
    }
    if (n_grp == 1) return;
    __syncthreads();
    for (int e = t; e < items * 4; e += blockDim.x) {
        const int g = over(e, inv_dv);
        const int head = p.group_size > 0 ? hoff + g : p.tree_q_heads[hoff + g];
        float sum = 0.0f;
        for (int r = 0; r < n_grp; ++r) sum += red[(size_t)r * items * 4 + e];
        const float L = s_l[g];
        store_out(p.attn_out, p.out_bf16, (size_t)head * Dv + (e - g * Dv), L == 0.0f ? 0.0f : sum / L);
    }
}

// The arguments that the kernel needs up to the keys, in registers from its first instructions on (asked for where they
// are used they came one after the other, each behind its branch and its wait).  Levels 1, 2 and the one above
// that the wave has for itself, whether they are there or not.  (4 trees x 5003 rows of 80 fp32, three
// heads each: 11.5 -> 11.15 us.)
struct VecArgs {
    const void *q, *keys, *queue_keys, *centers[3];
    const float *tau, *scaling, *radii[3];
    const int32_t* counts;
    int32_t level_cap[3], dim, num_levels, group_size, tree_blocks, num_queue_blocks, num_nodes, queue_nodes, nodes_per_wg;
    int32_t queue_cap, cap[1], queue_len, size[1], bf, layout, key_layout, wgs;
    uint32_t bf_magic;
};
__device__ __forceinline__ VecArgs vec_arguments(const SearchParams& p, int upper) {
    VecArgs v{p.q, p.keys, p.queue_keys, {p.centers[1], p.centers[2], p.centers[upper]}, p.tau, p.scaling,
              {p.radii[1], p.radii[2], p.radii[upper]}, p.counts[1], {p.cap[1], p.cap[2], p.cap[upper]}, p.dim, p.num_levels,
              p.group_size, p.tree_blocks, p.num_queue_blocks, p.num_nodes, p.queue_nodes, p.nodes_per_wg, p.queue_cap, {p.cap[0]},
              p.queue_len, {p.size[0]}, p.bf, p.layout, p.key_layout, (int)gridDim.x, p.bf_magic};
    auto at = [](const void* a) { return reinterpret_cast<uintptr_t>(a); };
    uintptr_t q = at(v.q), keys = at(v.keys), queue = at(v.queue_keys), tau = at(v.tau), scaling = at(v.scaling),
              c0 = at(v.centers[0]), c1 = at(v.centers[1]), c2 = at(v.centers[2]), r0 = at(v.radii[0]), r1 = at(v.radii[1]),
              r2 = at(v.radii[2]), counts = at(v.counts);
    asm volatile("" : "+s"(v.queue_cap), "+s"(v.cap[0]), "+s"(v.queue_len), "+s"(v.size[0]), "+s"(v.bf), "+s"(v.layout),
                      "+s"(v.key_layout), "+s"(v.wgs), "+s"(v.bf_magic));
    asm volatile("" : "+s"(v.level_cap[0]), "+s"(v.level_cap[1]), "+s"(v.level_cap[2]), "+s"(v.dim), "+s"(v.num_levels),
                      "+s"(v.group_size), "+s"(v.tree_blocks), "+s"(v.num_queue_blocks), "+s"(v.num_nodes), "+s"(v.queue_nodes),
                      "+s"(v.nodes_per_wg));
    asm volatile("" : "+s"(q), "+s"(keys), "+s"(queue), "+s"(tau), "+s"(scaling), "+s"(c0), "+s"(c1), "+s"(c2), "+s"(r0),
                      "+s"(r1), "+s"(r2), "+s"(counts));
    v.q = global_at<char>(q), v.keys = global_at<char>(keys), v.queue_keys = global_at<char>(queue);
    v.tau = global_at<float>(tau), v.scaling = global_at<float>(scaling), v.counts = global_at<int32_t>(counts);
    v.centers[0] = global_at<char>(c0), v.centers[1] = global_at<char>(c1), v.centers[2] = global_at<char>(c2);
    v.radii[0] = global_at<float>(r0), v.radii[1] = global_at<float>(r1), v.radii[2] = global_at<float>(r2);
    return v;
}

// Argument x of the kernel: with ONE as vec_arguments has it, else where it lies.  (The general way, which asks for keys
// once it has its list of nodes, was slower with all of them in registers from the start: 90000 rows of 128 fp32 8.6 -> 8.8 us.)
#define VEC_ARG(x) (ONE ? va.x : p.x)

// ONE > 0: every workgroup of the launch has one batch of nodes whose key slots are one block of rows for
// each of its eight waves (of ONE elements a lane).  A wave then asks for its block together with the gates'
// operands of all levels, whether the nodes survive or not: no list, two trips to memory and a barrier less,
// and no loop, at whose head the waits would be for everything asked for so far.  Every row being in some
// wave's block, a dense output's fill value goes out with the scores.
// SAMPLED: (with ONE, bf16 rows of 8 * LPR columns) the launch makes its thresholds itself, in workgroups ahead of the
// searching ones of a tree (threshold_stretch); a workgroup looks for them with its keys on their way.
template <typename T, int LPR, int GMAX, int ONE, bool SAMPLED = false>
__global__ __launch_bounds__(kVecThreads) __attribute__((amdgpu_waves_per_eu(GMAX == 1 ? 3 : 2)))
void search_kernel(const SearchParams p) {
    constexpr int EPL = Elem<T>::kPerChunk;
    constexpr int RPW = kWave / LPR;  // rows per wave-wide load
    constexpr int DVP = LPR * EPL;    // widest row a lane group can hold
    constexpr int KU = (ONE ? vec_one_rows(RPW, EPL, ONE) : vec_rows(RPW, GMAX, EPL)) / RPW;  // row loads in flight per lane
    constexpr int ROWS = KU * RPW;
    constexpr int NV = KU * GMAX;                  // scores a lane group makes of a block
    constexpr int KEPT = vec_kept(NV, LPR);
    constexpr VecLanes<GMAX, NV, LPR> LANES{};
    constexpr int WAVES = kVecThreads / 64;

    extern __shared__ float smem[];
    // logits, then weights, of a block's rows (-inf / 0: not selected): the wave's lanes share the
    // work on them, and no lane keeps its rows' scores while the values are on their way
    __shared__ __attribute__((aligned(16))) float s_tab[WAVES][ROWS * GMAX];
    __shared__ uint32_t s_pass[HIRA_MAX_LEVELS][kBatch + 1];  // heads a row passes for | 1 << 31: not empty
    __shared__ uint32_t s_list[kBatch];  // survivors: node - first | child count << 8 | heads << 16
    __shared__ int s_count;
    static_assert(!SAMPLED || (ONE > 0 && sizeof(T) == 2 && kVecThreads == kTauStretch), "");
    __shared__ float s_tau[SAMPLED ? GMAX : 1], s_scores[SAMPLED ? kTauFewRows : 1];

    touch_kernel_arguments();
    const int lane = lane_id();
    // (uniform, as the compiler would not know: a level picked by it has its arguments read by vector loads otherwise,
    // a trip to memory ahead of the rows')
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    // (the level above the second that a wave has for itself: ONE's workgroups are full ones, whose first wave has none)
    [[maybe_unused]] VecArgs va;
    if constexpr (ONE) va = vec_arguments(p, min(2 + wave, HIRA_MAX_LEVELS - 1));
    const int nwaves = ONE ? WAVES : (int)(blockDim.x >> 6);
    const int rg = lane / LPR;
    const int ch = lane % LPR;
    const int tree = blockIdx.y;
    const int D = VEC_ARG(dim);
    const int Dv = p.vdim;
    const int L = VEC_ARG(num_levels);
    const bool chunk_ok = ch * EPL < D;
    const bool vchunk_ok = ch * EPL < Dv;
    const bool want_attn = p.part_acc != nullptr;

    // (group_size > 0: head h of the launch belongs to tree h / group_size; the head map is not
    // read, which saves every wave two dependent trips to memory)
    const bool by_group = VEC_ARG(group_size) > 0;
    const int hoff = (by_group ? tree * VEC_ARG(group_size) : p.tree_q_off[tree]) + blockIdx.z * GMAX;
    const int G = min(GMAX, (by_group ? (tree + 1) * VEC_ARG(group_size) : p.tree_q_off[tree + 1]) - hoff);
    if (G <= 0) return;  // uniform for the workgroup
    int wgs = ONE ? va.wgs : (int)gridDim.x, wg = blockIdx.x;  // searching workgroups of the tree, my number among them
    if constexpr (SAMPLED) {
        wgs -= p.sample_wgs;
        wg -= p.sample_wgs;
        if (wg < 0) {  // uniform
            threshold_stretch<LPR>(p.sample, p.sample_rows, p.q, tree, G, (int)blockIdx.x, p.sample_best, s_scores, p.done + tree,
                                   wgs + p.sample_wgs * kTauMade);
            return;
        }
    }
    // (what a launch that makes its thresholds keeps lies where the others have their dense output)
    const bool dense = !SAMPLED && p.dense != nullptr, lists = !SAMPLED && p.sel_count != nullptr;
    const unsigned gmask = (1u << G) - 1u;
    auto head_of = [&](int g) { return by_group ? hoff + g : p.tree_q_heads[hoff + g]; };

    const bool is_queue = wg >= VEC_ARG(tree_blocks);
    const int blk = is_queue ? wg - VEC_ARG(tree_blocks) : wg;
    const int n_nodes = is_queue ? VEC_ARG(num_queue_blocks) : VEC_ARG(num_nodes);
    const bool real_nodes = !is_queue && L >= 2;
    const int wg_nodes = is_queue ? VEC_ARG(queue_nodes) : VEC_ARG(nodes_per_wg);
    const int node_first = blk * wg_nodes;
    const int node_last = min(node_first + wg_nodes, n_nodes);

    // threshold, scale and head of the values whose sums this lane ends up with
    int vfirst = 0;  // vec_value_of(ch)
    {
        int n = NV;
#pragma unroll
        for (int bit = LPR / 2; bit >= 1; bit /= 2)
            if (n > 1) {
                n /= 2;
                if (ch & bit) vfirst += n;
            }
    }
    const int my_u = vfirst / GMAX, my_g = vfirst % GMAX;  // row of the block, first head
    // ---- queries of the group: this lane's chunk of each (asked for here, first used at the gates).
    // Heads first, then straight-line loads, those of a head or a chunk that is not there the last one's
    // again, dropped where they are used: with a condition around each head's (its number, `g < G`) the
    // waits at the joins made them a trip to memory after the other ahead of the gates (4 trees x 5003 rows of 80 fp32, three heads each:
    // 15.6 -> 15.25 us, seven heads of 64 16.95 -> 16.55) ----
    int hd[GMAX], my_h[KEPT];
#pragma unroll
    for (int g = 0; g < GMAX; ++g) hd[g] = hoff + min(g, G - 1);
#pragma unroll
    for (int i = 0; i < KEPT; ++i) my_h[i] = hoff + min(my_g + i % GMAX, G - 1);
    if (!by_group) {  // uniform
#pragma unroll
        for (int g = 0; g < GMAX; ++g) hd[g] = p.tree_q_heads[hd[g]];
#pragma unroll
        for (int i = 0; i < KEPT; ++i) my_h[i] = p.tree_q_heads[my_h[i]];
    }
    uint4 qraw[GMAX];
    float tau[GMAX], my_tau[KEPT], my_sc[KEPT];
#pragma unroll
    for (int g = 0; g < GMAX; ++g) {
        qraw[g] = load_chunk<T>(VEC_ARG(q), (size_t)hd[g] * D, chunk_ok ? ch : 0);
        tau[g] = SAMPLED ? 0.0f : VEC_ARG(tau)[hd[g]];
    }
#pragma unroll
    for (int i = 0; i < KEPT; ++i) {
        my_tau[i] = SAMPLED ? 0.0f : VEC_ARG(tau)[my_h[i]];
        my_sc[i] = VEC_ARG(scaling)[my_h[i]];
    }

    const void* kbase = is_queue ? VEC_ARG(queue_keys) : VEC_ARG(keys);
    const void* vbase = is_queue ? p.queue_values : p.values;
    const size_t krow0 = (size_t)tree * (is_queue ? VEC_ARG(queue_cap) : VEC_ARG(cap[0]));
    const int n_rows = is_queue ? VEC_ARG(queue_len) : VEC_ARG(size[0]);
    const int block_rows = real_nodes ? VEC_ARG(bf) : kPseudoBlock;
    const float inv_rows = 1.0f / (float)block_rows;
    const int klayout = is_queue ? HIRA_ROW_MAJOR : VEC_ARG(key_layout);
    auto over_bf = [&](unsigned n) { return VEC_ARG(bf) == 1 ? n : __umulhi(n, VEC_ARG(bf_magic)); };  // n / bf

    // counters, straight to memory (registers are worth more here than the few calls that count)
    auto count = [&](int i, unsigned n) {
        atomicAdd(p.stats + (size_t)tree * HIRA_STATS_COLS + i, (unsigned long long)n);
    };

    // ---- attention state: each lane group's sums under the wave's maximum; lane l keeps maximum
    // and denominator of head l % GMAX (the denominator in parts) ----------------------------
    float acc[GMAX][EPL];
    float m_run = -INFINITY, l_run = 0.0f;
#pragma unroll
    for (int g = 0; g < GMAX; ++g)
#pragma unroll
        for (int e = 0; e < EPL; ++e) acc[g][e] = 0.0f;

    // ---- a wave's block of rows once it has arrived: scores, sums over the lanes, the selection, outputs, the
    // selected rows' values.  slot[u]: key slot of row u of the lane group; mine(): slot of the row
    // whose sums this lane ends up with, whether it is one, the heads it may be selected for --------
    float* tab = s_tab[wave];
    auto take = [&](const uint4 (&raw)[KU], const int (&slot)[KU], auto mine) {
        float s[NV];
#pragma unroll
        for (int u = 0; u < KU; ++u) {
#pragma unroll
            for (int g = 0; g < GMAX; ++g) s[u * GMAX + g] = chunk_dot<T>(raw[u], qraw[g]);
        }
        reduce_scatter<NV, LPR / 2>(s, lane);
        int my_slot;
        bool my_row;
        const unsigned my_am = mine(my_slot, my_row);
        unsigned sel = 0;  // bit i: value i
#pragma unroll
        for (int i = 0; i < KEPT; ++i)
            if (((my_am >> (my_g + i)) & 1u) && (is_queue || s[i] >= my_tau[i])) sel |= 1u << i;
        const bool owner = LANES.any == ~0ull || ((LANES.any >> lane) & 1ull);
        const uint64_t B = __ballot(owner && sel != 0u);  // lanes that hold a selected score
        if constexpr (ONE) {
            // (every row of the workgroup's nodes is in some wave's block: fill value or score)
            if (dense && p.dense_fill && !is_queue && owner && my_row) {
#pragma unroll
                for (int i = 0; i < KEPT; ++i)
                    if (my_g + i < G)
                        p.dense[(int64_t)my_h[i] * p.dense_stride + my_slot] =
                            (sel >> i) & 1u ? s[i] * my_sc[i] : p.dense_fill_value;
            }
        }
        if (B == 0ull) return;  // uniform in the wave
        if (p.stats) {
            // a key is selected where any of its heads is: every row once
#pragma unroll
            for (int u = 0; u < KU; ++u) {
                const uint64_t lanes = B & LANES.row[u];
                for (int r = 0; r < RPW; ++r) {
                    const uint64_t group = LPR == 64 ? ~0ull : ((1ull << (LPR & 63)) - 1ull) << (r * LPR);
                    if (lane == 0 && (lanes & group)) count(HIRA_MAX_LEVELS, 1);
                }
            }
            if (owner && sel) count(HIRA_MAX_LEVELS + 1, (unsigned)__popc(sel));
        }
        if (!is_queue && (dense || lists)) {
            int idx = my_slot;
            if (owner && sel && p.dense_by_position) idx = p.perm[krow0 + my_slot];
            if (dense && owner && !(ONE && p.dense_fill)) {
#pragma unroll
                for (int i = 0; i < KEPT; ++i)
                    if ((sel >> i) & 1u) p.dense[(int64_t)my_h[i] * p.dense_stride + idx] = s[i] * my_sc[i];
            }
            if (lists) {
#pragma unroll
                for (int i = 0; i < KEPT; ++i) {
                    const uint64_t Bi = __ballot(owner && ((sel >> i) & 1u));
#pragma unroll
                    for (int g = 0; g < GMAX; ++g) {
                        // (a head's entries of the wave go side by side: one atomic)
                        const bool mine = owner && ((sel >> i) & 1u) && my_g + i == g;
                        const uint64_t bal = __ballot(mine);
                        if (Bi == 0ull || bal == 0ull) continue;  // uniform
                        int base = 0;
                        if (mine && (bal & ((1ull << lane) - 1ull)) == 0ull)
                            base = atomicAdd(&p.sel_count[my_h[i]], __popcll(bal));
                        base = __shfl(base, __ffsll((long long)bal) - 1, 64);
                        const int pos = base + __popcll(bal & ((1ull << lane) - 1ull));
                        if (mine && pos < p.sel_cap) {
                            p.sel_index[(int64_t)my_h[i] * p.sel_cap + pos] = idx;
                            p.sel_score[(int64_t)my_h[i] * p.sel_cap + pos] = s[i];
                        }
                    }
                }
            }
        }
        if (!want_attn) return;  // uniform
        // ---- the values of the rows that some head selected -------------------------------
        uint4 vraw[KU];
#pragma unroll
        for (int u = 0; u < KU; ++u) {
            vraw[u] = make_uint4(0, 0, 0, 0);
            const uint64_t lanes = B & LANES.row[u];
            const uint64_t group = LPR == 64 ? ~0ull : ((1ull << (LPR & 63)) - 1ull) << (rg * LPR);
            if ((lanes & group) != 0ull && vchunk_ok) vraw[u] = load_chunk<T>(vbase, (krow0 + slot[u]) * Dv, ch);
        }
        if (owner) {
#pragma unroll
            for (int i = 0; i < KEPT; ++i) {
                // (fminf: a logit that is no number becomes +inf.  A maximum does not see the former,
                // and what follows makes NaN of both, as a softmax does)
                const float z = fminf(s[i] * my_sc[i] * kLog2e, INFINITY);
                tab[(my_u * RPW + rg) * GMAX + my_g + i] = (sel >> i) & 1u ? z : -INFINITY;
            }
        }
        // weights while the values are on their way: lane l takes the table's entries
        // l, l + 64, ..., all of head l % GMAX
        constexpr int NE = (ROWS * GMAX + 63) / 64;
        __builtin_amdgcn_wave_barrier();
        float z[NE], mx = -INFINITY;
#pragma unroll
        for (int i = 0; i < NE; ++i) {
            const bool mine = ROWS * GMAX >= 64 || lane < ROWS * GMAX;
            z[i] = mine ? tab[i * 64 + lane] : -INFINITY;
            mx = fmaxf(mx, z[i]);
        }
        mx = fmaxf(cross_group_max<GMAX>(mx), m_run);
        const float f = m_run == -INFINITY ? 0.0f : exp2f(m_run - mx);
        l_run *= f;
        m_run = mx;
#pragma unroll
        for (int i = 0; i < NE; ++i) {
            // (zero says "not selected": a selected row's weight stays above it)
            float w = z[i] > -INFINITY ? exp2f(z[i] - mx) : 0.0f;
            l_run += w;
            if (GMAX > 1 && w == 0.0f && z[i] > -INFINITY) w = 1e-45f;
            if (ROWS * GMAX >= 64 || lane < ROWS * GMAX) tab[i * 64 + lane] = w;
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int g = 0; g < GMAX; ++g) {
            const float fg = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(f), g));
#pragma unroll
            for (int e = 0; e < EPL; ++e) acc[g][e] *= fg;
        }
        // (a row's weights are asked for with the row before it.  The heads that did not select the row
        // are masked out, not multiplied by zero: a value that is not finite stays with those that did.
        // As masks on straight-line code it costs nothing to be seen with up to four heads a pass and 2 %
        // with eight -- 2 trees x 20000 rows of 64 bf16 25.8 -> 26.2 us --, as branches 2 and 7 %)
        float wt[GMAX];
#pragma unroll
        for (int g = 0; g < GMAX; ++g) wt[g] = tab[rg * GMAX + g];
#pragma unroll
        for (int u = 0; u < KU; ++u) {
            float next[GMAX];
#pragma unroll
            for (int g = 0; g < GMAX; ++g) next[g] = tab[(min(u + 1, KU - 1) * RPW + rg) * GMAX + g];
            if ((B & LANES.row[u]) != 0ull) {  // uniform in the wave
                float vf[EPL];
                unpack<T>(vraw[u], vf);
#pragma unroll
                for (int g = 0; g < GMAX; ++g)
                    if (GMAX == 1 || __builtin_expect(wt[g] != 0.0f, 1)) {
#pragma unroll
                        for (int e = 0; e < EPL; ++e) acc[g][e] += wt[g] * vf[e];
                    }
            }
#pragma unroll
            for (int g = 0; g < GMAX; ++g) wt[g] = next[g];
        }
    };
    if constexpr (ONE) {
        float qn[GMAX];
        auto queries = [&]() {
    #pragma unroll
            for (int g = 0; g < GMAX; ++g) {
                if (!chunk_ok) qraw[g] = make_uint4(0, 0, 0, 0);
                float qf[EPL], ss = 0.0f;
                unpack<T>(qraw[g], qf);
    #pragma unroll
                for (int e = 0; e < EPL; ++e) ss += qf[e] * qf[e];
                qn[g] = sqrtf(group_sum<LPR>(ss));
            }
        };
        // row r of level l's rows of the batch: which heads pass, and is there a node at all
        auto judge = [&](int l, int rows, int r, const uint4& raw, float rad) {
            unsigned pass = 0;
    #pragma unroll
            for (int g = 0; g < GMAX; ++g) {
                const float d = group_sum<LPR>(chunk_dot<T>(raw, qraw[g]));
                if (d + qn[g] * rad >= tau[g]) pass |= 1u << g;
            }
            if (ch == 0 && r < rows) s_pass[l][r] = pass | (rad > -INFINITY ? 0x80000000u : 0u);
        };
        auto ask = [&](int l, int first, int rows, int r, uint4& raw, float& rad) {
            raw = make_uint4(0, 0, 0, 0);
            rad = -INFINITY;
            if (r < rows) {
                const size_t t0 = (size_t)tree * p.cap[l];
                if (chunk_ok) raw = load_row_chunk<T>(p.centers[l], p.layout, D, t0, first + r, ch);
                rad = p.radii[l][t0 + first + r];
            }
        };
        // a level-1 node, lane `lane` of the batch: a node counts where a head is alive above it, by its
        // first level-1 descendant
        auto count_nodes = [&](int n0) {
            unsigned a = gmask;
            for (int l = L - 1; l >= 1; --l) {
                unsigned id = (unsigned)(n0 + lane), fl = (unsigned)n0;
                bool lead = true;
                for (int i = 1; i < l; ++i) {
                    const unsigned up = over_bf(id);
                    lead = lead && up * (unsigned)p.bf == id;
                    id = up;
                    fl = over_bf(fl);
                }
                const uint32_t w = s_pass[l][id - fl];
                if (a && (w >> 31) && lead) count(l, 1);
                a &= w;
            }
        };
        const int n0 = node_first, nb = node_last - node_first;  // (never empty, kBatch at most)
        const int cc = chunk_ok ? ch : 0;
        auto row_at = [&](const void* base, int layout, size_t row0, int row) {
            const T* b = reinterpret_cast<const T*>(base) + row0 * (size_t)D;
            const size_t at = sizeof(T) == 4 || layout == HIRA_ROW_MAJOR ? (size_t)row * D + cc * EPL
                                                                         : elem_index(HIRA_TILE16, D, (size_t)row, cc * EPL);
            return *reinterpret_cast<const uint4*>(b + at);
        };
        const uint4 none = make_uint4(0, 0, 0, 0);
        // gates: rows of levels 1 and 2 over all waves, every level above on a wave of its own; a row that
        // is not there is the last one again, a level that is not there level 1
        constexpr int KA = kOneGateRows;
        const int r0 = wave * RPW + rg, rstep = nwaves * RPW;
        const int l3w = 2 + (wave == 0 ? nwaves : wave), l3 = l3w < L ? l3w : 1;
        const int at2 = L > 2 ? 1 : 0, at3 = l3w < L ? 2 : 0;  // theirs of va
        int first2 = 0, rows2 = 0, first3 = 0, rows3 = 0, cnt = 0;
        uint4 raw1[KA], raw2 = none, raw3 = none, kraw[KU];
        float rad1[KA], rad2 = 0.0f, rad3 = 0.0f;
        const int i0 = wave * ROWS, wg_rows = nb * block_rows;  // my block's first row
        const int slot0 = n0 * block_rows + i0 + rg;
        if (real_nodes) {  // uniform
            first2 = (int)over_bf((unsigned)n0);
            int last2 = (int)over_bf((unsigned)(n0 + nb - 1));
            rows2 = L > 2 ? last2 - first2 + 1 : 0;
            first3 = first2;
            int last3 = last2;
            for (int l = 3; l <= l3; ++l) {
                first3 = (int)over_bf((unsigned)first3);
                last3 = (int)over_bf((unsigned)last3);
            }
            rows3 = l3w < L ? last3 - first3 + 1 : 0;
            const size_t t1 = (size_t)tree * va.level_cap[0], t2 = (size_t)tree * va.level_cap[at2], t3 = (size_t)tree * va.level_cap[at3];
            const float *radii1 = va.radii[0], *radii2 = va.radii[at2],
                        *radii3 = va.radii[at3];
#pragma unroll
            for (int k = 0; k < KA; ++k) {
                const int row = n0 + min(r0 + k * rstep, nb - 1);
                raw1[k] = row_at(va.centers[0], va.layout, t1, row);
                rad1[k] = radii1[t1 + row];
            }
            const int row2 = rows2 > 0 ? first2 + min(r0, rows2 - 1) : 0;
            raw2 = row_at(va.centers[at2], va.layout, t2, row2);
            rad2 = radii2[t2 + row2];
            const int row3 = rows3 > 0 ? first3 + min(rg, rows3 - 1) : 0;
            raw3 = row_at(va.centers[at3], va.layout, t3, row3);
            rad3 = radii3[t3 + row3];
            cnt = va.counts[t1 + n0 + min(lane, nb - 1)];
        }
#pragma unroll
        for (int u = 0; u < KU; ++u) kraw[u] = row_at(kbase, klayout, krow0, min(slot0 + u * RPW, n_rows - 1));
        __builtin_amdgcn_sched_barrier(0);  // (nothing that uses a load moves above this line)
        queries();
        if constexpr (SAMPLED) {
            if (real_nodes) {  // uniform
                if (wave == 0)
                    threshold_join<LPR, (GMAX < 4 ? 4 : GMAX)>(p.sample, p.sample_rows, p.q, tree, hoff, G, p.sample_k, p.sample_best,
                                                               p.sample_wait, s_tau, s_scores);
                __syncthreads();
                if (wg == 0 && wave == 0 && lane < G) const_cast<float*>(p.tau)[hoff + lane] = s_tau[lane];
#pragma unroll
                for (int g = 0; g < GMAX; ++g) tau[g] = s_tau[min(g, G - 1)];
#pragma unroll
                for (int i = 0; i < KEPT; ++i) my_tau[i] = s_tau[min(my_g + i % GMAX, G - 1)];
            }
        }
        unsigned alive = gmask;
        if (real_nodes) {  // uniform
            if (wave * RPW < rows2) judge(2, rows2, r0, chunk_ok ? raw2 : none, rad2);  // (uniform in the wave)
            if (rows3 > 0) judge(l3, rows3, rg, chunk_ok ? raw3 : none, rad3);
#pragma unroll
            for (int k = 0; k < KA; ++k)
                if (wave * RPW + k * rstep < nb) judge(1, nb, r0 + k * rstep, chunk_ok ? raw1[k] : none, rad1[k]);
#pragma unroll 1
            for (int r = r0 + rstep; r - rg < rows2; r += rstep) {  // (fan-outs of two or three)
                ask(2, first2, rows2, r, raw2, rad2);
                judge(2, rows2, r, raw2, rad2);
            }
#pragma unroll 1
            for (int r = rg + RPW; r - rg < rows3; r += RPW) {
                ask(l3, first3, rows3, r, raw2, rad2);
                judge(l3, rows3, r, raw2, rad2);
            }
            __syncthreads();
            // a node is alive for the heads that it and all its ancestors pass for (every wave for itself: no
            // second barrier)
            alive = lane < nb && cnt > 0 ? gmask & s_pass[1][lane] : 0u;
            unsigned id = (unsigned)(n0 + min(lane, nb - 1)), fl = (unsigned)n0;
#pragma unroll 1
            for (int l = 2; l < L; ++l) {
                id = over_bf(id);
                fl = over_bf(fl);
                alive &= s_pass[l][id - fl];
            }
            if (p.stats && wave == 0) {
                if (lane < nb) count_nodes(n0);
                if (alive) count(0, (unsigned)cnt);
            }
        }
        if (i0 < wg_rows) {  // uniform in the wave
            int slot[KU];
#pragma unroll
            for (int u = 0; u < KU; ++u) {
                slot[u] = min(slot0 + u * RPW, n_rows - 1);
                if (!chunk_ok) kraw[u] = none;
            }
            take(kraw, slot, [&](int& my_slot, bool& my_row) -> unsigned {
                const int row = i0 + my_u * RPW + rg, k = (int)(((float)row + 0.5f) * inv_rows);
                const int node = __shfl((int)(alive | ((unsigned)cnt << 16)), min(k, 63), 64);
                my_slot = n0 * block_rows + row;
                my_row = row < wg_rows && my_slot < n_rows;
                if (!real_nodes) return my_row ? gmask : 0u;
                return my_row && row - k * block_rows < (node >> 16) ? (unsigned)node & 0xFFFFu : 0u;
            });
        }
    } else {
    for (int n0 = node_first; n0 < node_last; n0 += kBatch) {  // uniform in the workgroup
        const int nb = min(kBatch, node_last - n0);
        if (n0 > node_first) __syncthreads();  // (the list of the batch before is done with)
        int cnt = 0;  // child count of node n0 + thread
        if ((int)threadIdx.x < nb)
            cnt = real_nodes ? p.counts[1][(size_t)tree * p.cap[1] + n0 + threadIdx.x]
                             : min(kPseudoBlock, n_rows - (n0 + (int)threadIdx.x) * kPseudoBlock);
        // ---- gates: rows of levels 1 and 2 over all waves, every level above on a wave of its own ----
        if (real_nodes) {
            constexpr int KA = 4;  // level-1 rows a lane group has in flight
            const int rb0 = wave * RPW, rstep = nwaves * RPW;
            // A lane group's row of those that the wave asks for, from number rb on, the last one again where there is none.  (Under a
            // condition of the lanes' own every row held registers of zeros, and level 2 was asked for when level 1 had arrived.
            // Searches of 8 x 60000 rows of 128 fp32 27.1 -> 26.6 us, 8 x 20000 15.1 -> 14.75, 8 x 90000 bf16 at a fan-out of 8 25.0 ->
            // 24.55; attention over 16 trees x 19889 x 96 bf16, seven heads 64.4 -> 61.6, 4 x 30000 x 32 at a fan-out of 4, eight
            // heads 27.8 -> 25.4: these were short of registers.)
            auto ask = [&](int l, int first, int rows, int rb, uint4& raw, float& rad) {
                if (rb < rows) {  // uniform in the wave
                    const size_t t0 = (size_t)tree * p.cap[l];
                    const int row = first + min(rb + rg, rows - 1);
                    raw = load_row_chunk<T>(p.centers[l], p.layout, D, t0, row, chunk_ok ? ch : 0);
                    rad = p.radii[l][t0 + row];
                }
            };
            uint4 raw1[KA], raw2 = make_uint4(0, 0, 0, 0);
            float rad1[KA], rad2 = 0.0f;
#pragma unroll
            for (int k = 0; k < KA; ++k) {
                raw1[k] = raw2, rad1[k] = rad2;
                ask(1, n0, nb, rb0 + k * rstep, raw1[k], rad1[k]);
            }
            const int first2 = (int)over_bf((unsigned)n0);
            const int rows2 = L > 2 ? (int)over_bf((unsigned)(n0 + nb - 1)) - first2 + 1 : 0;
            ask(2, first2, rows2, rb0, raw2, rad2);
            __builtin_amdgcn_sched_barrier(0);  // (nothing that uses a load moves above this line)
            // (nor do the queries' norms leave the loop, to be waited for ahead of it)
#pragma unroll
            for (int g = 0; g < GMAX; ++g) asm volatile("" : "+v"(qraw[g].x), "+v"(qraw[g].y), "+v"(qraw[g].z), "+v"(qraw[g].w));
            float qn[GMAX];
#pragma unroll
            for (int g = 0; g < GMAX; ++g) {
                if (!chunk_ok) qraw[g] = make_uint4(0, 0, 0, 0);
                float qf[EPL], ss = 0.0f;
                unpack<T>(qraw[g], qf);
#pragma unroll
                for (int e = 0; e < EPL; ++e) ss += qf[e] * qf[e];
                qn[g] = sqrtf(group_sum<LPR>(ss));
            }
            auto judge = [&](int l, int rows, int rb, const uint4& raw, float rad) {
                const int r = rb + rg;
                const uint4 x = chunk_ok ? raw : make_uint4(0, 0, 0, 0);
                unsigned pass = 0;
#pragma unroll
                for (int g = 0; g < GMAX; ++g) {
                    const float d = group_sum<LPR>(chunk_dot<T>(x, qraw[g]));
                    if (d + qn[g] * rad >= tau[g]) pass |= 1u << g;
                }
                if (ch == 0 && r < rows) s_pass[l][r] = pass | (rad > -INFINITY ? 0x80000000u : 0u);
            };
            if (rb0 < rows2) judge(2, rows2, rb0, raw2, rad2);  // (conditions: uniform in the wave)
#pragma unroll
            for (int k = 0; k < KA; ++k)
                if (rb0 + k * rstep < nb) judge(1, nb, rb0 + k * rstep, raw1[k], rad1[k]);
#pragma unroll 1
            for (int rb = rb0 + rstep; rb < rows2; rb += rstep) {  // (fan-outs of one or two)
                ask(2, first2, rows2, rb, raw2, rad2);
                judge(2, rows2, rb, raw2, rad2);
            }
#pragma unroll 1
            for (int rb = rb0 + KA * rstep; rb < nb; rb += rstep) {  // (small workgroups)
                ask(1, n0, nb, rb, raw2, rad2);
                judge(1, nb, rb, raw2, rad2);
            }
            int fl = first2, ll = first2 + rows2 - 1;  // first and last row of level l - 1
#pragma unroll 1
            for (int l = 3; l < L; ++l) {
                fl = (int)over_bf((unsigned)fl);
                ll = (int)over_bf((unsigned)ll);
                if ((l - 2) % nwaves != wave) continue;
                const int rows = ll - fl + 1;
#pragma unroll 1
                for (int rb = 0; rb < rows; rb += RPW) {
                    ask(l, fl, rows, rb, raw2, rad2);
                    judge(l, rows, rb, raw2, rad2);
                }
            }
        } else {
#pragma unroll
            for (int g = 0; g < GMAX; ++g)
                if (!chunk_ok) qraw[g] = make_uint4(0, 0, 0, 0);
        }
        // The dense output's stretch under the batch starts out as the fill value; the scores of
        // selected keys follow behind the barriers.
        if (p.dense_fill && !is_queue) {
            const int f0 = n0 * block_rows, f1 = min((n0 + nb) * block_rows, n_rows);
#pragma unroll
            for (int g = 0; g < GMAX; ++g)
                if (g < G) {
                    float* row = p.dense + (int64_t)head_of(g) * p.dense_stride;
                    for (int i = f0 + (int)threadIdx.x; i < f1; i += blockDim.x) row[i] = p.dense_fill_value;
                }
        }
        __syncthreads();
        // ---- list ---------------------------------------------------------------------------
        if (wave == 0) {
            unsigned alive = lane < nb ? gmask : 0u;
            if (real_nodes && lane < nb) {
                alive &= s_pass[1][lane];
                int at = lane, below = n0;  // place of my ancestor in the batch, first row of the level below
#pragma unroll 1
                for (int l = 2; l < L; ++l) {
                    const int fl = (int)over_bf((unsigned)below);
                    // (places inside the batch are small: the float quotient is exact)
                    at = (int)(((float)(below - fl * p.bf + at) + 0.5f) * inv_rows);
                    alive &= s_pass[l][at];
                    below = fl;
                }
                if (p.stats) {
                    // a node counts where a head is alive above it, by its first level-1 descendant
                    unsigned a = gmask;
                    for (int l = L - 1; l >= 1; --l) {
                        unsigned id = (unsigned)(n0 + lane), fl = (unsigned)n0;
                        bool lead = true;
                        for (int i = 1; i < l; ++i) {
                            const unsigned up = over_bf(id);
                            lead = lead && up * (unsigned)p.bf == id;
                            id = up;
                            fl = over_bf(fl);
                        }
                        const uint32_t w = s_pass[l][id - fl];
                        if (a && (w >> 31) && lead) count(l, 1);
                        a &= w;
                    }
                }
            }
            if (cnt <= 0) alive = 0u;
            if (p.stats && alive) count(0, (unsigned)cnt);
            const unsigned long long bal = __ballot(alive != 0u);
            if (alive) s_list[__popcll(bal & ((1ull << lane) - 1ull))] = (uint32_t)lane | ((uint32_t)cnt << 8) | (alive << 16);
            if (lane == 0) s_count = __popcll(bal);
        }
        __syncthreads();
        // ---- scan ---------------------------------------------------------------------------
        const int nrows = s_count * block_rows;
        // row `row` of the survivors' rows: its key slot, the heads it may be selected for (0: none)
        auto row_info = [&](int row, int& slot) -> unsigned {
            // (rows of a batch stay far below 2^22: the float quotient is exact enough)
            const int k = min((int)(((float)row + 0.5f) * inv_rows), kBatch - 1);
            const uint32_t info = row < nrows ? s_list[k] : 0u;
            const int j = row - k * block_rows;
            slot = (n0 + (int)(info & 0xFFu)) * block_rows + j;
            return j < (int)((info >> 8) & 0xFFu) ? info >> 16 : 0u;
        };
#pragma unroll 1
        for (int i0 = wave * ROWS; i0 < nrows; i0 += nwaves * ROWS) {
            uint4 raw[KU];
            int slot[KU];
#pragma unroll
            for (int u = 0; u < KU; ++u) {
                const unsigned am = row_info(i0 + u * RPW + rg, slot[u]);
                raw[u] = make_uint4(0, 0, 0, 0);
                if (am != 0u && chunk_ok) raw[u] = load_row_chunk<T>(kbase, klayout, D, krow0, slot[u], ch);
            }
            take(raw, slot, [&](int& my_slot, bool&) { return row_info(i0 + my_u * RPW + rg, my_slot); });
        }
    }
    }  // ONE or loops

    if (!want_attn) return;  // uniform

    // ---- merge the lane groups of the wave, then the waves of the workgroup (a wave, or a
    // workgroup, without a selected key for a head only says so) -------------------------------
    float* wsm = smem + (size_t)wave * GMAX * (DVP + 2);
    l_run = cross_group_sum<GMAX>(l_run);
    if (lane < GMAX) {
        wsm[lane * (DVP + 2) + DVP] = m_run;
        wsm[lane * (DVP + 2) + DVP + 1] = l_run;
    }
#pragma unroll
    for (int g = 0; g < GMAX; ++g) {
        if (__int_as_float(__builtin_amdgcn_readlane(__float_as_int(m_run), g)) == -INFINITY) continue;  // uniform
#pragma unroll
        for (int e = 0; e < EPL; ++e) {
            const float a = cross_group_sum<LPR>(acc[g][e]);
            if (rg == 0) wsm[g * (DVP + 2) + ch * EPL + e] = a;
        }
    }
    __syncthreads();
    const float inv_dv = 1.0f / (float)Dv;  // (quotients below some thousands: exact)
    for (int t = threadIdx.x; t < G * Dv; t += blockDim.x) {
        const int g = (int)(((float)t + 0.5f) * inv_dv), e = t - g * Dv;
        // (what every wave has, read at once: one wave's after the other's was a chain of 16 reads, and with the fold's
        // maxima asked for twice 0.3 us of 15.9 at 4 trees x 5003 rows of 80 columns, 3 heads each)
        float mw[WAVES], aw[WAVES], lw[WAVES], mall = -INFINITY;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
            const float* ws = smem + ((size_t)min(w, nwaves - 1) * GMAX + g) * (DVP + 2);
            mw[w] = w < nwaves ? ws[DVP] : -INFINITY;
            aw[w] = ws[e];  // (anything, where the wave has no selected key)
            lw[w] = ws[DVP + 1];
        }
#pragma unroll
        for (int w = 0; w < WAVES; ++w) mall = fmaxf(mall, mw[w]);
        float a = 0.0f, lsum = 0.0f;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
            const float f = exp2f(mw[w] - mall);
            if (mw[w] != -INFINITY) {
                a += aw[w] * f;
                lsum += lw[w] * f;
            }
        }
        const size_t slot = (size_t)head_of(g) * p.num_parts + wg;
        // device-scope stores: written through, so that the workgroup that folds the partials
        // (maybe behind another L2) reads them without cache-wide flushes
        if (mall > -INFINITY)
            __hip_atomic_store(&p.part_acc[slot * Dv + e], a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (e == 0) {
            __hip_atomic_store(&p.part_m[slot], mall, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(&p.part_l[slot], lsum, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    if (p.done == nullptr) return;  // the caller folds the partials in a second launch

    // ---- the last workgroup of this tree (and head pass) to arrive folds its partials ----
    __shared__ int s_last;
    hand_off_release();
    __syncthreads();
    if constexpr (SAMPLED) {
        if (wave == 0) {
            const bool last = sampled_ticket(p, tree, wgs, hoff, G);
            if (lane == 0) s_last = last;
        }
    } else if (threadIdx.x == 0) {
        int* ctr = p.done + (size_t)tree * gridDim.z + blockIdx.z;
        const int ticket = __hip_atomic_fetch_add(ctr, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        s_last = ticket == (int)gridDim.x - 1;
        if (s_last) __hip_atomic_store(ctr, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!s_last) return;
    fold_heads(p, hoff, G, smem);
}

template <typename T, int LPR, int GMAX>
inline void launch_search(const SearchPlan& plan, const SearchParams& p, dim3 grid, hipStream_t s) {
    const size_t smem = p.part_acc ? plan.smem : 0;
    const dim3 block(plan.threads);
    // (a block of the larger kind holds more scores a lane than eight heads leave registers for)
    if constexpr (sizeof(T) == 2 && (LPR == 8 || LPR == 16)) {
        if (p.sample_wgs > 0) {
            if (plan.ahead == kOneSmall) hipLaunchKernelGGL((search_kernel<T, LPR, GMAX, kOneSmall, true>), grid, block, smem, s, p);
            else hipLaunchKernelGGL((search_kernel<T, LPR, GMAX, (GMAX <= 4 ? kOneLarge : kOneSmall), true>), grid, block, smem, s, p);
            return;
        }
    }
    if (plan.ahead == kOneSmall) hipLaunchKernelGGL((search_kernel<T, LPR, GMAX, kOneSmall>), grid, block, smem, s, p);
    else if (plan.ahead) hipLaunchKernelGGL((search_kernel<T, LPR, GMAX, (GMAX <= 4 ? kOneLarge : kOneSmall)>), grid, block, smem, s, p);
    else hipLaunchKernelGGL((search_kernel<T, LPR, GMAX, 0>), grid, block, smem, s, p);
}

template <typename T, int LPR>
inline void launch_search(const SearchPlan& plan, const SearchParams& p, dim3 grid,
                          hipStream_t s) {
    switch (plan.gmax) {
        case 1: launch_search<T, LPR, 1>(plan, p, grid, s); break;
        case 4: launch_search<T, LPR, 4>(plan, p, grid, s); break;
        default: launch_search<T, LPR, 8>(plan, p, grid, s); break;
    }
}

template <typename T>
inline int dispatch_lpr(const SearchPlan& plan, const SearchParams& p, dim3 grid,
                        hipStream_t s) {
    switch (plan.lpr) {
        case 2: launch_search<T, 2>(plan, p, grid, s); break;
        case 4: launch_search<T, 4>(plan, p, grid, s); break;
        case 8: launch_search<T, 8>(plan, p, grid, s); break;
        case 16: launch_search<T, 16>(plan, p, grid, s); break;
        case 32: launch_search<T, 32>(plan, p, grid, s); break;
        case 64: launch_search<T, 64>(plan, p, grid, s); break;
        default: return fail(HIRA_EINVAL, "unsupported row width");
    }
    return HIRA_OK;
}

#undef VEC_ARG

}  // namespace hira
