// The threshold kernel's device code (see threshold.hip for what it computes), as the work of
// one workgroup: the kernel of hira_threshold runs it in every workgroup, the kernel of
// hira_update_threshold in the workgroups behind those that append.
#pragma once
#include <type_traits>

#include "search.h"

namespace hira {

constexpr int kTauThreads = 1024;
constexpr int kTauWaves = kTauThreads / 64;
constexpr int kTauMaxSamples = 4096;
constexpr int kTauRows = 16;  // sample rows a lane group has in flight

__device__ __forceinline__ float tau_block_reduce(float v, bool is_max, float* s_red) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    v = is_max ? wave_max(v) : wave_sum(v);
    if (lane == 0) s_red[wave] = v;
    __syncthreads();
    float r = s_red[0];
#pragma unroll
    for (int w = 1; w < kTauWaves; ++w) r = is_max ? fmaxf(r, s_red[w]) : r + s_red[w];
    return r;
}

constexpr int kTauSorters = 256;  // threads that hold the scores during the sort

// The value that lane ^ J holds: moves inside a row of 16 lanes (J < 16) are data-path moves,
// J = 16 and 32 swaps of rows and halves.  rot4_first: which rotation by 4 brings lane ^ 4.
template <int J>
__device__ __forceinline__ float tau_partner(float v, bool rot4_first) {
    if constexpr (J >= 16) {  // a swap leaves the lower and the upper row's (half's) value in either
        const auto r = J == 32 ? __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false)
                               : __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
        return __uint_as_float((threadIdx.x & J) != 0 ? r[0] : r[1]);
    } else if constexpr (J == 8) {
        return dpp_move<0x128>(v);  // row rotate by 8
    } else if constexpr (J == 4) {
        const float a = dpp_move<0x124>(v), b = dpp_move<0x12C>(v);  // by 4, by 12
        return rot4_first ? a : b;
    } else if constexpr (J == 2) {
        return dpp_move<0x4E>(v);  // quad [2,3,0,1]
    } else {
        return dpp_move<0xB1>(v);  // quad [1,0,3,2]
    }
}

// One merge stage (stretches of LEN, partners J = LEN/2 .. 1) of a wave's 64 values, one a lane,
// largest first in the end (the last stage sorts the whole wave one way).
template <int LEN, int J>
__device__ __forceinline__ void tau_wave_stage(float& x, int ln, bool rot4_first) {
    const float o = tau_partner<J>(x, rot4_first);
    const bool down = (ln & LEN) == 0 || LEN == 64, lower = (ln & J) == 0;
    x = (down == lower) ? fmaxf(x, o) : fminf(x, o);
    if constexpr (J > 1) tau_wave_stage<LEN, J / 2>(x, ln, rot4_first);
}

// One step of the bitonic sort (largest first) of 256 * EE entries, entry e*256 + tid in v[e]
// of thread tid < 256: entry i meets entry i ^ J; in a stretch that ends up descending
// ((i & LEN) == 0) the lower index keeps the larger value.  Every thread of the workgroup
// calls it (the steps through LDS hold a barrier); only the sorters hold data.
template <int EE, int LEN, int J>
__device__ __forceinline__ void tau_sort_step(float (&v)[EE], float* s0, float* s1, int& buf,
                                              int tid, bool sorter, bool rot4_first) {
    constexpr int ST = kTauSorters;
    if constexpr (J >= ST) {  // partner in another register of this thread
        constexpr int JE = J / ST;
        if (!sorter) return;
#pragma unroll
        for (int e = 0; e < EE; ++e) {
            if ((e & JE) == 0 && (e | JE) < EE) {
                const bool down = (((e * ST) & LEN) == 0);
                const float lo = v[e], hi = v[e | JE];
                const bool swap = down ? lo < hi : lo > hi;
                v[e] = swap ? hi : lo;
                v[e | JE] = swap ? lo : hi;
            }
        }
    } else {
        auto meet = [&](int e, float o) {
            const int i = e * ST + tid;
            const bool down = (i & LEN) == 0, lower = (i & J) == 0;
            v[e] = (down == lower) ? fmaxf(v[e], o) : fminf(v[e], o);
        };
        if constexpr (J >= 64) {  // partner in another wave
            float* sb = buf ? s1 : s0;
            if (sorter) {
#pragma unroll
                for (int e = 0; e < EE; ++e) sb[e * ST + tid] = v[e];
            }
            __syncthreads();
            if (sorter) {
#pragma unroll
                for (int e = 0; e < EE; ++e) meet(e, sb[e * ST + (tid ^ J)]);
            }
            buf ^= 1;  // the next exchange writes the other half: one barrier per step
        } else if (!sorter) {
            // (whole waves: the steps inside a wave are not theirs to spend issue slots on)
        } else if constexpr (J >= 16) {
#pragma unroll
            for (int e = 0; e < EE; ++e) meet(e, tau_partner<J>(v[e], rot4_first));
        } else if constexpr (J == 8) {
#pragma unroll
            for (int e = 0; e < EE; ++e) meet(e, dpp_move<0x128>(v[e]));  // row rotate by 8
        } else if constexpr (J == 4) {
#pragma unroll
            for (int e = 0; e < EE; ++e) {
                const float a = dpp_move<0x124>(v[e]), b = dpp_move<0x12C>(v[e]);  // by 4, by 12
                meet(e, rot4_first ? a : b);
            }
        } else if constexpr (J == 2) {
#pragma unroll
            for (int e = 0; e < EE; ++e) meet(e, dpp_move<0x4E>(v[e]));  // quad [2,3,0,1]
        } else {
#pragma unroll
            for (int e = 0; e < EE; ++e) meet(e, dpp_move<0xB1>(v[e]));  // quad [1,0,3,2]
        }
    }
}

// All steps from (LEN = 2^LL, J = 2^JJ) on, in order.
template <int EE, int LOGN, int LL, int JJ>
struct TauSortFrom {
    static __device__ __forceinline__ void run(float (&v)[EE], float* s0, float* s1, int& buf,
                                               int tid, bool sorter, bool rot4_first) {
        tau_sort_step<EE, (1 << LL), (1 << JJ)>(v, s0, s1, buf, tid, sorter, rot4_first);
        if constexpr (JJ > 0)
            TauSortFrom<EE, LOGN, LL, JJ - 1>::run(v, s0, s1, buf, tid, sorter, rot4_first);
        else if constexpr (LL < LOGN)
            TauSortFrom<EE, LOGN, LL + 1, LL>::run(v, s0, s1, buf, tid, sorter, rot4_first);
    }
};

// Scores of the kTauThreads sample rows from r0 on, one a thread, bf16 rows of 8 * LPR columns: LPR lanes hold a row
// in 16-byte chunks, LPR passes of kTauThreads / LPR rows are on their way at once, two products an instruction
// (v_dot2_f32_bf16: fp32 sums, error against 64 bits 0.96 of a chain of fmas' over 128 normal columns, 0.75 with some of
// them twenty times as large), and the sums over the lanes halve in number as they go, so that lane i ends with pass
// i's row.  With an fma a product, a sum over all lanes a row and the scores through LDS a wave has some 400 vector
// instructions and not 130, four waves a SIMD: a launch of 32 heads, 1000 samples of 128 columns 8.8 us, now
// 6.2 (with the merge below), 8 heads, 64 columns 8.7, now 5.1.  What bounds it is the launch, one trip to memory
// and 256 KB through a compute unit's L1 at 64 bytes a clock, 1.8 us.
// (On the matrix cores, rows as the A operand, a load is half lines of sixteen rows, and what is on its way is
// more than the L1: 11.2 us.)
// Loads: buffer loads, the tree's sample behind one scalar descriptor, the pass in a scalar offset, one
// address register for all of them.  The range check of a buffer load looks at the vector offset only, so the
// scalar one must stay inside the sample by itself: a pass that reaches past the end is moved back to end with
// the sample, and its rows that an earlier pass has are none here (row -1, score -INFINITY).
// (Workgroups of NT threads, at most 1024, score NT rows at a time.)
template <int LPR, int NT = kTauThreads>
__device__ __forceinline__ float tau_dot_scores(const void* xs, const void* qh, int r0, int S, bool rot4_first, int& row) {
    typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    constexpr int D = 8 * LPR, PASS = NT / LPR;
    const int tid = threadIdx.x, sub = tid % LPR, grp = tid / LPR;
    const __amdgpu_buffer_rsrc_t rsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(xs), 0, S * D * 2, 0x00020000);
    const unsigned voff = (unsigned)(grp * D + sub * 8) * 2u;
    const int last_pass = max(S - PASS, 0);
    u32x4 raw[LPR];
#pragma unroll
    for (int u = 0; u < LPR; ++u) {
        raw[u] = u32x4{0, 0, 0, 0};
        if (r0 + u * PASS < S)  // uniform
            raw[u] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, voff, (unsigned)(min(r0 + u * PASS, last_pass) * (D * 2)), 0);
    }
    const u32x4 b = reinterpret_cast<const u32x4*>(qh)[sub];
    float dot[LPR];
#pragma unroll
    for (int u = 0; u < LPR; ++u) {
        float d = 0.0f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const uint32_t x = raw[u][e], y = b[e];  // (an element of a vector cannot be bit-cast where it is)
            d = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, x), __builtin_bit_cast(bf16x2, y), d, false);
        }
        dot[u] = d;
    }
    auto halve = [&](auto step) {
        constexpr int J = decltype(step)::value;
        const bool high = (sub & J) != 0;
#pragma unroll
        for (int u = 0; u < J; ++u) {
            const float keep = high ? dot[u + J] : dot[u], give = high ? dot[u] : dot[u + J];
            dot[u] = keep + tau_partner<J>(give, rot4_first);
        }
    };
    if constexpr (LPR == 16) halve(std::integral_constant<int, 8>{});
    halve(std::integral_constant<int, 4>{});
    halve(std::integral_constant<int, 2>{});
    halve(std::integral_constant<int, 1>{});
    const int base = r0 + sub * PASS;
    row = min(base, last_pass) + grp;
    if (base >= S || row < base || row >= S) row = -1;
    return row >= 0 ? dot[0] : -INFINITY;
}

// The 16 largest of two rows of 16 lanes, each sorted largest first, sorted the same way.
__device__ __forceinline__ float tau_merge16(float a, float b, int ln, bool rot4_first) {
    float m = fmaxf(a, dpp_move<0x140>(b));  // (the row mirrored)
    auto step = [&](float o, bool lower) { m = lower ? fmaxf(m, o) : fminf(m, o); };
    step(tau_partner<8>(m, rot4_first), (ln & 8) == 0);
    step(tau_partner<4>(m, rot4_first), (ln & 4) == 0);
    step(tau_partner<2>(m, rot4_first), (ln & 2) == 0);
    step(tau_partner<1>(m, rot4_first), (ln & 1) == 0);
    return m;
}

// A wave's 64 values, one a lane, sorted largest first.
__device__ __forceinline__ float tau_wave_sort(float x, int ln, bool rot4) {
    tau_wave_stage<2, 1>(x, ln, rot4);
    tau_wave_stage<4, 2>(x, ln, rot4);
    tau_wave_stage<8, 4>(x, ln, rot4);
    tau_wave_stage<16, 8>(x, ln, rot4);
    tau_wave_stage<32, 16>(x, ln, rot4);
    tau_wave_stage<64, 32>(x, ln, rot4);
    return x;
}

// ---- thresholds in the launch that searches with them -------------------------------------------------
// A search of few workgroups needs its thresholds only where its gates are compared, some 2.5 us after its start,
// and a launch ahead of it is one more for the host and the queue.  So the first workgroups of the search's launch
// score the sample, kTauStretch rows of a tree for a head each, and leave the stretch's 16 best in memory; every
// workgroup of higher number looks for them behind its own loads (threshold_join).  Only those wait, for ones
// that never do.  Up to kTauFewRows sample rows, the mean of at most 16 best, bf16 rows of 64 or 128 columns; the
// arithmetic is threshold_block's, the same bits.
// us, two launches / this, 8 trees x 4 heads, 1000 samples: 4001 rows of 128 columns 15.0 / 12.3 (waiting for a
// counter and then asking for the scores 15.3), 8000 16.6 / 13.6, 1000 14.0 / 11.0, 4001 x 64 13.0 / 10.8;
// 8 heads a tree 16.9 / 14.4; 300 rows, as many samples 12.0 / 9.4; on the vector units 2 trees x 4 heads,
// 1111 rows of 64 columns in five levels 15.4 / 12.5.  What bounds it is the chain: arguments, one trip and
// half the sample through a compute unit's L1, the sorts (some 6 us from the start), two trips of the hand-over,
// then the search from its gates on.
//   best    (H_q, 2, 16) scores, largest first; 0 between launches, which says: not there yet (a score of 0 is
//           left as -0, which adds up to the same).  So what is waited for is the scores themselves; behind a
//           counter, two trips later, nothing was won
//   ready   the tree's arrival counter: tickets of the searching workgroups in the low half, finished stretches in
//           the high half.  Whoever comes last of all sets it and `best` back to zero (threshold_reset)
constexpr int kTauFewRows = 1024, kTauStretch = 512;
constexpr int kTauMade = 1 << 16;

// By one wave: the tree's thresholds are used by all, its counter and its n words of `best` go back to zero.
__device__ __forceinline__ void threshold_reset(float* best, int n, int* ready) {
    for (int i = threadIdx.x & 63; i < n; i += 64) __hip_atomic_store(best + i, 0.0f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if ((threadIdx.x & 63) == 0) __hip_atomic_store(ready, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// heads: of a tree; all: the counter's value behind the last of all
template <int LPR>
__device__ __forceinline__ void threshold_stretch(const void* samples, int S, const void* q, int tree, int heads, int index,
                                                  float* best, float* lds, int* ready, int all) {
    const int head = tree * heads + index % heads, stretch = index / heads;
    constexpr int D = 8 * LPR;
    const int ln = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const bool rot4 = __builtin_amdgcn_update_dpp(0, ln, 0x124, 0xF, 0xF, true) == (ln ^ 4);
    const uint16_t* xs = reinterpret_cast<const uint16_t*>(samples) + (size_t)tree * S * D;
    const uint16_t* qh = reinterpret_cast<const uint16_t*>(q) + (size_t)head * D;
    int row;
    const float x = tau_wave_sort(tau_dot_scores<LPR, kTauStretch>(xs, qh, stretch * kTauStretch, S, rot4, row), ln, rot4);
    if (ln < 16) lds[wv * 16 + ln] = x;  // 8 waves
    __syncthreads();
    if (wv != 0) return;
    float m = tau_merge16(lds[ln], lds[64 + ln], ln, rot4);
    m = tau_merge16(m, tau_partner<16>(m, rot4), ln, rot4);
    m = tau_merge16(m, tau_partner<32>(m, rot4), ln, rot4);
    if (ln < 16)
        __hip_atomic_store(best + (head * 2 + stretch) * 16 + ln, m == 0.0f ? -0.0f : m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // (written through and complete before it is counted: the hand-off of search.h)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    int before = 0;
    if (ln == 0) before = __hip_atomic_fetch_add(ready, kTauMade, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (__builtin_amdgcn_readfirstlane(before) + kTauMade == all) threshold_reset(best + (size_t)tree * heads * 32, heads * 32, ready);
}

// The mean of the k best of every row of 16 lanes, sorted largest first: added up in that order.
__device__ __forceinline__ float tau_row_mean(float m, int k) {
    float sum = 0.0f;
    auto add = [&](auto at) {
        constexpr int R = decltype(at)::value;
        const float v = dpp_move<0x150 + R>(m);  // (lane R of the row to all of it)
        if (R < k) sum += v;                     // uniform
    };
#define HIRA_TAU_ADD(R) add(std::integral_constant<int, R>{})
    HIRA_TAU_ADD(0), HIRA_TAU_ADD(1), HIRA_TAU_ADD(2), HIRA_TAU_ADD(3), HIRA_TAU_ADD(4), HIRA_TAU_ADD(5), HIRA_TAU_ADD(6), HIRA_TAU_ADD(7);
    HIRA_TAU_ADD(8), HIRA_TAU_ADD(9), HIRA_TAU_ADD(10), HIRA_TAU_ADD(11), HIRA_TAU_ADD(12), HIRA_TAU_ADD(13), HIRA_TAU_ADD(14), HIRA_TAU_ADD(15);
#undef HIRA_TAU_ADD
    return sum / (float)k;
}

// The threshold of a head by one wave, slowly and in few registers: for a workgroup that gave up waiting.
// scores: kTauFewRows floats of LDS.
template <int LPR>
__device__ __forceinline__ float threshold_by_wave(const void* samples, int S, const void* q, int tree, int head, int k, float* scores) {
    typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
    constexpr int D = 8 * LPR;
    const int ln = threadIdx.x & 63;
    const uint4* xs = reinterpret_cast<const uint4*>(reinterpret_cast<const uint16_t*>(samples) + (size_t)tree * S * D);
    const uint4* qh = reinterpret_cast<const uint4*>(reinterpret_cast<const uint16_t*>(q) + (size_t)head * D);
#pragma unroll 1
    for (int r = ln; r < S; r += 64) {
        float d[LPR];
#pragma unroll
        for (int c = 0; c < LPR; ++c) {
            const uint4 a = xs[(size_t)r * LPR + c], b = qh[c];
            const uint32_t u[4] = {a.x, a.y, a.z, a.w}, v[4] = {b.x, b.y, b.z, b.w};
            d[c] = 0.0f;
#pragma unroll
            for (int e = 0; e < 4; ++e)
                d[c] = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, u[e]), __builtin_bit_cast(bf16x2, v[e]), d[c], false);
        }
#pragma unroll
        for (int half = LPR / 2; half >= 1; half /= 2)
#pragma unroll
            for (int c = 0; c < half; ++c) d[c] += d[c + half];
        scores[r] = d[0];
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
    float sum = 0.0f;
#pragma unroll 1
    for (int i = 0; i < k; ++i) {  // uniform: the largest one that is left
        float best = -INFINITY;
        int at = -1;
        for (int r = ln; r < S; r += 64) {
            const float v = scores[r];
            if (v > best || at < 0) best = v, at = r;
        }
        const float top = wave_max(best);
        const unsigned long long who = __ballot(at >= 0 && best == top);
        if (ln == __ffsll((long long)who) - 1) scores[at] = -INFINITY;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
        sum += top;
    }
    return sum / (float)k;
}

// By one wave of a workgroup that searches for the G <= GS heads from `head0` on of a tree: their thresholds to
// s_tau, as soon as the stretches are there.  `limit` looks without success: it makes them itself.
// scores: kTauFewRows floats of LDS.
template <int LPR, int GS>
__device__ __forceinline__ void threshold_join(const void* samples, int S, const void* q, int tree, int head0, int G, int k,
                                               const float* best, int limit, float* s_tau, float* scores) {
    const int ln = threadIdx.x & 63;
    float a[GS / 4], b[GS / 4];  // of four heads at a time, a row of 16 lanes each
    bool made = false;
    for (int look = 0; look < limit && !made; ++look) {  // uniform
        made = true;
#pragma unroll
        for (int i = 0; i < GS / 4; ++i) {
            const float* at = best + (head0 + min(4 * i + ln / 16, G - 1)) * 32 + ln % 16;
            a[i] = __hip_atomic_load(at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            b[i] = -INFINITY;
            if (S > kTauStretch) b[i] = __hip_atomic_load(at + 16, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // uniform
        }
#pragma unroll
        for (int i = 0; i < GS / 4; ++i) made = made && __float_as_uint(a[i]) != 0u && __float_as_uint(b[i]) != 0u;
        made = __ballot(!made) == 0ull;
    }
    if (made) {
        const bool rot4 = __builtin_amdgcn_update_dpp(0, ln, 0x124, 0xF, 0xF, true) == (ln ^ 4);
#pragma unroll
        for (int i = 0; i < GS / 4; ++i) {
            const float tau = tau_row_mean(tau_merge16(a[i], b[i], ln, rot4), k);
            if (ln % 16 == 0 && 4 * i + ln / 16 < G) s_tau[4 * i + ln / 16] = tau;
        }
    } else {
        for (int g = 0; g < G; ++g) {  // uniform
            const float tau = threshold_by_wave<LPR>(samples, S, q, tree, head0 + g, k, scores);
            if (ln == 0) s_tau[g] = tau;
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
}

// The ticket of one of a tree's `wgs` searching workgroups, by its first wave: is it the last of them?  Behind the
// last of all, stretches too, the tree's counter and scores go back to zero.
__device__ __forceinline__ bool sampled_ticket(const SearchParams& p, int tree, int wgs, int head0, int G) {
    int before = 0;
    if ((threadIdx.x & 63) == 0) before = __hip_atomic_fetch_add(p.done + tree, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    before = __builtin_amdgcn_readfirstlane(before);
    if (before + 1 == wgs + p.sample_wgs * kTauMade) threshold_reset(p.sample_best + (size_t)head0 * 32, G * 32, p.done + tree);
    return (before & (kTauMade - 1)) == wgs - 1;
}

// E = registers per thread of the sort: the padded array has 1024 * E entries
// The work of one workgroup of kTauThreads threads: the threshold of the head that place `pos`
// of the launch stands for.
template <typename T, int E>
__device__ __forceinline__ void threshold_block(
    const T* __restrict__ samples, int S, int D, const T* __restrict__ q,
    const int32_t* __restrict__ tree_q_off, const int32_t* __restrict__ tree_q_heads,
    int group_size, int num_trees, int method, int k, float* __restrict__ tau, const int pos) {
    constexpr int EPL = Elem<T>::kPerChunk;
    constexpr int NPAD = kTauThreads * E;
    __shared__ float s_sc[2][NPAD];  // the scores; the two sides of an exchange through LDS
    __shared__ float s_red[kTauWaves];
    const int tid = threadIdx.x;

    // the head of this workgroup and its tree
    int head, tree;
    if (group_size > 0) {
        // trees in the fast index: workgroup i takes head i / T of tree i % T
        tree = pos % num_trees;
        head = tree * group_size + pos / num_trees;
    } else {
        tree = 0;
        while (tree + 1 < num_trees && tree_q_off[tree + 1] <= pos) ++tree;  // uniform
        head = tree_q_heads[pos];
    }

    // ---- few of up to 1024, a score a thread: every wave sorts its 64, largest first; the sixteen best of every
    // wave meet in LDS, and one wave merges them, two sorted rows of 16 lanes at a time, down to sixteen.
    // (Picking the k best of those 256 one maximum at a time: 0.7 us more.)
    auto few_best = [&](float x) {
        const int ln = tid & 63, wv = tid >> 6;
        const bool rot4 = __builtin_amdgcn_update_dpp(0, ln, 0x124, 0xF, 0xF, true) == (ln ^ 4);
        x = tau_wave_sort(x, ln, rot4);
        if (ln < 16) s_sc[1][wv * 16 + ln] = x;
        __syncthreads();
        if (wv != 0) return;
        float c[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) c[e] = s_sc[1][e * 64 + ln];
        float m = tau_merge16(tau_merge16(c[0], c[1], ln, rot4), tau_merge16(c[2], c[3], ln, rot4), ln, rot4);
        m = tau_merge16(m, tau_partner<16>(m, rot4), ln, rot4);
        m = tau_merge16(m, tau_partner<32>(m, rot4), ln, rot4);
        float sum = 0.0f;
        for (int r = 0; r < k; ++r)  // uniform
            sum += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(m), r));
        if (ln == 0) tau[head] = sum / (float)k;
    };
    const T* xs = samples + (size_t)tree * S * D;
    const T* qh = q + (size_t)head * D;
    if (sizeof(T) == 2 && (D == 64 || D == 128)) {
        const int ln = tid & 63;
        const bool rot4 = __builtin_amdgcn_update_dpp(0, ln, 0x124, 0xF, 0xF, true) == (ln ^ 4);
        for (int r0 = 0; r0 < S; r0 += kTauThreads) {  // uniform
            int row;
            const float x = D == 64 ? tau_dot_scores<8>(xs, qh, r0, S, rot4, row) : tau_dot_scores<16>(xs, qh, r0, S, rot4, row);
            if (E == 1 && k <= 16 && method != HIRA_TAU_SAMPLE_MAX) {
                few_best(x);
                return;
            }
            if (row >= 0) s_sc[0][row] = x;
        }
    } else {
    // ---- scores: 16 lanes per sample row, 64 rows per pass, kTauRows passes at a time ---------
    // (buffer loads: the tree's sample behind one scalar descriptor, the pass in a scalar offset,
    // one address register for all the rows a lane has in flight -- which is what lets sixteen of
    // them fit.  The range check of a buffer load looks at the vector offset only, so the scalar
    // one must stay inside the sample by itself: the last pass is moved back to end with the
    // sample and scores some rows a second time; with fewer than 64 rows the vector offset alone
    // says which lanes have none.)
    const int sub = tid & 15, grp = tid >> 4;
    const int chunks = D / EPL;
    constexpr int PASS = kTauThreads / 16;
    const __amdgpu_buffer_rsrc_t xrsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<T*>(xs), 0, (int)((size_t)S * D * sizeof(T)), 0x00020000);
    const int last_pass = max(S - PASS, 0);
    for (int r0 = 0; r0 < S; r0 += PASS * kTauRows) {  // uniform
        float dot[kTauRows];
#pragma unroll
        for (int u = 0; u < kTauRows; ++u) dot[u] = 0.0f;
        for (int c = sub; c < chunks; c += 16) {
            typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
            const unsigned voff = (unsigned)((grp * D + c * EPL) * (int)sizeof(T));
            uint4 raw[kTauRows];
#pragma unroll
            for (int u = 0; u < kTauRows; ++u) {
                raw[u] = make_uint4(0, 0, 0, 0);
                if (r0 + u * PASS < S) {  // uniform
                    const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(
                        xrsrc, voff, (unsigned)(min(r0 + u * PASS, last_pass) * D * (int)sizeof(T)), 0);
                    raw[u] = make_uint4(v.x, v.y, v.z, v.w);
                }
            }
            const uint4 b = load_chunk<T>(qh, 0, c);
#pragma unroll
            for (int u = 0; u < kTauRows; ++u) dot[u] = chunk_dot<T>(raw[u], b, dot[u]);
        }
#pragma unroll
        for (int u = 0; u < kTauRows; ++u) {
            const float d = group_sum<16>(dot[u]);
            const int row = min(r0 + u * PASS, last_pass) + grp;
            if (sub == 0 && r0 + u * PASS < S && row < S) s_sc[0][row] = d;
        }
    }
    }
    __syncthreads();
    // ---- from here on only the first four waves hold data; the others keep the barriers company
    constexpr int ST = kTauSorters;
    constexpr int EE = NPAD / ST;     // entries per sorting thread
    constexpr int LOGN = E == 1 ? 10 : (E == 2 ? 11 : 12);
    const bool sorter = tid < ST;
    float v[EE];
#pragma unroll
    for (int e = 0; e < EE; ++e)
        v[e] = (sorter && e * ST + tid < S) ? s_sc[0][e * ST + tid] : -INFINITY;

    if (method == HIRA_TAU_SAMPLE_MAX) {
        float m = v[0];
#pragma unroll
        for (int e = 1; e < EE; ++e) m = fmaxf(m, v[e]);
        m = tau_block_reduce(m, true, s_red);
        if (tid == 0) tau[head] = m;
        return;
    }

    if (E == 1 && k <= 16) {
        few_best(tid < S ? s_sc[0][tid] : -INFINITY);
        return;
    }

    // ---- bitonic sort, largest first ---------------------------------------------------------
    // Which of the two rotations by 4 inside a row of 16 lanes brings lane ^ 4: asked of the
    // lane numbers themselves.
    const int lane = tid & 63;
    const bool rot4_first =
        __builtin_amdgcn_update_dpp(0, lane, 0x124, 0xF, 0xF, true) == (lane ^ 4);
    int buf = 1;
    TauSortFrom<EE, LOGN, 1, 0>::run(v, s_sc[0], s_sc[1], buf, tid, sorter, rot4_first);
    float sum = 0.0f;
#pragma unroll
    for (int e = 0; e < EE; ++e)
        if (sorter && e * ST + tid < k) sum += v[e];
    sum = tau_block_reduce(sum, false, s_red);
    if (tid == 0) tau[head] = sum / (float)k;
}

// What hira_threshold checks of its arguments before the launch.
static int check_threshold_arguments(const void* samples, int32_t dtype, int32_t num_trees,
                                     int32_t num_samples, int32_t dim, const HiraQuery* query,
                                     int32_t method, int32_t k, const float* tau_out) {
    HIRA_CHECK_ARG(samples && query && tau_out, "hira_threshold: null argument");
    HIRA_CHECK_ARG(dtype == HIRA_F32 || dtype == HIRA_BF16, "hira_threshold: dtype %d", dtype);
    HIRA_CHECK_ARG(num_trees >= 1 && dim >= 1, "hira_threshold: num_trees %d, dim %d", num_trees, dim);
    const int epl = dtype == HIRA_F32 ? 4 : 8;
    HIRA_CHECK_ARG(dim % epl == 0, "hira_threshold: dim %d must be a multiple of %d (16-byte chunks)", dim, epl);
    HIRA_CHECK_ARG(num_samples >= 1 && num_samples <= kTauMaxSamples,
                   "hira_threshold: %d samples per tree (1..%d)", num_samples, kTauMaxSamples);
    HIRA_CHECK_ARG(method == HIRA_TAU_SAMPLE_MAX || method == HIRA_TAU_SAMPLE_MEAN_TOPK,
                   "hira_threshold: method %d", method);
    HIRA_CHECK_ARG(method == HIRA_TAU_SAMPLE_MAX || (k >= 1 && k <= num_samples),
                   "hira_threshold: k = %d with %d samples", k, num_samples);
    HIRA_CHECK_ARG(query->q && query->num_q_heads >= 1, "hira_threshold: query missing");
    if (query->group_size > 0)
        HIRA_CHECK_ARG(query->num_q_heads == num_trees * query->group_size,
                       "hira_threshold: %d heads != %d trees x group of %d", query->num_q_heads,
                       num_trees, query->group_size);
    else
        HIRA_CHECK_ARG(query->tree_q_off && query->tree_q_heads, "hira_threshold: head map missing");
    return HIRA_OK;
}

// registers per thread of the sort for this many samples: the E of threshold_block
static inline int threshold_sort_registers(int num_samples) {
    return num_samples <= kTauThreads ? 1 : (num_samples <= 2 * kTauThreads ? 2 : 4);
}

}  // namespace hira
