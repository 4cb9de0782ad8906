// MFMA search + sparse attention kernel: bf16 keys/centers in the tiled layout
// (HIRA_TILE16), fan-out a multiple of 16, D = Dv in {64, 128, 256}, at least two levels.
//
// One workgroup (8 waves; 256 registers a wave, so the only one on its CU) owns a few
// tiles of 16 level-1 nodes of one tree, a stride apart; workgroup ids run fastest over the trees
// so that, with 8 L2 slices (XCDs) served round-robin, the workgroups of one tree share a
// slice.  After a common gate every wave scans and gathers on its own; the waves meet again
// for the merge:
//   gate   wave w gates the workgroup's tile w: it issues, before it waits for anything, every
//          load it needs (queries, the 16 x D tile of level-1 centres, the tiles holding the
//          tile's ancestors, radii, child counts) and gates with v_mfma_f32_16x16x32_bf16:
//          a wave-wide 128-bit load fetches a 16 x 32 operand tile from 1 KiB of contiguous
//          memory (that is what the tiled layout is for), the B operand holds the (up to 16)
//          query heads of the GQA group, so the D registers hold score(row, head) with
//          head = lane % 16 and row = 4*(lane/16) + j; a node survives for a head when
//          score + ||q|| r >= tau.  Head masks and child counts of the nodes go to LDS.
//   scan   the surviving nodes of these tiles are dealt round-robin to the waves; from here to
//          the merge a wave works on its own (no barrier).  In each round it takes NB of its
//          nodes: their key tiles were requested a round earlier (buffer loads: scalar base and
//          tile offset, no address registers), the B operand now comes from LDS; all products
//          first, then the next round's tiles are requested, then the leaf filter (q.k >= tau
//          against the lane's own threshold).  A tile with a selected row writes the scaled
//          scores of its rows to the wave's stretch of a table in LDS (-inf: not selected) and
//          appends the selected rows to the wave's row list.
//          (A small launch, whose workgroups own one tile: the waves ask for the key tiles of their two
//          nodes each beside the gates' operands, see AHEAD below.)
//   gather the wave raises its running maximum per head, turns the listed scores into weights
//          2^(z - m) with lane = (row, head), and fetches the value rows of its list, kVBatch
//          in flight, each row once however many heads selected it:
//          acc[head][:] += weight(row, head) * v[:] with the accumulators in registers
//          (lane owns Dv/64 columns of every head).
//          (Over an 8-bit shadow, scan and gather are two phases of the workgroup: first all tiles, the rows that
//          the shadow cannot rule out listed; then those rows, dealt out evenly over the waves.)
//   merge  the waves agree on one maximum per head, rescale their sums to it and add them up
//          through LDS.
// Keys queued since the tree was last updated (row-major, attended by every head) get one
// more workgroup per tree.  One partial (m, l, acc) per head and workgroup goes to global
// memory; the last workgroup of a tree to arrive folds the tree's partials.
//
// Register arrays are only ever indexed by compile-time constants: a run-time index would
// push them to scratch memory.
#pragma once

#include <type_traits>

#include "search.h"
#include "search_mfma_timeline.h"
#include "threshold_kernel.h"

namespace hira {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef __attribute__((ext_vector_type(4))) int i32x4_t;

constexpr int kHeadsPerPass = 16;   // MFMA N
constexpr int kMaxTiles = 4;        // key tiles per block: bf <= 64
constexpr int kMfmaWaves = kMfmaThreads / 64;  // waves per workgroup, at most: one workgroup of 8
                                                // waves on a CU leaves every wave 256 registers
#ifndef HIRA_VBATCH
#define HIRA_VBATCH 32
#endif
constexpr int kVBatch = HIRA_VBATCH;         // value rows in flight per wave
constexpr int kQ8Batch = 16;                 // rows that pass the 8-bit shadow, looked at together

__device__ __forceinline__ bf16x8_t as_bf16x8(const uint4& v) {
    return __builtin_bit_cast(bf16x8_t, v);
}

// Tile `tile` of one tree's tiled matrix (D = 32*KS columns): a uniform base address, to
// which every lane adds its own 16 bytes' offset, so that the loads can take the base from
// scalar registers.
struct TilePtr {
    const char* base;  // uniform
    unsigned lane_off; // lane * 16
};
template <int KS>
__device__ __forceinline__ TilePtr tile_ptr(const void* base, size_t tree_row0, size_t tile, int lane) {
    return TilePtr{reinterpret_cast<const char*>(base) +
                       (tree_row0 * (size_t)(32 * KS) * 2 + tile * (size_t)(KS * 1024)),
                   (unsigned)lane * 16u};
}

template <int KS>
__device__ __forceinline__ void load_tile(const TilePtr tp, uint4 (&a)[KS]) {
#pragma unroll
    for (int s = 0; s < KS; ++s)
        a[s] = *reinterpret_cast<const uint4*>(tp.base + (size_t)tp.lane_off + s * 1024);
}

template <int KS>
__device__ __forceinline__ f32x4_t tile_scores(const uint4 (&a)[KS], const bf16x8_t (&bq)[KS]) {
    f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < KS; ++s)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a[s]), bq[s], acc, 0, 0, 0);
    return acc;
}

// Buffer addressing for the two streams of the scan and the gather (key tiles, value rows): the
// base sits in a scalar resource descriptor, the part that differs per load in a scalar offset,
// and every lane adds the same small offset of its own, so that no load needs vector registers
// for its address.  (One tree's keys or values must stay under 4 GiB.)
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, size_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)(uint32_t)bytes, 0x00020000);
}

// Cache policy of the scan's two streams.  A step reads a key tile once, so where the keys of a
// launch are more than the L2s hold they are better loaded non-temporal: they then do not push the
// centres, the queries and the value rows out on their way through.  POL 0: default policy for
// both; 1: key tiles non-temporal; 2: key tiles and value rows non-temporal.  Measured per step
// (keys of the launch: 67 MB / 268 MB / 1.07 GB): POL 0 20.11 / 65.05 / 197.3 us, POL 1 21.34 /
// 65.6 / 181.3 us, POL 2 19.86 / 66.1 / 185.1 us; with eight 67 MB indexes taking turns 22.9 /
// 22.2 / 22.2 us; and 15 % MORE than POL 0 where a caller searches the same 23 MB of keys again
// and again, which the L2s would have kept.  The host picks by the size of the launch's keys; a
// branch around the loads instead of instantiations costs the small launches a microsecond.  The
// coherence bits of the policy (sc0, sc1) change nothing.
// 8-bit shadow: POL 0 or 1 (its tiles).  Decode steps over 1 / 2 / 6 indexes in turn, POL 0 and POL 1: 128 MiB of shadow in the
// launch (8 heads a tree) 44.7 / 54.8 / 56.3 us and 48.9 / 49.1 / 52.8, 256 MiB 66.7 / 71.5 / - and 62.0 / 62.2 / -, 64 MiB 29.2 / 29.4 /
// 36.4 and 31.0 / 31.5 / 32.6, 32 MiB 19.8 / 19.8 / 20.2 and 18.8 / 19.8 / 20.4: what the cache behind the L2s could hold of
// one index or two is lost, what it holds of several gained -- the rows, which are read behind their tiles.  The line goes by
// two indexes in turn: at 64 MiB they lose with POL 1, as one does, where six gain a tenth; at 128 MiB they gain, as six do,
// where one loses a tenth.  The rows non-temporal too gain nothing (128 MiB 49.5 / 50.9 / 52.4).
constexpr int kReadOnce = 2;   // the `nt` bit of a buffer load's cache policy

template <int KS, bool ONCE>
__device__ __forceinline__ void load_tile_buf(__amdgpu_buffer_rsrc_t rsrc, unsigned lane_off,
                                              unsigned tile_off, uint4 (&a)[KS]) {
#pragma unroll
    for (int s = 0; s < KS; ++s)
        a[s] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(
                                             rsrc, lane_off + (unsigned)(s * 1024), tile_off,
                                             ONCE ? kReadOnce : 0));
}

// the same with the B operand parked in LDS (chunk s of lane l at [s*64 + l]): the scan keeps
// its registers for keys in flight
template <int KS>
__device__ __forceinline__ f32x4_t tile_scores_lds(const uint4 (&a)[KS], const uint4* bq_lds, int lane) {
    f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < KS; ++s)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a[s]), as_bf16x8(bq_lds[s * 64 + lane]),
                                                      acc, 0, 0, 0);
    return acc;
}

// A 16 x 64 tile of the keys' 8-bit shadow against the 16-bit query steps of up to 16 heads,
// split into a high and a low byte (two v_mfma_i32_16x16x64_i8 per 64 columns): exact integers
//   sum_j (256 hi_j + lo_j) k8_j
// for (row 4*(lane/16) + j, head lane % 16).  Lane (kb, i) of the A operand and lane (kb, head)
// of the B operands both hold columns [64 s + 16 kb, +16): the order of the columns inside the
// instruction does not matter as long as both sides agree.
template <int KS8>
__device__ __forceinline__ i32x4_t tile_scores_i8(const uint4 (&a)[KS8], const uint4 (&bhi)[KS8],
                                                  const uint4 (&blo)[KS8]) {
    i32x4_t hi = {0, 0, 0, 0}, lo = {0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < KS8; ++s) {
        hi = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(i32x4_t, a[s]),
                                                   __builtin_bit_cast(i32x4_t, bhi[s]), hi, 0, 0, 0);
        lo = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(i32x4_t, a[s]),
                                                   __builtin_bit_cast(i32x4_t, blo[s]), lo, 0, 0, 0);
    }
    return hi * 256 + lo;
}

constexpr float kQ8Steps = 32000.0f;   // the largest |q_j kscale_j| of a head, in its 16-bit steps
constexpr float kQ8KeySlack = 4e-3f;   // added to a node's error bound (in steps of the shadow):
                                       // rounding in the bound itself, in sum |q_j kscale_j| and
                                       // in the fp32 scores of the exact test (D <= 256)
constexpr float kQ8QuerySlack = 0.51f; // a query component is at most this many steps off

__device__ __forceinline__ float pick4(const f32x4_t& v, int j) {
    return j == 0 ? v[0] : (j == 1 ? v[1] : (j == 2 ? v[2] : v[3]));
}

// score of row `i` (0..15) of a scored tile for this lane's head
__device__ __forceinline__ float row_score(const f32x4_t& acc, int i, int col) {
    return __shfl(pick4(acc, i & 3), col + 16 * (i >> 2), 64);
}

// What lane % GS of my row of 16 holds.
template <int GS>
__device__ __forceinline__ float of_head(float v) {
    int x = __float_as_int(v);
    if constexpr (GS == 8) {  // the row's upper half takes the lower's
        x = __builtin_amdgcn_update_dpp(x, x, 0x118, 0xF, 0xC, false);
    } else if constexpr (GS == 4) {  // the second quad the first's, then the upper half the lower's
        x = __builtin_amdgcn_update_dpp(x, x, 0x114, 0xF, 0x2, false);
        x = __builtin_amdgcn_update_dpp(x, x, 0x118, 0xF, 0xC, false);
    }
    return __int_as_float(x);
}

__device__ __forceinline__ void stat_add(unsigned long long* st, int slot, unsigned v) {
    if (v) atomicAdd(&st[slot], (unsigned long long)v);
}

// Compile-time shape of one instantiation.
template <int KS, int MT, int GS, bool Q8 = false>
struct MfmaShape {
    static constexpr int D = 32 * KS;
    static constexpr int ROWS = MT * 16;  // key slots of one node
    static constexpr int KA = Q8 ? KS / 2 : KS;  // 16-byte chunks a lane holds of a scanned tile
    static constexpr int NB = mfma_round_nodes(KS, MT, GS, Q8);
    static constexpr int LIST = kMfmaWaves * NB * ROWS;  // rows of the list of one round
    // 8-bit shadow: rows that a wave lists before the workgroup looks at them, and the rounds that never list more;
    // a batch of rows: its scores, key slots and list entries
    static constexpr int CAP = 512, CHUNK = CAP / (NB * ROWS);
    static_assert(!Q8 || CHUNK >= 1, "a round has to fit");
    static constexpr int SCAN_WORDS = Q8 ? kMfmaWaves * (CAP + kQ8Batch * (GS + 4))
                                         : LIST * (GS + 1) + LIST / 16;  // row list, tile slots, GS scores per row
    static constexpr int MERGE_WORDS = kMfmaWaves * 4 * D;  // four heads of every wave
    static constexpr int WORDS = SCAN_WORDS > MERGE_WORDS ? SCAN_WORDS : MERGE_WORDS;
};

// What a wave needs to gate one tile of 16 level-1 nodes, as it comes from memory.
template <int KS>
struct GateLoads {
    uint4 a1[KS];      // the tile of level-1 centres
    float4 r4;         // radii of rows 4*kb .. 4*kb+3
    int cn;            // child count of row lane % 16
    float en;          // (8-bit shadow) error bound of that row
    uint4 anc[2][KS];  // tiles holding the ancestors at levels min(L-1,3) and the one below
    float arad[2];
    unsigned aid[2];
};

// The arguments that the kernel needs up to the gates, in registers from its first instructions on.  Asked for where they
// are used they came one after the other, each behind its branch and its wait, a dozen hits of the scalar cache ahead of
// the last gate's operands (8 trees x 2000 keys 9.48 -> 9.21 us; x 32768, which waits for its fullest workgroup, 17.7 either way).
// (Addresses as numbers: global_at.)
struct GateArgs {
    uintptr_t q, centers, anc_centers[2], tau, scaling, radii, anc_radii[2], keps, counts, keys, part_acc, stats;
    int32_t num_levels, cap, anc_cap[2], size, group_size, tree_blocks, tiles, bf, cap0, wgs, threads;
    uint32_t bf_magic;
};
__device__ __forceinline__ GateArgs gate_arguments(const SearchParams& p) {
    auto at = [](const void* a) { return reinterpret_cast<uintptr_t>(a); };
    GateArgs g{at(p.q), at(p.centers[1]), {at(p.anc_centers[0]), at(p.anc_centers[1])}, at(p.tau), at(p.scaling), at(p.radii[1]),
               {at(p.anc_radii[0]), at(p.anc_radii[1])}, at(p.keps), at(p.counts[1]), at(p.keys), at(p.part_acc), at(p.stats),
               p.num_levels, p.cap[1], {p.anc_cap[0], p.anc_cap[1]}, p.size[1], p.group_size,
               p.tree_blocks, p.nodes_per_wave, p.bf, p.cap[0], (int)gridDim.y, (int)blockDim.x, p.bf_magic};
    asm volatile("" : "+s"(g.q), "+s"(g.centers), "+s"(g.anc_centers[0]), "+s"(g.anc_centers[1]), "+s"(g.tau), "+s"(g.scaling),
                      "+s"(g.radii), "+s"(g.anc_radii[0]), "+s"(g.anc_radii[1]), "+s"(g.keps), "+s"(g.counts),
                      "+s"(g.keys), "+s"(g.part_acc), "+s"(g.stats));
    asm volatile("" : "+s"(g.num_levels), "+s"(g.cap), "+s"(g.anc_cap[0]), "+s"(g.anc_cap[1]), "+s"(g.size), "+s"(g.group_size),
                      "+s"(g.tree_blocks), "+s"(g.tiles), "+s"(g.bf), "+s"(g.cap0), "+s"(g.wgs), "+s"(g.threads), "+s"(g.bf_magic));
    return g;
}

// Parent of node n.  By a multiplication: the quotients of 64-bit numbers that stood here, one after the
// other ahead of the ancestors' loads, were 0.3 us of every step (8 trees x 2000 keys 12.7 -> 12.4 us, x 32768 19.6 -> 19.2).
__device__ __forceinline__ unsigned node_over_bf(const GateArgs& p, unsigned n) {
    return __umulhi(n, p.bf_magic);  // (fan-outs of 16 and more: never 1)
}

template <int KS, bool Q8>
__device__ __forceinline__ void gate_issue(const GateArgs& p, int tree, int t1, int lane,
                                           int kb, GateLoads<KS>& g) {
    const int L = p.num_levels;
    const size_t row1 = (size_t)tree * p.cap;
    load_tile<KS>(tile_ptr<KS>(global_at<char>(p.centers), row1, (size_t)t1, lane), g.a1);
    g.r4 = *reinterpret_cast<const float4*>(global_at<float>(p.radii) + row1 + (size_t)t1 * 16 + 4 * kb);
    g.cn = global_at<int32_t>(p.counts)[row1 + (size_t)t1 * 16 + (lane & 15)];
    if (Q8) g.en = global_at<float>(p.keps)[row1 + (size_t)t1 * 16 + (lane & 15)];
    const int n_par = min(max(L - 2, 0), 2);
    const unsigned id2 = node_over_bf(p, (unsigned)t1 * 16u);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        g.arad[i] = 0.f;
        g.aid[i] = 0;
        if (i < n_par) {
            const int l = min(L - 1, 3) - i;
            g.aid[i] = l == 3 ? node_over_bf(p, id2) : id2;
            load_tile<KS>(tile_ptr<KS>(global_at<char>(p.anc_centers[i]), (size_t)tree * p.anc_cap[i], g.aid[i] / 16, lane), g.anc[i]);
            g.arad[i] = global_at<float>(p.anc_radii[i])[(size_t)tree * p.anc_cap[i] + g.aid[i]];
        }
    }
}

// OUT: the launch also wants dense scores or selection lists (kept out of the attention-only
// instantiation, whose registers are all spoken for).
// Q8: the index keeps an 8-bit shadow of its keys (HIRA_TILE16_Q8).  The scan then reads the
// shadow's tiles (half the bytes) and lists the rows that the shadow cannot rule out for some
// head; their bf16 rows (row-major) are fetched, 16 at a time as one MFMA operand, and take the
// exact test -- with the very products of the other layout, so the selected set and the scores
// are the same bit for bit.
// ONE: every workgroup of the launch scans in a single round (the host knows: its tiles hold no
// more nodes than its waves take at once).  The round is then straight-line code without a loop
// around it, in which the compiler's waits count the loads still in flight and a node's products
// start when ITS tiles have arrived; at the head of a loop they fall back to waiting for
// everything asked for so far.
// AHEAD: (small launches) a workgroup owns one tile, and its waves ask for the key tiles of their two
// nodes each together with the gates' operands, whether the nodes survive or not: a trip to memory less,
// and no list of survivors.  As a number: the nodes of a wave; with one, two workgroups share a tile (SearchPlan.slices).
// SAMPLED: (with AHEAD) the launch makes its thresholds itself, in workgroups ahead of the searching ones.
template <int KS, int MT, int GS, bool OUT, bool Q8, int POL, int HV, bool ONE, int AHEAD = 0, bool SAMPLED = false>
__global__ __launch_bounds__(64 * kMfmaWaves, 2) void search_mfma_kernel(const SearchParams p) {
    using S = MfmaShape<KS, MT, GS, Q8>;
    constexpr int D = S::D;
    constexpr int NB = AHEAD ? AHEAD : S::NB;
    constexpr int SLICES = AHEAD ? kAheadNodes / AHEAD : 1;  // workgroups that share a tile
    static_assert(!AHEAD || (ONE && !OUT && !Q8 && HV == 1 && NB <= S::NB), "");
    constexpr int KA = S::KA;          // 16-byte chunks per lane of a scanned tile
    constexpr int KS8 = Q8 ? KS / 2 : 1;
    constexpr int VPL = KS / 2;        // value elements per lane: Dv = D = 64 * VPL
    constexpr int VW = (VPL + 1) / 2;  // dwords of a value row per lane
    __shared__ __align__(16) uint32_t s_words[S::WORDS];  // the round's list; the merge; the fold
    // a node of my tiles: heads for which it survives (16 bits) | child count << 16
    __shared__ uint32_t s_ninfo[kMfmaMaxTilesPerWg * 16];
    // the surviving ones in order, a copy per wave (each wave makes its own: no barrier):
    // node | child count << 8 | heads << 16
    __shared__ uint32_t s_order[kMfmaWaves][kMfmaMaxTilesPerWg * 16 * HV];
    __shared__ float s_mxw[kMfmaWaves * 16];           // a wave's running maximum per head
    __shared__ float s_lw[kMfmaWaves * 16];
    __shared__ float s_mh[kHeadsPerPass];
    __shared__ float s_red[2 * kHeadsPerPass];
    __shared__ int s_nc[kHeadsPerPass];
    __shared__ int s_last;
    __shared__ uint4 s_bq[KS * 64];  // the B operand (queries) of the scan
    // 8-bit shadow: the queries in steps of the shadow, high and low bytes, as B operands; the
    // step and sum_j |q_j kscale_j| of every head; the error bounds of my nodes
    __shared__ uint4 s_bq8[Q8 ? 2 * KS8 * 64 : 1];
    __shared__ float s_qc[Q8 ? 2 * kHeadsPerPass : 1];
    __shared__ float s_keps[Q8 ? kMfmaMaxTilesPerWg * 16 : 1];
    __shared__ int s_rows[Q8 ? kMfmaWaves : 1];  // rows that the waves have listed
    __shared__ int s_places[Q8 && OUT ? kMfmaWaves * 16 : 1], s_place0[Q8 && OUT ? 16 : 1];  // of a batch on the heads' lists

    touch_kernel_arguments();
    const GateArgs ga = gate_arguments(p);
    const int lane = lane_id();
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int nw = ga.threads >> 6;
    const int col = lane & 15;  // head within the pass
    const int kb = lane >> 4;   // column block of 8 inside each 32-column step
    const int tree = blockIdx.x;
    const int L = ga.num_levels, bf = ga.bf;
    const bool want_attn = ga.part_acc != 0;
    static_assert(!SAMPLED || (AHEAD && S::WORDS >= kTauFewRows), "");
    __shared__ float s_tau[SAMPLED ? kHeadsPerPass : 1];
    int wgs = ga.wgs, wg = blockIdx.y;  // searching workgroups of the tree, my number among them
    if constexpr (SAMPLED) {
        wgs -= p.sample_wgs;
        wg -= p.sample_wgs;
        if (wg < 0) {  // uniform
            threshold_stretch<4 * KS>(p.sample, p.sample_rows, p.q, tree, p.group_size, (int)blockIdx.y, p.sample_best,
                                      reinterpret_cast<float*>(s_words), p.done + tree, wgs + p.sample_wgs * kTauMade);
            return;
        }
    }
    // Workgroup y of a tree owns the tree's tiles y, y + (workgroups of the tree), ...: a stride
    // apart, since neighbouring tiles hold sibling nodes, which tend to survive (and be selected
    // from) together.
    const int wg_tiles = (ga.size + 15) >> 4;
    const int n_groups = ga.tree_blocks / SLICES;
    const int grp = wg / SLICES, slice = wg % SLICES;
    const int ntile = wg < ga.tree_blocks
                          ? min(ga.tiles, (wg_tiles - grp + n_groups - 1) / n_groups)
                          : 0;
    auto tile_of = [&](int tl) { return grp + tl * n_groups; };
    // level-1 node behind entry n (tile n / 16 of mine, node n % 16 of the tile)
    auto node_of = [&](int n) { return tile_of(n >> 4) * 16 + (n & 15); };
    const bool is_queue = wg >= ga.tree_blocks;  // the workgroup after the tree's
    Timeline tline(p);  // (empty unless the library is built with time stamps)
    unsigned long long* stats =
        (ga.stats != 0 && !Timeline::kOn) ? p.stats + (size_t)tree * HIRA_STATS_COLS : nullptr;
    tline.stamp(kTlStart);

    // ---- heads of this pass ----------------------------------------------------------
    int hoff, G;
    if (ga.group_size > 0) {  // head h of the launch belongs to tree h / group_size
        hoff = tree * ga.group_size + blockIdx.z * kHeadsPerPass;
        G = min(kHeadsPerPass, ga.group_size - (int)blockIdx.z * kHeadsPerPass);
    } else {
        hoff = p.tree_q_off[tree] + blockIdx.z * kHeadsPerPass;
        G = min(kHeadsPerPass, p.tree_q_off[tree + 1] - hoff);
    }
    if (G <= 0 || (ntile <= 0 && !is_queue)) return;  // uniform
    G = min(G, GS);
    tline.stamp(kTlArgs);
    const bool head_ok = col < G;
    int qh = 0;
    if (head_ok) qh = ga.group_size > 0 ? hoff + col : p.tree_q_heads[hoff + col];

    // ---- softmax state: running maximum m of the lane's head (the same in every wave);
    // per wave: l over the rows it gathered, acc[g][e] = column lane*VPL + e of head g -------
    float m_run = -INFINITY;
    float l_mine = 0.0f;  // this lane's share of l of head lane % GS, over the rows this wave gathered
    float acc[GS][VPL];
#pragma unroll
    for (int g = 0; g < GS; ++g)
#pragma unroll
        for (int e = 0; e < VPL; ++e) acc[g][e] = 0.0f;
    // The gather of the single-round instantiations (up to 8 heads a pass, rows of 256 bytes)
    // fetches value rows 16 bytes a lane: LR lanes share a row, one load instruction brings RPI
    // rows, and lane (row group rg, chunk cc) sums columns 8 cc .. 8 cc + 7 of the rows of its
    // group in acc8; the row groups' sums meet before the merge.  (A quarter of the load
    // instructions and half the instructions per row of the gather below, which holds a row in
    // 4 bytes a lane.  A launch of several rounds keeps the next round's tiles in flight during
    // the gather: its registers take the eight columns of up to four heads, 233 in all.)
    constexpr bool WIDE = (ONE || Q8 ? GS <= 8 : GS <= 4) && KS == 4;
    constexpr int LR = D / 8;     // lanes per value row
    constexpr int RPI = 64 / LR;  // rows per load instruction
    const int rg = lane / LR, cc = lane % LR;
    float acc8[WIDE ? GS : 1][8];
#pragma unroll
    for (int g = 0; g < (WIDE ? GS : 1); ++g)
#pragma unroll
        for (int j = 0; j < 8; ++j) acc8[g][j] = 0.0f;

    if (is_queue) {
        // ---- the queue of keys appended since the last update of the tree: row-major, every
        // row counts for every head (no threshold).  Lane owns VPL columns; a wave takes rows
        // wave, wave + nw, ..., eight at a time, and keeps its own (m, l, acc) per head. -------
        float qf[GS][VPL], sc2g[GS], mq[GS], lq[GS];
#pragma unroll
        for (int g = 0; g < GS; ++g) {
            mq[g] = -INFINITY;
            lq[g] = 0.0f;
            sc2g[g] = 0.0f;
#pragma unroll
            for (int e = 0; e < VPL; ++e) qf[g][e] = 0.0f;
            if (g < G) {  // uniform
                const int head = p.group_size > 0 ? hoff + g : p.tree_q_heads[hoff + g];
                sc2g[g] = p.scaling[head] * kLog2e;
                const uint16_t* qp = reinterpret_cast<const uint16_t*>(p.q) + (size_t)head * D + lane * VPL;
#pragma unroll
                for (int e = 0; e < VPL; ++e) qf[g][e] = bf16_lo((uint32_t)qp[e]);
            }
        }
        const uint16_t* qk = reinterpret_cast<const uint16_t*>(p.queue_keys) + (size_t)tree * p.queue_cap * D + lane * VPL;
        const uint16_t* qv = reinterpret_cast<const uint16_t*>(p.queue_values) + (size_t)tree * p.queue_cap * D + lane * VPL;
        for (int r0 = wave; r0 < p.queue_len; r0 += 8 * nw) {  // uniform in the wave
            uint16_t kraw[8][VPL], vraw[8][VPL];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int row = min(r0 + i * nw, p.queue_len - 1);
#pragma unroll
                for (int e = 0; e < VPL; ++e) {
                    kraw[i][e] = qk[(size_t)row * D + e];
                    vraw[i][e] = qv[(size_t)row * D + e];
                }
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                if (r0 + i * nw >= p.queue_len) break;  // uniform
#pragma unroll
                for (int g = 0; g < GS; ++g) {
                    if (g >= G) continue;  // uniform (no break: the loop has to unroll)
                    float sdot = 0.0f;
#pragma unroll
                    for (int e = 0; e < VPL; ++e) sdot += bf16_lo((uint32_t)kraw[i][e]) * qf[g][e];
                    sdot = wave_sum(sdot);
                    const float z = sdot * sc2g[g];
                    const float mnew = fmaxf(mq[g], z);
                    const float f = exp2f(mq[g] - mnew);  // 0 the first time
                    const float w = exp2f(z - mnew);
                    lq[g] = lq[g] * f + w;
#pragma unroll
                    for (int e = 0; e < VPL; ++e)
                        acc[g][e] = acc[g][e] * f + w * bf16_lo((uint32_t)vraw[i][e]);
                    mq[g] = mnew;
                }
            }
        }
        // hand the wave's state over in the form the merge below expects
#pragma unroll
        for (int g = 0; g < GS; ++g) {
            if (lane == g) l_mine = lq[g];
            if (col == g) m_run = mq[g];
        }
    } else {
        // ---- queries and the first tile's gate operands, issued before the first wait --------
        // (only the waves that gate need the queries in registers: the scan reads them from LDS)
        // (No load here depends on whether the LANE has a head: a lane without one asks for head
        // 0 of the launch and drops what comes back.  Loads under a per-lane condition end up in
        // blocks of their own, and a use that the compiler moves into such a block is waited for
        // there, with everything else still in flight -- the scaling times log2 e was: a whole
        // trip to memory before the gates' operands were even asked for.  Measured on the 32k
        // benchmark step, with the arguments touched as above: 19.74 -> 19.40 us.)
        int tl_mine = wave;  // of my tiles, the one this wave gates next
        uint4 qraw[KS];
#pragma unroll
        for (int s = 0; s < KS; ++s) qraw[s] = make_uint4(0, 0, 0, 0);
        float tau = SAMPLED ? 0.0f : global_at<float>(ga.tau)[qh];
        float sc = global_at<float>(ga.scaling)[qh];
        GateLoads<KS> gl;
        uint4 a[NB][MT][KA];  // key tiles of the nodes that a wave takes in a round
        if (tl_mine < ntile) {
#pragma unroll
            for (int s = 0; s < KS; ++s)
                qraw[s] = *reinterpret_cast<const uint4*>(global_at<uint16_t>(ga.q) +
                                                          (size_t)qh * D + s * 32 + kb * 8);
            gate_issue<KS, Q8>(ga, tree, tile_of(tl_mine), lane, kb, gl);
        }
        if constexpr (AHEAD) {
            // (slots beyond the capacity, under nodes that pad the tile or a last node of 48: zeros, no memory
            // access)
            const size_t r0 = (size_t)tree * ga.cap0;
            const __amdgpu_buffer_rsrc_t rsrc = make_rsrc(
                global_at<uint16_t>(ga.keys) + r0 * (size_t)D, (size_t)ga.cap0 * D * 2);
#pragma unroll
            for (int u = 0; u < NB; ++u)
#pragma unroll
                for (int tt = 0; tt < MT; ++tt)
                    load_tile_buf<KA, POL != 0>(
                        rsrc, (unsigned)lane * 16u,
                        ((unsigned)(node_of((slice * NB + u) * kMfmaWaves + wave) * bf) / 16u + tt) * (unsigned)(KA * 1024), a[u][tt]);
        }
        __builtin_amdgcn_sched_barrier(0);  // (nothing that uses a load moves above this line)
        tline.stamp(kTlGateIssued);
        if (!head_ok) {
            tau = INFINITY;
            sc = 0.0f;
#pragma unroll
            for (int s = 0; s < KS; ++s) qraw[s] = make_uint4(0, 0, 0, 0);
        }
        if constexpr (Q8) {
            // ---- the queries in steps of the shadow (the last wave, which has the fewest tiles to
            // gate, for all): lane (kb, head) takes
            // columns [64 s + 16 kb, +16) as the shadow's tiles hold them: u_j = q_j kscale_j,
            // the head's step su = max_j |u_j| / kQ8Steps, U_j = round(u_j / su) in two bytes -------
            if (wave == nw - 1) {
                float uf[KS8][16];
                float umax = 0.0f, asum = 0.0f;
#pragma unroll
                for (int s = 0; s < KS8; ++s) {
                    const int c0 = 64 * s + 16 * kb;
                    uint4 qa = make_uint4(0, 0, 0, 0), qb = make_uint4(0, 0, 0, 0);
                    if (head_ok) {
                        const uint16_t* qp = reinterpret_cast<const uint16_t*>(p.q) + (size_t)qh * D + c0;
                        qa = *reinterpret_cast<const uint4*>(qp);
                        qb = *reinterpret_cast<const uint4*>(qp + 8);
                    }
                    float qf[16];
                    {
                        float f[8];
                        unpack<bf16_t>(qa, f);
#pragma unroll
                        for (int e = 0; e < 8; ++e) qf[e] = f[e];
                        unpack<bf16_t>(qb, f);
#pragma unroll
                        for (int e = 0; e < 8; ++e) qf[8 + e] = f[e];
                    }
                    const float4* kp = reinterpret_cast<const float4*>(p.kscale + (size_t)tree * D + c0);
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        const float4 k4 = kp[c];
                        uf[s][4 * c + 0] = qf[4 * c + 0] * k4.x;
                        uf[s][4 * c + 1] = qf[4 * c + 1] * k4.y;
                        uf[s][4 * c + 2] = qf[4 * c + 2] * k4.z;
                        uf[s][4 * c + 3] = qf[4 * c + 3] * k4.w;
                    }
#pragma unroll
                    for (int e = 0; e < 16; ++e) {
                        umax = fmaxf(umax, fabsf(uf[s][e]));
                        asum += fabsf(uf[s][e]);
                    }
                }
                umax = cross_group_max<16>(umax);
                asum = cross_group_sum<16>(asum);
                const float su = fmaxf(umax, 1e-30f) / kQ8Steps;
                const float inv = kQ8Steps / fmaxf(umax, 1e-30f);  // (u * inv: within 0.004 of u / su)
#pragma unroll
                for (int s = 0; s < KS8; ++s) {
                    uint32_t hi[4], lo[4];
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        hi[c] = 0u;
                        lo[c] = 0u;
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const int U = (int)rintf(uf[s][4 * c + e] * inv);
                            const int h = (U + 128) >> 8;  // U = 256 h + l, l in [-128, 127]
                            const int l = U - (h << 8);
                            hi[c] |= ((uint32_t)h & 0xFFu) << (8 * e);
                            lo[c] |= ((uint32_t)l & 0xFFu) << (8 * e);
                        }
                    }
                    s_bq8[s * 64 + lane] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
                    s_bq8[(KS8 + s) * 64 + lane] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
                }
                if (kb == 0) {
                    s_qc[col] = su;
                    s_qc[kHeadsPerPass + col] = asum;
                }
            }
        }

        // ---- B operand and ||q|| -----------------------------------------------------------
        bf16x8_t bq[KS];
        float ss = 0.0f;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            bq[s] = as_bf16x8(qraw[s]);
            float f[8];
            unpack<bf16_t>(qraw[s], f);
#pragma unroll
            for (int e = 0; e < 8; ++e) ss += f[e] * f[e];
        }
        ss = cross_group_sum<16>(ss);
        const float qn = sqrtf(ss);
        if (wave == 0) {
#pragma unroll
            for (int s = 0; s < KS; ++s) s_bq[s * 64 + lane] = qraw[s];
        }

        if constexpr (SAMPLED) {
            // the thresholds: wave 0, which alone gates, waits for them and leaves them to the others
            if (wave == 0) {
                threshold_join<4 * KS, GS>(p.sample, p.sample_rows, p.q, tree, hoff, G, p.sample_k, p.sample_best, p.sample_wait, s_tau,
                                           reinterpret_cast<float*>(s_words));
                tau = head_ok ? s_tau[col] : INFINITY;
                if (wg == 0 && lane < G) const_cast<float*>(p.tau)[hoff + lane] = s_tau[lane];
            }
        }

        // ---- gate: one tile per wave at a time ------------------------------------------------
        while (tl_mine < ntile) {  // uniform in the wave
            const int t1 = tile_of(tl_mine);
            if constexpr (OUT) {
                // the dense output's stretch under this tile starts out as the fill value (the
                // barrier behind the gates has every wave wait for these stores, so the scores
                // that any wave writes later come after them)
                if (p.dense_fill) {
                    const int r0 = t1 * 16 * bf, r1 = min(r0 + 16 * bf, p.size[0]);
                    for (int g = 0; g < G; ++g) {
                        const int head = p.group_size > 0 ? hoff + g : p.tree_q_heads[hoff + g];
                        for (int i = r0 + lane; i < r1; i += 64)
                            p.dense[(int64_t)head * p.dense_stride + i] = p.dense_fill_value;
                    }
                }
            }
            const bool count_nodes = stats != nullptr && lane == 0 && slice == 0;
            int lcur = L - 1;
            bool chain = head_ok;  // this head is still alive above the current level
            // the tile's ancestor at level l; is the tile's first node its first descendant?
            auto ancestor = [&](int l) {
                unsigned id = (unsigned)t1 * 16u;
                for (int i = 1; i < l; ++i) id = node_over_bf(ga, id);
                return id;
            };
            auto leads = [&](int l) {
                unsigned id = ancestor(l);
                for (int i = 1; i < l; ++i) id *= (unsigned)bf;
                return id == (unsigned)t1 * 16u;
            };
            for (; lcur > 3; --lcur) {  // trees deeper than four levels: one level at a time
                const unsigned a = ancestor(lcur);
                uint4 t[KS];
                load_tile<KS>(tile_ptr<KS>(p.centers[lcur], (size_t)tree * p.cap[lcur], a / 16, lane), t);
                const float rad = p.radii[lcur][(size_t)tree * p.cap[lcur] + a];
                const bool any_alive = __ballot(chain) != 0ull;
                if (count_nodes && any_alive && rad > -INFINITY && leads(lcur))
                    stat_add(stats, lcur, 1u);
                const float d = row_score(tile_scores<KS>(t, bq), (int)(a % 16), col);
                chain = chain && (d + qn * rad >= tau);
            }
            const int n_par = min(max(L - 2, 0), 2);
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                if (i < n_par) {
                    const bool any_alive = __ballot(chain) != 0ull;
                    if (count_nodes && any_alive && gl.arad[i] > -INFINITY && leads(lcur))
                        stat_add(stats, lcur, 1u);
                    const float d = row_score(tile_scores<KS>(gl.anc[i], bq), (int)(gl.aid[i] % 16), col);
                    chain = chain && (d + qn * gl.arad[i] >= tau);
                    --lcur;
                }
            }
            const bool tile_live = __ballot(chain) != 0ull;  // uniform

            // level-1 gates: 16 nodes at once
            unsigned alive4 = 0u;
            if (tile_live) {
                const f32x4_t g1 = tile_scores<KS>(gl.a1, bq);
                const float rr[4] = {gl.r4.x, gl.r4.y, gl.r4.z, gl.r4.w};
                unsigned real = 0u;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    if (chain && (g1[j] + qn * rr[j] >= tau)) alive4 |= 1u << j;
                    if (stats) real += (unsigned)__popcll(__ballot(col == 0 && rr[j] > -INFINITY));
                }
                if (count_nodes) stat_add(stats, 1, real);
            }
            unsigned long long nb[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) nb[j] = __ballot((alive4 >> j) & 1u);
            // node n = 4*kb' + j of the tile: its heads are field kb' of nb[j]
            if (lane < 16) {
                const int jn = lane & 3;
                const unsigned long long bits = jn == 0 ? nb[0] : (jn == 1 ? nb[1] : (jn == 2 ? nb[2] : nb[3]));
                s_ninfo[tl_mine * 16 + lane] =
                    (uint32_t)((bits >> (16 * (lane >> 2))) & 0xFFFFull) | ((uint32_t)gl.cn << 16);
            }
            if constexpr (Q8) {
                if (lane < 16) s_keps[tl_mine * 16 + lane] = gl.en;
            }
            tl_mine += nw;
            if (tl_mine < ntile) gate_issue<KS, Q8>(ga, tree, tile_of(tl_mine), lane, kb, gl);
        }
        tline.stamp(kTlGated);
        __syncthreads();
        tline.stamp(kTlBarrier);
        if constexpr (SAMPLED) tau = head_ok ? s_tau[col] : INFINITY;

        // ---- the surviving nodes of my tiles in order, dealt round-robin to the waves ----------
        int rounds = 1, alive = 0;
        if constexpr (!AHEAD) {
            const int n_info = ntile * 16;
            const unsigned long long lt = (1ull << lane) - 1ull;
#pragma unroll
            for (int i = 0; i < kMfmaMaxTilesPerWg * 16 / 64; ++i) {
                if (64 * i >= n_info) break;  // uniform
                const uint32_t info = 64 * i + lane < n_info ? s_ninfo[64 * i + lane] : 0u;
                const bool live = (info & 0xFFFFu) != 0u;
                const unsigned long long all = __ballot(live);
                if (live) {
                    // (HV = 2: a node goes in as two entries of MT tiles each, the second marked
                    // by bit 15; a half without keys costs its wave nothing but the entry)
                    const int at = (alive + __popcll(all & lt)) * HV;
                    const int cnt_n = (int)(info >> 16);
#pragma unroll
                    for (int h = 0; h < HV; ++h)
                        s_order[wave][at + h] =
                            (uint32_t)(64 * i + lane) | ((uint32_t)min(max(cnt_n - h * MT * 16, 0), MT * 16) << 8) |
                            ((uint32_t)h << 15) | (info << 16);
                }
                alive += __popcll(all);
            }
            alive *= HV;
            rounds = ((alive + nw - 1) / nw + NB - 1) / NB;
            tline.set(kTlAlive, (unsigned long long)alive);
        }

        float sc2 = sc * kLog2e;
        asm volatile("" : "+v"(sc2));  // (computed here, where its load has long arrived, and not
                                       // behind the key tiles' requests, where it would be waited
                                       // for with all of them)
        const size_t row0 = (size_t)tree * ga.cap0;

        // (8-bit shadow: krsrc = the bf16 rows of the exact test, row-major; k8rsrc = the tiles
        // of the shadow, which the scan reads)
        const __amdgpu_buffer_rsrc_t krsrc = make_rsrc(
            global_at<uint16_t>(ga.keys) + row0 * (size_t)D, (size_t)ga.cap0 * D * 2);
        const __amdgpu_buffer_rsrc_t k8rsrc =
            Q8 ? make_rsrc(p.keys8 + row0 * (size_t)D, (size_t)ga.cap0 * D) : krsrc;
        uint4 bq8h[KS8], bq8l[KS8];
        float su = 0.0f, asum = 0.0f;
        if constexpr (Q8) {
#pragma unroll
            for (int s = 0; s < KS8; ++s) {
                bq8h[s] = s_bq8[s * 64 + lane];
                bq8l[s] = s_bq8[(KS8 + s) * 64 + lane];
            }
            su = s_qc[col];
            asum = s_qc[kHeadsPerPass + col];
        }
        const __amdgpu_buffer_rsrc_t vrsrc = make_rsrc(
            reinterpret_cast<const uint16_t*>(p.values) + row0 * (size_t)D, (size_t)ga.cap0 * D * 2);
        // The nodes a wave takes in a round (up to NB of its share), what LDS says about them,
        // and the loads of their key tiles.
        int nx_node[NB], nx_cnt[NB], nx_half[NB];
        uint32_t nx_mask[NB];
        float nx_eps[Q8 ? NB : 1];
        auto fetch = [&](int round, int u_only) {  // u_only < 0: all NB nodes of the round
            // my nodes of the round: entries (round*NB + u) * nw + wave of the survivors
            uint32_t ent[NB];
#pragma unroll
            for (int u = 0; u < NB; ++u) {
                if (u_only >= 0 && u != u_only) continue;
                const int k = (round * NB + u) * nw + wave;
                ent[u] = k < alive ? s_order[wave][k] : 0xFFu;
            }
#pragma unroll
            for (int u = 0; u < NB; ++u) {
                if (u_only >= 0 && u != u_only) continue;
                const uint32_t e = (uint32_t)__builtin_amdgcn_readfirstlane((int)ent[u]);
                const int n = (e >> 16) != 0u ? (int)(e & 0xFFu) : -1;
                nx_node[u] = n;
                nx_cnt[u] = (int)((e >> 8) & 0x7Fu);
                nx_half[u] = (int)((e >> 15) & 1u);
                nx_mask[u] = e >> 16;
                if constexpr (Q8) nx_eps[u] = s_keps[max(n, 0)];
                const unsigned tile_first = (unsigned)(node_of(max(n, 0)) * bf) / 16u + (unsigned)(nx_half[u] * MT);
#pragma unroll
                for (int tt = 0; tt < MT; ++tt) {
                    if constexpr (Q8) {
                        // every load is issued, whatever the node (straight-line code, so that the
                        // waits further down can count the loads behind them); a tile that is not
                        // there is asked for beyond the end of the buffer: zeros, no memory access
                        load_tile_buf<KA, POL != 0>(k8rsrc, (unsigned)lane * 16u + (tt * 16 < nx_cnt[u] ? 0u : 0x80000000u),
                                          (tile_first + tt) * (unsigned)(KA * 1024), a[u][tt]);
                    } else {
                        // (every load is issued, a tile that is not there beyond the end of the
                        // buffer -- zeros, no memory access: straight-line code, in which the waits
                        // further down can count the loads behind them)
                        load_tile_buf<KA, POL != 0>(krsrc, (unsigned)lane * 16u + (tt * 16 < nx_cnt[u] ? 0u : 0x80000000u),
                                          (tile_first + tt) * (unsigned)(KA * 1024), a[u][tt]);
                    }
                }
            }
        };
        if constexpr (AHEAD) {
#pragma unroll
            for (int u = 0; u < NB; ++u) {
                const int n = (slice * NB + u) * kMfmaWaves + wave;
                const uint32_t info = (uint32_t)__builtin_amdgcn_readfirstlane((int)s_ninfo[n]);
                nx_node[u] = n;
                nx_half[u] = 0;
                nx_mask[u] = info & 0xFFFFu;
                nx_cnt[u] = nx_mask[u] != 0u ? (int)(info >> 16) : 0;
            }
        } else {
            if (!Q8 && rounds > 0) fetch(0, -1);
        }
        tline.stamp(kTlFetched);

        // dense scores / compact lists of the selected rows among 16 scored ones: lane
        // (kb, head) holds rows 4*kb + j, whose key slots are slot4[j]; reserve: so many places on the lane's head's list
        auto emit = [&](int col, int kb, unsigned sel4, const f32x4_t& sco, const unsigned (&slot4)[4], auto reserve) {
            unsigned long long sb[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) sb[j] = __ballot((sel4 >> j) & 1u);
            int base = 0;
            if (p.sel_count != nullptr) {
                int mine = 0;
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    mine += __popcll(sb[j] & (0x0001000100010001ull << col));
                base = reserve(mine);
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if ((sel4 >> j) & 1u) {
                    const unsigned slot = slot4[j];
                    int idx = (int)slot;
                    if (p.dense_by_position) idx = p.perm[row0 + slot];
                    if (p.dense != nullptr)
                        p.dense[(int64_t)qh * p.dense_stride + idx] = sco[j] * sc;
                    if (p.sel_count != nullptr) {
                        // hits of my head ordered before (kb, j): rows j' < j of any
                        // kb, then row j of lower kb
                        int before = 0;
#pragma unroll
                        for (int j2 = 0; j2 < 4; ++j2) {
                            unsigned long long bits = sb[j2] & (0x0001000100010001ull << col);
                            if (j2 == j) bits &= (1ull << (16 * kb)) - 1ull;
                            if (j2 <= j) before += __popcll(bits);
                        }
                        const int pos = base + before;
                        if (pos < p.sel_cap) {
                            p.sel_index[(int64_t)qh * p.sel_cap + pos] = idx;
                            p.sel_score[(int64_t)qh * p.sel_cap + pos] = sco[j];
                        }
                    }
                }
            }
        };
        // rows (of 16) for which some head's bit is set: OR over the 16 lanes (heads) of my
        // row group by rotating inside the group, then the four groups side by side
        auto rows_of = [&](unsigned sel4) {
            unsigned any4 = sel4;
            any4 |= (unsigned)__builtin_amdgcn_update_dpp(0, (int)any4, 0x121, 0xF, 0xF, false);
            any4 |= (unsigned)__builtin_amdgcn_update_dpp(0, (int)any4, 0x122, 0xF, 0xF, false);
            any4 |= (unsigned)__builtin_amdgcn_update_dpp(0, (int)any4, 0x124, 0xF, 0xF, false);
            any4 |= (unsigned)__builtin_amdgcn_update_dpp(0, (int)any4, 0x128, 0xF, 0xF, false);
            return (unsigned)__builtin_amdgcn_readlane((int)any4, 0) |
                   ((unsigned)__builtin_amdgcn_readlane((int)any4, 16) << 4) |
                   ((unsigned)__builtin_amdgcn_readlane((int)any4, 32) << 8) |
                   ((unsigned)__builtin_amdgcn_readlane((int)any4, 48) << 12);
        };
        auto count_selected = [&](unsigned sel4, unsigned rowmask) {
            const unsigned pairs = (unsigned)__popcll(__ballot(sel4 & 1u)) +
                                   (unsigned)__popcll(__ballot(sel4 & 2u)) +
                                   (unsigned)__popcll(__ballot(sel4 & 4u)) +
                                   (unsigned)__popcll(__ballot(sel4 & 8u));
            if (lane == 0) {
                stat_add(stats, HIRA_MAX_LEVELS, (unsigned)__popc(rowmask));
                stat_add(stats, HIRA_MAX_LEVELS + 1, pairs);
            }
        };
        // ---- the best selected score of every head among rows just scored (zmax), the new
        // running maximum, and what it does to the sums so far; head g lives in lane g; the
        // weights are computed with lane = (row, head), head = lane % GS.  Returns the running maximum of head
        // lane % GS (a finite stand-in for -inf) -----------------------
        auto raise_max = [&](float zmax) {
            zmax = cross_group_max<16>(zmax);
            const float mnew = fmaxf(m_run, zmax);
            const float f = (m_run == mnew) ? 1.0f : exp2f(m_run - mnew);
            m_run = mnew;
            if (__ballot(f != 1.0f) != 0ull) {  // uniform
                l_mine *= of_head<GS>(f);
#pragma unroll
                for (int g = 0; g < GS; ++g) {
                    const float fg = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(f), g));
                    if constexpr (WIDE) {
#pragma unroll
                        for (int j = 0; j < 8; ++j) acc8[g][j] *= fg;
                    } else {
#pragma unroll
                        for (int e = 0; e < VPL; ++e) acc[g][e] *= fg;
                    }
                }
            }
            // a head without a selected key has m = -inf and only z = -inf: any finite stand-in
            return of_head<GS>(mnew == -INFINITY ? 0.0f : mnew);
        };
        constexpr int RP = 64 / GS;               // rows whose weights one pass over the lanes computes
        constexpr int NPASS = kVBatch / RP;       // GS = 4: 2, GS = 8: 4, GS = 16: 8
        if constexpr (Q8) {
            // ---- 8-bit shadow: first all tiles, then all rows.  A wave goes through its nodes and lists the rows that
            // the shadow cannot rule out, with the heads they passed for: a word a row.  Behind a barrier the rows of all
            // waves (but the first few of each) are dealt out evenly, kQ8Batch of a wave at a time: their values and keys asked for together, the exact
            // test, the running maximum raised to the batch's best scores, the values into the sums.  (Rows looked at
            // round by round, a batch of 32 places for the twelve that a round of four nodes lists on average, cost every
            // round a trip to memory, and a wave with many rows kept its workgroup: a step of 8 trees x 131072 keys x 8 heads
            // 63.6 us instead of 56.  What bounds it now is the rows phase, a burst of 51 MB of scattered rows.)
            constexpr int CAP = S::CAP;
            uint32_t* const lists = s_words;                                                   // (waves, CAP)
            float* const ztab = reinterpret_cast<float*>(s_words + kMfmaWaves * CAP) + wave * (kQ8Batch * GS);
            uint32_t* const b_row = s_words + kMfmaWaves * (CAP + kQ8Batch * GS) + wave * (4 * kQ8Batch);
            uint32_t* const b_word = b_row + 2 * kQ8Batch;
            const float slack = su * (kQ8QuerySlack * 127.0f * (float)D), inv_su = 1.0f / su;
            for (int c0 = 0; c0 < rounds; c0 += S::CHUNK) {  // uniform in the workgroup
                if (c0 > 0) __syncthreads();  // (the rows listed before have been dealt with)
                const int c1 = min(c0 + S::CHUNK, rounds);
                int nl = 0;  // rows on my list
                fetch(c0, -1);
                for (int r = c0; r < c1; ++r) {  // uniform
#pragma unroll
                    for (int u = 0; u < NB; ++u) {
                        const int node = nx_node[u], cnt = nx_cnt[u];
                        const uint32_t heads = nx_mask[u];
                        // the score q.k lies within `marg` of su * (the integer): the keys' rounding
                        // (nx_eps steps a component at most) and the query's (kQ8QuerySlack steps of su)
                        const float marg = (nx_eps[u] + kQ8KeySlack) * asum + slack;
                        i32x4_t est[MT];
#pragma unroll
                        for (int tt = 0; tt < MT; ++tt)  // (every tile: one that is not there came as zeros)
                            est[tt] = tile_scores_i8<KS8>(a[u][tt], bq8h, bq8l);
                        fetch(r + 1 < c1 ? r + 1 : 1 << 20, u);  // (past the last round: no node, nothing read)
                        if (cnt == 0) continue;  // uniform
                        if (stats && lane == 0) stat_add(stats, 0, (unsigned)cnt);
                        // (in whole steps, one below: the comparison is one of integers)
                        const float thr = (tau - marg - 1e-6f * (fabsf(tau) + marg)) * inv_su;
                        const int least = head_ok && ((heads >> col) & 1u) ? (int)fminf(fmaxf(thr - 1.0f, -2e9f), 2e9f) - 1 : INT32_MAX;
#pragma unroll
                        for (int tt = 0; tt < MT; ++tt) {
                            if (tt * 16 >= cnt) continue;  // uniform
                            unsigned long long pass[4];
#pragma unroll
                            for (int j = 0; j < 4; ++j) pass[j] = __ballot(est[tt][j] >= least);
                            if ((pass[0] | pass[1] | pass[2] | pass[3]) == 0ull) continue;  // uniform
                            // row 4 k + j of the tile: its heads are field k of pass[j]; lane i < 16 takes row i
                            const int j = lane & 3;
                            const unsigned long long mine = j == 0 ? pass[0] : j == 1 ? pass[1] : j == 2 ? pass[2] : pass[3];
                            const uint32_t who = (uint32_t)(mine >> (16 * ((lane >> 2) & 3))) & 0xffffu;
                            const bool in = lane < 16 && who != 0u && tt * 16 + lane < cnt;
                            const unsigned long long rows = __ballot(in);
                            if (in)
                                lists[wave * CAP + nl + __popcll(rows & ((1ull << lane) - 1ull))] =
                                    (uint32_t)node | ((uint32_t)(tt * 16 + lane) << 8) | (who << 16);
                            nl += __popcll(rows);
                        }
                    }
                }
                // sixteen rows at a time, the next sixteen on their way meanwhile: what LDS says about them and their loads
                constexpr int NLD = WIDE ? kQ8Batch / RPI : 1;
                struct Batch {
                    uint4 kr[KS];   // the exact test's A operand: lane (kb, i) holds columns [32 s + 8 kb, +8) of the i-th row
                    uint4 vr[NLD];  // WIDE: values, lane (row group, chunk)
                    uint32_t vraw[WIDE ? 1 : kQ8Batch][VW];
                };
                // row `lane` of a batch: what its list says (0: it is not there)
                auto ask = [&](uint32_t word, int half, Batch& o) {
                    uint32_t* const row_at = b_row + half * kQ8Batch;
                    if (lane < kQ8Batch) {
                        b_word[half * kQ8Batch + lane] = word;
                        // (past the end: beyond the buffer, zeros and no memory access)
                        row_at[lane] = word != 0u ? ((uint32_t)(node_of((int)(word & 0xffu)) * bf) + ((word >> 8) & 0x3fu)) * (uint32_t)(D * 2) : 0xfffff000u;
                    }
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    if (want_attn) {
                        if constexpr (WIDE) {
#pragma unroll
                            for (int i = 0; i < NLD; ++i)
                                o.vr[i] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(
                                                                        vrsrc, row_at[i * RPI + rg] + (unsigned)cc * 16u, 0, 0));
                        } else {
                            const int rows = (int)row_at[lane & (kQ8Batch - 1)];
#pragma unroll
                            for (int i = 0; i < kQ8Batch; ++i) {
                                const unsigned at = (unsigned)__builtin_amdgcn_readlane(rows, i) + (unsigned)lane * (unsigned)(VPL * 2);
                                if (VPL == 1) o.vraw[i][0] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b16(vrsrc, at, 0, 0);
                                else o.vraw[i][0] = __builtin_amdgcn_raw_buffer_load_b32(vrsrc, at, 0, 0);
                            }
                        }
                    }
#pragma unroll
                    for (int s = 0; s < KS; ++s)
                        o.kr[s] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(
                                                                krsrc, row_at[col] + (unsigned)(kb * 16 + s * 64), 0, 0));
                    __builtin_amdgcn_sched_barrier(0);
                };
                // The first sixteen of a list are its wave's, asked for ahead of the barrier; what is left of the lists
                // is dealt out behind it.  (8 trees x 131072 keys x 8 heads 57.2 -> 56.0 us; 32 of them: 56.2.)
                Batch even, odd;
                const int own = min(nl, kQ8Batch);
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                ask(lane < own ? lists[wave * CAP + lane] : 0u, 0, even);
                if (lane == 0) s_rows[wave] = nl;
                if (c0 == 0) {
                    tline.stamp_wave(kTlWaveScanned);
                    tline.stamp(kTlListed);
                    tline.set(kTlRows, (unsigned long long)nl);
                    tline.set(kTlRounds, (unsigned long long)rounds);
                }
                tline.add_rows(nl);
                __syncthreads();
                int ahead[kMfmaWaves + 1];  // rows left on the lists of the waves ahead
                ahead[0] = 0;
                int total = 0;
#pragma unroll
                for (int w = 0; w < kMfmaWaves; ++w) {
                    const int listed = w < nw ? s_rows[w] : 0;
                    ahead[w + 1] = ahead[w] + max(listed - kQ8Batch, 0);
                    total += listed;
                }
                const int left = __builtin_amdgcn_readfirstlane(ahead[kMfmaWaves]);
                const int q0 = left * wave / nw, q1 = left * (wave + 1) / nw;  // my rows of them
                if (stats && lane == 0 && wave == 0) stat_add(stats, HIRA_MAX_LEVELS + 2, (unsigned)total);
                auto dealt = [&](int e0) {  // word of row e0 + lane of mine
                    const int q = max(min(e0 + lane, q1 - 1), 0);
                    int at = q + kQ8Batch;  // (of wave w's list, behind those ahead)
#pragma unroll
                    for (int w = 1; w < kMfmaWaves; ++w) at = q >= ahead[w] ? w * CAP + kQ8Batch + q - ahead[w] : at;
                    return lane < kQ8Batch && e0 + lane < q1 ? lists[at] : 0u;
                };
                // (selection lists: every wave is here as often as any other)
                auto use = [&](int there, int half, const Batch& o) {  // so many rows of it
                    const bool lists_out = OUT && p.sel_count != nullptr;  // uniform in the launch
                    if (there <= 0 && !lists_out) return;  // uniform
                    const f32x4_t sco = tile_scores_lds<KS>(o.kr, s_bq, lane);
                    const uint4 w4 = *reinterpret_cast<const uint4*>(b_word + half * kQ8Batch + 4 * kb);
                    const uint32_t words[4] = {w4.x, w4.y, w4.z, w4.w};
                    unsigned sel4 = 0u;
                    float zmax = -INFINITY;
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        // (its head must be one the shadow let the row pass for)
                        const bool sel = ((words[j] >> 16 >> col) & 1u) != 0u && sco[j] >= tau;
                        if (sel) sel4 |= 1u << j;
                        const float z = sel ? sco[j] * sc2 : -INFINITY;
                        zmax = fmaxf(zmax, z);
                        if (col < GS) ztab[(4 * kb + j) * GS + col] = z;
                    }
                    if (stats) count_selected(sel4, rows_of(sel4));
                    if (OUT && (p.dense != nullptr || p.sel_count != nullptr)) {
                        const uint4 r4 = *reinterpret_cast<const uint4*>(b_row + half * kQ8Batch + 4 * kb);
                        const unsigned slot4[4] = {r4.x / (D * 2), r4.y / (D * 2), r4.z / (D * 2), r4.w / (D * 2)};
                        // One atomic per head of the workgroup's batches: all waves have their rows at once, and with
                        // one each they stood in line for the few cache lines that all heads' counters are.  (Lists,
                        // 8 heads a tree: 8 x 32768 keys of fan-out 64, 1 % selected, 33.6 -> 21.0 us, 8 x 131072, 10 %,
                        // 256 -> 93; round by round, before there were two phases, 26.3 and 256.)
                        emit(col, kb, sel4, sco, slot4, [&](int mine) {
                            if (kb == 0) s_places[wave * 16 + col] = mine;
                            __syncthreads();
                            int before = 0, all = 0;
#pragma unroll
                            for (int w = 0; w < kMfmaWaves; ++w) {
                                const int n = w < nw ? s_places[w * 16 + col] : 0;
                                if (w < wave) before += n;
                                all += n;
                            }
                            if (wave == 0 && kb == 0) s_place0[col] = all > 0 ? atomicAdd(&p.sel_count[qh], all) : 0;
                            __syncthreads();
                            return s_place0[col] + before;
                        });
                    }
                    if (!want_attn || there <= 0) return;  // uniform
                    const float m_lane = raise_max(zmax);
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    // scores -> weights, in place, 64 (row, head) pairs at a time (past the end: -inf, nothing)
                    uint64_t taken[kQ8Batch / RP];  // pairs of a row and a head that selects it
#pragma unroll
                    for (int ps = 0; ps < kQ8Batch / RP; ++ps) {
                        float* zp = ztab + ps * 64 + lane;
                        const float z = *zp, w = __builtin_amdgcn_exp2f(z - m_lane);
                        taken[ps] = __ballot(z != -INFINITY);
                        l_mine += w;
                        *zp = w;
                    }
                    // The values of a row that no head selects may be anything: zeros in their place.  (They came with the
                    // rest: the shadow lets few rows pass in vain.)  Is row i0 + more one that some head selects?  (The
                    // pairs of both lie in the same 32.)
                    auto some = [&](int i0, int more) {
                        const uint32_t w = (uint32_t)(taken[i0 / RP] >> (i0 % RP * GS / 32 * 32));
                        return ((w >> (i0 % RP * GS % 32 + more * GS)) & ((1u << GS) - 1u)) != 0u;
                    };
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    if constexpr (WIDE) {
#pragma unroll
                        for (int i = 0; i < NLD; ++i) {
                            if (i * RPI >= there) break;  // uniform
                            float wv[GS];
#pragma unroll
                            for (int g4 = 0; g4 < GS / 4; ++g4) {
                                const float4 w = *reinterpret_cast<const float4*>(ztab + (i * RPI + rg) * GS + 4 * g4);
                                wv[4 * g4 + 0] = w.x;
                                wv[4 * g4 + 1] = w.y;
                                wv[4 * g4 + 2] = w.z;
                                wv[4 * g4 + 3] = w.w;
                            }
                            float vf[8];
                            static_assert(RPI * GS <= 32, "");
                            unpack<bf16_t>(some(i * RPI, rg) ? o.vr[i] : make_uint4(0, 0, 0, 0), vf);
#pragma unroll
                            for (int g = 0; g < GS; ++g)
#pragma unroll
                                for (int j = 0; j < 8; ++j) acc8[g][j] += wv[g] * vf[j];
                        }
                    } else {
#pragma unroll
                        for (int i = 0; i < kQ8Batch; ++i) {
                            if ((i & 7) == 0 && i >= there) break;  // uniform
                            float vf[VPL];
                            const uint32_t v = some(i, 0) ? o.vraw[i][0] : 0u;
                            vf[0] = bf16_lo(v);
                            if (VPL > 1) vf[VPL - 1] = bf16_hi(v);
                            const float* wr = ztab + i * GS;  // (a broadcast read)
#pragma unroll
                            for (int g = 0; g < GS; ++g)
#pragma unroll
                                for (int e = 0; e < VPL; ++e) acc[g][e] += wr[g] * vf[e];
                        }
                    }
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // (the next sixteen write where these read)
                };
                const int end = OUT ? q0 + (left + nw - 1) / nw : q1;  // (OUT: as many steps in every wave)
                for (int e0 = q0 - kQ8Batch; e0 < end; e0 += 2 * kQ8Batch) {  // uniform in the wave
                    ask(dealt(e0 + kQ8Batch), 1, odd);
                    use(e0 < q0 ? own : q1 - e0, 0, even);
                    if (c0 == 0 && e0 < q0) tline.stamp_wave(kTlWaveIssued);
                    // (no wave has more than its first sixteen, uniform in the workgroup: lists of 8 x 4096 keys, 16 heads a
                    // tree, 12.7 -> 11.6 us.  Attention alone gains nothing: 8 x 131072 keys 50.2 -> 50.6.)
                    if (OUT && left == 0) break;
                    ask(dealt(e0 + 2 * kQ8Batch), 0, even);
                    use(q1 - e0 - kQ8Batch, 1, odd);
                    if (c0 == 0 && e0 < q0) tline.stamp_wave(kTlWaveConsumed);
                }
                if (c0 == 0) tline.stamp(kTlGathered);
            }
        } else {
            // one round of a wave
            auto do_round = [&](const int r) {
                constexpr bool SINGLE = ONE;
                // the round's score table and row list; every wave has a stretch of ROWS * NB rows of
                // its own and nobody else looks at it: no barrier inside the rounds
                uint32_t* lst_row = s_words;                                        // (LIST) listed row -> table row
                uint32_t* lst_tslot = lst_row + S::LIST;                            // (LIST/16) table tile -> key slot
                float* lst_z = reinterpret_cast<float*>(lst_tslot + S::LIST / 16);  // (LIST, GS) the table

                // ---- scan: the key tiles of this round's nodes were asked for a round ago; node by
                // node: the products, at once the request for the node that takes its place in the
                // next round, then the node's bookkeeping while the other tiles arrive -------------------
                // The bookkeeping below derives everything per-lane from this copy, which the compiler
                // cannot see through: otherwise it computes those values once, ahead of the loop, and
                // they crowd out the registers that the loads above need.
                int lane_o = lane;
                asm volatile("" : "+v"(lane_o));
                const int col = lane_o & 15, kb = lane_o >> 4;

                int nsel = 0;  // rows of my stretch of the list
                float zmax = -INFINITY;
                const int zrow0 = wave * (NB * S::ROWS);  // my stretch of the round's rows
                int node[NB], cnt[NB];
                uint32_t nmask[NB];
#pragma unroll
                for (int u = 0; u < NB; ++u) {
                    node[u] = nx_node[u];
                    cnt[u] = nx_cnt[u];
                    nmask[u] = nx_mask[u];
                    const unsigned slot0 = (unsigned)(node_of(max(node[u], 0)) * bf) + (unsigned)(nx_half[u] * MT * 16);
                    if (AHEAD && cnt[u] == 0) continue;  // uniform
                    f32x4_t sco_u[MT];
#pragma unroll
                    for (int tt = 0; tt < MT; ++tt)  // (a tile that is not there came as zeros)
                        sco_u[tt] = tile_scores_lds<KS>(a[u][tt], s_bq, lane);
                    if (r == 0 && u == 0) tline.stamp(kTlTiles);
                    if constexpr (!SINGLE) fetch(r + 1, u);  // (past the last round: no node, nothing read)
                    // a head for which the node did not survive selects nothing
                    const float tau_u = ((nmask[u] >> col) & 1u) ? tau : INFINITY;
                    if (stats && lane == 0) stat_add(stats, 0, (unsigned)cnt[u]);
#pragma unroll
                    for (int tt = 0; tt < MT; ++tt) {
                        if (tt * 16 >= cnt[u]) continue;  // uniform
                        const f32x4_t sco = sco_u[tt];
                        const int lim = cnt[u] - tt * 16 - 4 * kb;  // my rows j < lim hold keys
                        unsigned sel4 = 0u;
#pragma unroll
                        for (int j = 0; j < 4; ++j)
                            if (sco[j] >= tau_u && j < lim) sel4 |= 1u << j;
                        if (__ballot(sel4 != 0u) == 0ull) continue;  // uniform
                        const unsigned rowmask = rows_of(sel4);  // rows selected by some head
                        if (stats) count_selected(sel4, rowmask);
                        const unsigned tslot = slot0 + tt * 16;

                        // ---- dense scores / compact lists ------------------------------------------
                        if (OUT && (p.dense != nullptr || p.sel_count != nullptr)) {
                            const unsigned slot4[4] = {tslot + 4 * kb, tslot + 4 * kb + 1, tslot + 4 * kb + 2,
                                                       tslot + 4 * kb + 3};
                            emit(col, kb, sel4, sco, slot4, [&](int mine) {  // one atomic per head of the tile
                                int b0 = 0;
                                if (kb == 0 && mine > 0) b0 = atomicAdd(&p.sel_count[qh], mine);
                                return __shfl(b0, col, 64);
                            });
                        }

                        // ---- the tile's scores go to the table, its selected rows join my list -----------
                        if (want_attn) {
                            const int trow = zrow0 + (u * MT + tt) * 16;  // the tile's rows in the table
                            float zs[4];
#pragma unroll
                            for (int j = 0; j < 4; ++j) {
                                zs[j] = ((sel4 >> j) & 1u) ? sco[j] * sc2 : -INFINITY;
                                zmax = fmaxf(zmax, zs[j]);
                            }
                            if (col < GS) {
                                float* zp = lst_z + (trow + 4 * kb) * GS + col;
#pragma unroll
                                for (int j = 0; j < 4; ++j) zp[j * GS] = zs[j];
                            }
                            if (lane_o < 16 && ((rowmask >> lane_o) & 1u))
                                lst_row[zrow0 + nsel + __popc(rowmask & ((1u << lane_o) - 1u))] = (uint32_t)(trow + lane_o);
                            if (lane_o == 0) lst_tslot[trow >> 4] = tslot;
                        }
                        nsel += __popc(rowmask);
                    }
                }
                const int tot = nsel;  // rows on my list
                if (r == 0) {
                    tline.stamp_wave(kTlWaveScanned);
                    tline.stamp(kTlListed);
                    tline.set(kTlRows, (unsigned long long)tot);
                    tline.set(kTlRounds, (unsigned long long)rounds);
                }
                tline.add_rows(tot);

                // ---- value rows: kVBatch in flight; the rows of a batch in the score table (lane =
                // (row of the pass, head)), their key slots, and the loads ---------------------------------
                auto issue = [&](int e0, int (&at_v)[NPASS], uint32_t (&vraw)[kVBatch][VW]) {
#pragma unroll
                    for (int ps = 0; ps < NPASS; ++ps) {
                        const int le = e0 + ps * RP + lane_o / GS;
                        at_v[ps] = le < tot ? (int)lst_row[zrow0 + le] : -1;  // (-1: past the end)
                    }
                    int slot_v[NPASS];  // the key slots of all the rows of a pass
#pragma unroll
                    for (int ps = 0; ps < NPASS; ++ps)
                        slot_v[ps] = at_v[ps] >= 0 ? (int)(lst_tslot[at_v[ps] >> 4] + (unsigned)(at_v[ps] & 15)) : 0;
                    // (a batch is always loaded whole, rows past the end as slot 0: straight-line code;
                    // loads under conditions of their own cost more than they save)
#pragma unroll
                    for (int i = 0; i < kVBatch; ++i) {
                        {
                            const unsigned slot = (unsigned)__builtin_amdgcn_readlane(slot_v[i / RP], (i % RP) * GS);
                            const unsigned voff = (unsigned)lane_o * (unsigned)(VPL * 2);
                            const unsigned soff = slot * (unsigned)(D * 2);
                            if (VPL == 1) {
                                vraw[i][0] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b16(vrsrc, voff, soff, POL == 2 ? kReadOnce : 0);
                            } else if (VPL == 2) {
                                vraw[i][0] = __builtin_amdgcn_raw_buffer_load_b32(vrsrc, voff, soff, POL == 2 ? kReadOnce : 0);
                            } else {
                                const u32x2_t v2 = __builtin_amdgcn_raw_buffer_load_b64(vrsrc, voff, soff, POL == 2 ? kReadOnce : 0);
                                vraw[i][0] = v2.x;
                                vraw[i][VW - 1] = v2.y;
                            }
                        }
                    }
                };
                float m_lane = 0.0f;  // (see raise_max)
                // ---- a batch of value rows into the sums -----------------------------------------------
                auto consume = [&](int e0, const int (&at_v)[NPASS], const uint32_t (&vraw)[kVBatch][VW]) {
                    // (nothing of what follows may be scheduled ahead of loads issued before this point)
                    __builtin_amdgcn_sched_barrier(0);
                    // scores -> weights, in place, 64 (row, head) pairs at a time
#pragma unroll
                    for (int ps = 0; ps < NPASS; ++ps) {
                        if (at_v[ps] >= 0) {
                            float* zp = lst_z + at_v[ps] * GS + (lane_o & (GS - 1));
                            const float w = __builtin_amdgcn_exp2f(*zp - m_lane);
                            l_mine += w;
                            *zp = w;
                        }
                    }
                    // eight rows at a time: one test whether the list goes that far, no branch between
                    // the rows of an eight (their weights and products can then be in flight together);
                    // a row past the end reads the weights of the batch's first row and counts for nothing
                    const int at_first = __builtin_amdgcn_readlane(at_v[0], 0);
#pragma unroll
                    for (int i = 0; i < kVBatch; ++i) {
                        if ((i & 7) == 0 && e0 + i >= tot) break;  // uniform
                        const bool there = e0 + i < tot;           // uniform
                        const int at_i = __builtin_amdgcn_readlane(at_v[i / RP], (i % RP) * GS);
                        const int at = there ? at_i : at_first;
                        float vf[VPL];
                        if (VPL == 1) {
                            vf[0] = there ? bf16_lo(vraw[i][0]) : 0.0f;
                        } else {
#pragma unroll
                            for (int e = 0; e < VPL / 2; ++e) {
                                vf[2 * e] = there ? bf16_lo(vraw[i][e]) : 0.0f;
                                vf[2 * e + 1] = there ? bf16_hi(vraw[i][e]) : 0.0f;
                            }
                        }
                        const float* wr = lst_z + at * GS;  // weights of this row, one per head
#pragma unroll
                        for (int g = 0; g < GS; ++g) {
                            const float w = wr[g];  // same address in every lane: a broadcast read
#pragma unroll
                            for (int e = 0; e < VPL; ++e) acc[g][e] += w * vf[e];
                        }
                    }
                };
                if constexpr (WIDE) {
                    if (want_attn && tot > 0) {  // uniform in the launch / in the wave
                        constexpr int NLD = kVBatch / RPI;  // load instructions of a batch
                        for (int e0 = 0; e0 < tot; e0 += kVBatch) {  // uniform in the wave
                            // the batch's rows in the score table: for the weights (lane = (row of
                            // the pass, head)) and for the loads (lane = (row group, chunk))
                            int at_w[NPASS], at_r[NLD];
#pragma unroll
                            for (int ps = 0; ps < NPASS; ++ps) {
                                const int le = e0 + ps * RP + lane_o / GS;
                                at_w[ps] = le < tot ? (int)lst_row[zrow0 + le] : -1;  // (-1: past the end)
                            }
#pragma unroll
                            for (int i = 0; i < NLD; ++i) {
                                const int le = e0 + i * RPI + rg;
                                at_r[i] = le < tot ? (int)lst_row[zrow0 + le] : -1;
                            }
                            uint4 vr[NLD];
#pragma unroll
                            for (int i = 0; i < NLD; ++i) {  // (rows past the end: slot 0, weight 0)
                                const unsigned slot =
                                    at_r[i] >= 0 ? lst_tslot[at_r[i] >> 4] + (unsigned)(at_r[i] & 15) : 0u;
                                vr[i] = __builtin_bit_cast(
                                    uint4, __builtin_amdgcn_raw_buffer_load_b128(
                                               vrsrc, slot * (unsigned)(D * 2) + (unsigned)cc * 16u, 0,
                                               POL == 2 ? kReadOnce : 0));
                            }
                            if (r == 0 && e0 == 0) tline.stamp_wave(kTlWaveIssued);
                            __builtin_amdgcn_sched_barrier(0);
                            if (e0 == 0) m_lane = raise_max(zmax);  // (while the first values are on their way)
                            // scores -> weights, in place, 64 (row, head) pairs at a time
#pragma unroll
                            for (int ps = 0; ps < NPASS; ++ps) {
                                if (at_w[ps] >= 0) {
                                    float* zp = lst_z + at_w[ps] * GS + (lane_o & (GS - 1));
                                    const float w = __builtin_amdgcn_exp2f(*zp - m_lane);
                                    l_mine += w;
                                    *zp = w;
                                }
                            }
#pragma unroll
                            for (int i = 0; i < NLD; ++i) {
                                if (e0 + i * RPI >= tot) break;  // uniform
                                float wv[GS];
#pragma unroll
                                for (int g4 = 0; g4 < GS / 4; ++g4) {
                                    float4 w4 = make_float4(0.f, 0.f, 0.f, 0.f);
                                    if (at_r[i] >= 0)
                                        w4 = *reinterpret_cast<const float4*>(lst_z + at_r[i] * GS + 4 * g4);
                                    wv[4 * g4 + 0] = w4.x;
                                    wv[4 * g4 + 1] = w4.y;
                                    wv[4 * g4 + 2] = w4.z;
                                    wv[4 * g4 + 3] = w4.w;
                                }
                                const uint4 raw = at_r[i] >= 0 ? vr[i] : make_uint4(0, 0, 0, 0);
                                float vf[8];
                                unpack<bf16_t>(raw, vf);
#pragma unroll
                                for (int g = 0; g < GS; ++g)
#pragma unroll
                                    for (int j = 0; j < 8; ++j) acc8[g][j] += wv[g] * vf[j];
                            }
                            if (r == 0 && e0 == 0) tline.stamp_wave(kTlWaveConsumed);
                        }
                    }
                } else
                if (want_attn && tot > 0) {  // uniform in the launch / in the wave
                    m_lane = raise_max(zmax);
                    for (int e0 = 0; e0 < tot; e0 += kVBatch) {  // uniform in the wave
                        int at_v[NPASS];
                        uint32_t vraw[kVBatch][VW];
                        issue(e0, at_v, vraw);
                        if (r == 0 && e0 == 0) tline.stamp_wave(kTlWaveIssued);
                        consume(e0, at_v, vraw);
                        if (r == 0 && e0 == 0) tline.stamp_wave(kTlWaveConsumed);
                    }
                }
                if (r == 0) tline.stamp(kTlGathered);
            };
            if constexpr (ONE) {
                if (rounds > 0) do_round(0);
            } else {
                for (int r = 0; r < rounds; ++r) do_round(r);  // uniform in the workgroup
            }
        }  // shadow or bf16 tiles
    }  // tree or queue
    if (!want_attn) return;  // uniform
    tline.stamp_wave(kTlWaveEnd);
    tline.set_wave(kTlWaveRows, tline.rows);
    tline.stamp(kTlWave0Done);

    // ---- merge the waves: first one maximum per head for the workgroup, to which every wave
    // brings its sums (m_run: lane = head col; l_mine: head lane % GS); then l and acc add up ---
    if (kb == 0) s_mxw[wave * 16 + col] = m_run;
    const bool wide = WIDE && !is_queue;  // uniform: my sums are in acc8
    __syncthreads();
    {
        float m_all = -INFINITY;
        for (int w = 0; w < nw; ++w) m_all = fmaxf(m_all, s_mxw[w * 16 + col]);
        const float fw = m_run == -INFINITY ? 0.0f : exp2f(m_run - m_all);
        l_mine *= of_head<GS>(fw);
#pragma unroll
        for (int g = 0; g < GS; ++g) {
            const float fg = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(fw), g));
#pragma unroll
            for (int e = 0; e < VPL; ++e) acc[g][e] *= fg;
            if constexpr (WIDE) {
#pragma unroll
                for (int j = 0; j < 8; ++j) acc8[g][j] *= fg;
            }
        }
        m_run = m_all;
    }
    l_mine = cross_group_sum<GS>(l_mine);
    if (lane < GS) s_lw[wave * 16 + lane] = l_mine;
    if (wave == 0 && kb == 0) s_mh[col] = m_run;
    int tid = threadIdx.x;  // (opaque, like lane_o above: nothing of the merge is computed early)
    asm volatile("" : "+v"(tid));
    float* macc = reinterpret_cast<float*>(s_words);  // (nw, 4, D): four heads at a time
    const int P = p.num_parts;
    // a tree's only workgroup writes the output itself: no partial, no ticket, no fold (8 trees x 500 keys in
    // two levels: 9.2 -> 7.5 us)
    const bool alone = wgs == 1 && p.done != nullptr;  // uniform
#pragma unroll
    for (int c = 0; c < GS / 4; ++c) {
        if (c * 4 >= G) continue;  // uniform (no break: the loop has to unroll)
        __syncthreads();           // the list (or the previous four heads) is not needed any more
        if (wide) {
            if constexpr (WIDE) {
                // The four row groups' sums of the four heads meet so that group rg ends up with
                // head rg: the halves of the wave trade heads (0,1) against (2,3) -- one swap
                // leaves, in the lower half, both halves' sums of head 0 or 1, in the upper half
                // those of head 2 or 3 --, then the rows of 16 lanes trade (0,2) against (1,3).
                float mine[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const auto s02 = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc8[c * 4 + 0][j]),
                                                                      __float_as_uint(acc8[c * 4 + 2][j]), false, false);
                    const auto s13 = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc8[c * 4 + 1][j]),
                                                                      __float_as_uint(acc8[c * 4 + 3][j]), false, false);
                    const float r02 = __uint_as_float(s02[0]) + __uint_as_float(s02[1]);
                    const float r13 = __uint_as_float(s13[0]) + __uint_as_float(s13[1]);
                    const auto t = __builtin_amdgcn_permlane16_swap(__float_as_uint(r02), __float_as_uint(r13), false, false);
                    mine[j] = __uint_as_float(t[0]) + __uint_as_float(t[1]);
                }
                float4* dst = reinterpret_cast<float4*>(macc + (wave * 4 + ((tid & 63) / LR)) * D + ((tid & 63) % LR) * 8);
                dst[0] = make_float4(mine[0], mine[1], mine[2], mine[3]);
                dst[1] = make_float4(mine[4], mine[5], mine[6], mine[7]);
            }
        } else {
#pragma unroll
            for (int gi = 0; gi < 4; ++gi)
#pragma unroll
                for (int e = 0; e < VPL; ++e) macc[(wave * 4 + gi) * D + (tid & 63) * VPL + e] = acc[c * 4 + gi][e];
        }
        __syncthreads();
        if (c == 0) tline.stamp(kTlMerged);
        for (int t = tid; t < 4 * D; t += blockDim.x) {
            const int gi = t / D, e = t % D, g = c * 4 + gi;
            if (g >= G) break;
            float a_sum = 0.0f, lsum = 0.0f;
            for (int w = 0; w < nw; ++w) {
                a_sum += macc[(w * 4 + gi) * D + e];
                lsum += s_lw[w * 16 + g];
            }
            const int head = p.group_size > 0 ? hoff + g : p.tree_q_heads[hoff + g];
            if (alone) {
                store_out(p.attn_out, p.out_bf16, (size_t)head * D + e, lsum > 0.0f ? a_sum * (1.0f / lsum) : 0.0f);
                continue;
            }
            const size_t slot = (size_t)head * P + wg;
            // device-scope stores: written through, so that the workgroup that folds the
            // partials (maybe on another L2 slice) reads them without cache-wide flushes;
            // a head without a selected key only says so (m = -inf)
            if (lsum > 0.0f)
                __hip_atomic_store(&p.part_acc[slot * D + e], a_sum, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (e == 0) {
                __hip_atomic_store(&p.part_m[slot], lsum > 0.0f ? s_mh[g] : -INFINITY, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(&p.part_l[slot], lsum, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
    }
    tline.stamp(kTlStoresIssued);
    if constexpr (SAMPLED) {
        if (alone && wave == 0) sampled_ticket(p, tree, wgs, hoff, G);
    }
    if (p.done == nullptr || alone) return;  // the caller folds the partials in a second launch, or there is one

    // ---- the last workgroup of this tree (and pass) to arrive folds the tree's partials ----
    hand_off_release();
    tline.stamp(kTlStored);
    __syncthreads();
    if constexpr (SAMPLED) {
        if (wave == 0) {
            const bool last = sampled_ticket(p, tree, wgs, hoff, G);
            if (lane == 0) s_last = last;
        }
    } else if (threadIdx.x == 0) {
        int* ctr = p.done + (size_t)tree * gridDim.z + blockIdx.z;
        const int ticket = __hip_atomic_fetch_add(ctr, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        s_last = ticket == (int)gridDim.y - 1;
        if (s_last) __hip_atomic_store(ctr, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    tline.stamp(kTlTicket);
    if (!s_last) return;

    auto ld = [](const float* q) {
        return __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    // Up to 16 partials in one trip to memory and without a barrier: a thread owns four columns of a head and
    // asks for maximum, sum and columns of all of them at once.  8 trees x 4 heads, with phases 1 and 2
    // below before: 4 partials a head 12.35 -> 11.2 us, 16 partials 13.8 -> 13.0 (13.5 where half of them
    // hold nothing -> 13.1).  With the 32 of a compute unit each it loses where many hold nothing (shared
    // out over the threads, which then meet in LDS: 14.6 -> 14.9 at 16000 keys whose balls prune half).
    auto few = [&](auto count, int g, int qd) {
        constexpr int N = decltype(count)::value;
        // (the descriptor is the tree's, the same in every lane; its heads are consecutive)
        const __amdgpu_buffer_rsrc_t arsrc = make_rsrc(p.part_acc + (size_t)hoff * P * D, 0x7fffffff);
        const float* pm = p.part_m + (size_t)(hoff + g) * P;
        const float* pl = p.part_l + (size_t)(hoff + g) * P;
        float m[N], l[N], M = -INFINITY, Lh = 0.0f;
        f32x4_t v[N], sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < N; ++i) {  // (beyond the last: the last one again, which then counts for nothing)
            const int pi = min(i, P - 1);
            m[i] = ld(pm + pi);
            l[i] = ld(pl + pi);
            v[i] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(  // (16: the device-scope bit)
                                                   arsrc, (unsigned)((g * P + pi) * D + 4 * qd) * 4u, 0, 16));
        }
#pragma unroll
        for (int i = 0; i < N; ++i) M = fmaxf(M, m[i]);
#pragma unroll
        for (int i = 0; i < N; ++i) {
            // (a partial without a selected key may hold anything: left out, not multiplied)
            const float w = i < P && m[i] > -INFINITY ? exp2f(m[i] - M) : 0.0f;
            if (w > 0.0f) {
                Lh += w * l[i];
                sum += w * v[i];
            }
        }
        const float inv = Lh > 0.0f ? 1.0f / Lh : 0.0f;
#pragma unroll
        for (int c = 0; c < 4; ++c)
            store_out(p.attn_out, p.out_bf16, (size_t)(hoff + g) * D + 4 * qd + c, sum[c] * inv);
    };
    if (P <= 16 && p.group_size > 0) {  // uniform
        auto all = [&](auto count) {
            for (int item = tid; item < G * (D / 4); item += blockDim.x) few(count, item / (D / 4), item % (D / 4));
        };
        if (P <= 4) all(std::integral_constant<int, 4>{});
        else if (P <= 8) all(std::integral_constant<int, 8>{});
        else all(std::integral_constant<int, 16>{});
        tline.stamp(kTlFoldDone);
        return;
    }
    // phase 1: wave w handles heads w, w + nw, ...: M = max m_p, L = sum 2^(m_p - M) l_p, and
    // the list of the partials that hold anything, with their weights 2^(m_p - M)
    const bool listed = 2 * (size_t)G * P <= (size_t)S::WORDS;
    int* clist = reinterpret_cast<int*>(s_words);                // (G, P)
    float* cwt = reinterpret_cast<float*>(s_words) + (size_t)G * P;  // (G, P)
    for (int g = wave; g < G; g += nw) {
        const int head = p.group_size > 0 ? hoff + g : p.tree_q_heads[hoff + g];
        const float* pm = p.part_m + (size_t)head * P;
        const float* pl = p.part_l + (size_t)head * P;
        const float mp0 = lane < P ? ld(pm + lane) : -INFINITY;
        const float lp0 = lane < P ? ld(pl + lane) : 0.0f;
        float mx = mp0;
        for (int i = lane + 64; i < P; i += 64) mx = fmaxf(mx, ld(pm + i));
        mx = wave_max(mx);
        float ls = 0.0f;
        int nc = 0;
        for (int i0 = 0; i0 < P; i0 += 64) {  // uniform
            const int i = i0 + lane;
            const float mp = i0 == 0 ? mp0 : (i < P ? ld(pm + i) : -INFINITY);
            const float lp = i0 == 0 ? lp0 : (i < P ? ld(pl + i) : 0.0f);
            const float w = (mp > -INFINITY) ? exp2f(mp - mx) : 0.0f;
            ls += w * lp;
            const bool nz = w > 0.0f && lp > 0.0f;
            const unsigned long long bal = __ballot(nz);
            if (listed && nz) {
                const int k = nc + __popcll(bal & ((1ull << lane) - 1ull));
                clist[g * P + k] = i;
                cwt[g * P + k] = w;
            }
            nc += __popcll(bal);
        }
        ls = wave_sum(ls);
        if (lane == 0) {
            s_red[2 * g] = mx;
            s_red[2 * g + 1] = ls;
            s_nc[g] = nc;
        }
    }
    __syncthreads();
    tline.stamp(kTlFoldListed);
    // phase 2, only partials that hold something.  Where the heads of the tree are consecutive and
    // the workgroup has threads to spare: a thread owns four output columns of a head and every
    // n_grp-th listed partial, eight 16-byte loads in flight (one or two trips to memory for the
    // whole fold instead of one per eight partials and column); the groups' sums meet in LDS.
    // Worth its set-up where the other way takes more than four trips (measured: 8 heads x 32
    // partials 5.9 -> 3.5 us; 4 heads x 32 partials 0.3 us slower).
    const int items = G * (D / 4);
    const int n_grp = items <= (int)blockDim.x ? (int)blockDim.x / items : 0;
    const int narrow_trips = ((G * D + (int)blockDim.x - 1) / (int)blockDim.x) * ((P + 7) / 8);
    if (narrow_trips > 4 && listed && p.group_size > 0 && n_grp >= 1 &&
        2 * (size_t)G * P + (size_t)n_grp * G * D <= (size_t)S::WORDS) {
        float* red = reinterpret_cast<float*>(s_words) + 2 * (size_t)G * P;  // (n_grp, G, D)
        const __amdgpu_buffer_rsrc_t arsrc =
            make_rsrc(p.part_acc + (size_t)hoff * P * D, (size_t)G * P * D * sizeof(float));
        const int item = tid % items, grp = tid / items;
        if (grp < n_grp) {
            const int g = item / (D / 4), qd = item % (D / 4);
            const int nc = s_red[2 * g + 1] > 0.0f ? s_nc[g] : 0;
            const int* cl = clist + g * P;
            const float* cw = cwt + g * P;
            const unsigned col0 = ((unsigned)g * (unsigned)P * (unsigned)D + 4u * (unsigned)qd) * 4u;
            float sx = 0.0f, sy = 0.0f, sz = 0.0f, sw = 0.0f;
            for (int k0 = grp; k0 < nc; k0 += 8 * n_grp) {
                u32x4_t v[8];
#pragma unroll
                for (int u = 0; u < 8; ++u)  // (16: the device-scope bit, as in `ld` above)
                    v[u] = __builtin_amdgcn_raw_buffer_load_b128(
                        arsrc, col0 + (unsigned)cl[min(k0 + u * n_grp, nc - 1)] * (unsigned)(D * 4), 0, 16);
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const float w = k0 + u * n_grp < nc ? cw[k0 + u * n_grp] : 0.0f;
                    sx += w * __uint_as_float(v[u].x);
                    sy += w * __uint_as_float(v[u].y);
                    sz += w * __uint_as_float(v[u].z);
                    sw += w * __uint_as_float(v[u].w);
                }
            }
            *reinterpret_cast<float4*>(red + ((size_t)grp * G + g) * D + 4 * qd) = make_float4(sx, sy, sz, sw);
        }
        __syncthreads();
        for (int t = tid; t < G * D; t += blockDim.x) {
            const int g = t / D;
            const float Lg = s_red[2 * g + 1];
            float sum = 0.0f;
            for (int r = 0; r < n_grp; ++r) sum += red[(size_t)r * G * D + t];
            store_out(p.attn_out, p.out_bf16, (size_t)(hoff + g) * D + (t % D), Lg > 0.0f ? sum / Lg : 0.0f);
        }
        tline.stamp(kTlFoldDone);
        return;
    }
    // otherwise: thread t owns output column e of head g
    for (int t = tid; t < G * D; t += blockDim.x) {
        const int g = t / D, e = t % D;
        const int head = p.group_size > 0 ? hoff + g : p.tree_q_heads[hoff + g];
        const float M = s_red[2 * g], Lg = s_red[2 * g + 1];
        const float* pm = p.part_m + (size_t)head * P;
        const float* pa = p.part_acc + (size_t)head * P * D + e;
        float s0 = 0.0f, s1 = 0.0f;
        if (Lg > 0.0f) {
            if (listed) {
                const int nc = s_nc[g];
                const int* cl = clist + g * P;
                const float* cw = cwt + g * P;
                int k = 0;
                for (; k + 8 < nc; k += 16) {  // uniform over the columns of a head (32 in flight: slower)
                    float v[16];
#pragma unroll
                    for (int u = 0; u < 16; ++u) v[u] = ld(pa + (size_t)cl[min(k + u, nc - 1)] * D);
#pragma unroll
                    for (int u = 0; u < 16; u += 2) {
                        s0 += (k + u < nc ? cw[k + u] : 0.0f) * v[u];
                        s1 += (k + u + 1 < nc ? cw[k + u + 1] : 0.0f) * v[u + 1];
                    }
                }
                for (; k < nc; k += 8) {  // (at most eight are left)
                    float v[8];
#pragma unroll
                    for (int u = 0; u < 8; ++u) v[u] = ld(pa + (size_t)cl[min(k + u, nc - 1)] * D);
#pragma unroll
                    for (int u = 0; u < 8; u += 2) {
                        s0 += (k + u < nc ? cw[k + u] : 0.0f) * v[u];
                        s1 += (k + u + 1 < nc ? cw[k + u + 1] : 0.0f) * v[u + 1];
                    }
                }
            } else {
                for (int i = 0; i < P; ++i) {
                    const float mi = ld(pm + i);
                    const float w = mi > -INFINITY ? exp2f(mi - M) : 0.0f;
                    if (w > 0.0f) s0 += w * ld(pa + (size_t)i * D);
                }
            }
        }
        const float inv = Lg > 0.0f ? 1.0f / Lg : 0.0f;
        store_out(p.attn_out, p.out_bf16, (size_t)head * D + e, (s0 + s1) * inv);
    }
    tline.stamp(kTlFoldDone);
}

// the attention-only scan of bf16 tiles has an instantiation for launches of a single round
template <int KS, int MT, int GS, bool Q8, int POL, int HV>
void launch_mfma_one(const SearchPlan& plan, const SearchParams& p, dim3 grid, hipStream_t s) {
    const dim3 block(plan.threads);
    const bool out = p.sample_wgs == 0 && (p.dense != nullptr || p.sel_count != nullptr);
    // nodes (entries of the survivors' list) a workgroup's tiles hold at most, against those its
    // waves take in one round
    const bool one = plan.nodes_per_wave * 16 * HV <= (plan.threads / 64) * MfmaShape<KS, MT, GS, Q8>::NB;
    if (out) {
        hipLaunchKernelGGL((search_mfma_kernel<KS, MT, GS, true, Q8, POL, HV, false>), grid, block, 0, s, p);
        return;
    }
    if constexpr (!Q8 && POL == 0 && HV == 1 && KS <= 4 && MfmaShape<KS, MT, GS>::NB >= kAheadNodes) {
        if constexpr (MT <= kSampledTiles) {
            if (plan.ahead && p.sample_wgs > 0) {
                hipLaunchKernelGGL((search_mfma_kernel<KS, MT, GS, false, false, 0, 1, true, kAheadNodes, true>), grid, block, 0, s, p);
                return;
            }
        }
        if constexpr (KS * MT >= 8) {  // (tiles of 128 KiB)
            if (plan.ahead == kAheadNodes / 2) {
                hipLaunchKernelGGL((search_mfma_kernel<KS, MT, GS, false, false, 0, 1, true, kAheadNodes / 2>), grid, block, 0, s, p);
                return;
            }
        }
        if (plan.ahead) {
            hipLaunchKernelGGL((search_mfma_kernel<KS, MT, GS, false, false, 0, 1, true, kAheadNodes>), grid, block, 0, s, p);
            return;
        }
    }
    if constexpr (!Q8) {
        if (one) {
            hipLaunchKernelGGL((search_mfma_kernel<KS, MT, GS, false, Q8, POL, HV, true>), grid, block, 0, s, p);
            return;
        }
    }
    hipLaunchKernelGGL((search_mfma_kernel<KS, MT, GS, false, Q8, POL, HV, false>), grid, block, 0, s, p);
}

template <int KS, int MT, bool Q8, int POL, int HV = 1>
void launch_mfma_gs(const SearchPlan& plan, const SearchParams& p, dim3 grid, hipStream_t s) {
    if (plan.gmax <= 4) launch_mfma_one<KS, MT, 4, Q8, POL, HV>(plan, p, grid, s);
    else if (plan.gmax <= 8) launch_mfma_one<KS, MT, 8, Q8, POL, HV>(plan, p, grid, s);
    else launch_mfma_one<KS, MT, 16, Q8, POL, HV>(plan, p, grid, s);
}

template <int KS, bool Q8, int POL>
void launch_mfma_mt(const SearchPlan& plan, const SearchParams& p, dim3 grid, hipStream_t s) {
    const int mt = p.bf / 16;
    if (mt <= 1)
        launch_mfma_gs<KS, 1, Q8, POL>(plan, p, grid, s);
    else if (mt == 2)
        launch_mfma_gs<KS, 2, Q8, POL>(plan, p, grid, s);
    else if (KS == 8 && plan.gmax > 4)
        // 256 columns x 64 keys a node x 8 or 16 heads: a node's four tiles do not fit the
        // registers next to the accumulators; it is scanned as two halves of two tiles
        launch_mfma_gs<KS, (KS == 8 ? 2 : 4), Q8, POL, (KS == 8 ? 2 : 1)>(plan, p, grid, s);
    else
        launch_mfma_gs<KS, 4, Q8, POL>(plan, p, grid, s);
}

// one translation unit per key width and per kind of scan (bf16 tiles and 8-bit shadow, under each
// cache policy) keeps the build parallel
void launch_mfma_d64(const SearchPlan& plan, const SearchParams& p, dim3 grid, hipStream_t s);
void launch_mfma_d128(const SearchPlan& plan, const SearchParams& p, dim3 grid, hipStream_t s);
void launch_mfma_d256(const SearchPlan& plan, const SearchParams& p, dim3 grid, hipStream_t s);
void launch_mfma_nt1_d64(const SearchPlan& plan, const SearchParams& p, dim3 grid, hipStream_t s);
void launch_mfma_nt2_d64(const SearchPlan& plan, const SearchParams& p, dim3 grid, hipStream_t s);
void launch_mfma_nt1_d128(const SearchPlan& plan, const SearchParams& p, dim3 grid, hipStream_t s);
void launch_mfma_nt2_d128(const SearchPlan& plan, const SearchParams& p, dim3 grid, hipStream_t s);
void launch_mfma_nt1_d256(const SearchPlan& plan, const SearchParams& p, dim3 grid, hipStream_t s);
void launch_mfma_nt2_d256(const SearchPlan& plan, const SearchParams& p, dim3 grid, hipStream_t s);
void launch_mfma_q8_d64(const SearchPlan& plan, const SearchParams& p, dim3 grid, hipStream_t s);
void launch_mfma_q8_d128(const SearchPlan& plan, const SearchParams& p, dim3 grid, hipStream_t s);
void launch_mfma_q8_nt1_d64(const SearchPlan& plan, const SearchParams& p, dim3 grid, hipStream_t s);
void launch_mfma_q8_nt1_d128(const SearchPlan& plan, const SearchParams& p, dim3 grid, hipStream_t s);

}  // namespace hira
