// Append-on-decode index update: m new keys/values per tree go into the existing tree.
//
// Replaces CUDAIndexer.update and its Triton kernels (indexer/cuda.py:544-701, 707-1231;
// kernels/triton_update_kernels.py:6-123, 126-235, 238-326) with one launch: one workgroup
// per tree walks that tree's new keys in insertion order, so slots, counts and radii need
// no global atomics and the result is reproducible.  For every key:
//   1. nearest level-1 node that still has a free child slot (exact fp32 L2 distance over
//      the nodes in use; full nodes are skipped before their centre is read) -- the
//      reference's nearest_l2 + valid-mask step;
//   2. the key takes the node's next slot (the reference's atomic slot reservation), the
//      node's radius grows to cover it (its atomic-max step) and every ancestor's radius is
//      re-inflated: R_a = max(R_a, ||c_child - c_a|| + r_child) (indexer/cuda.py:1200-1231);
//      centres never move, radii only grow, exactly as in the reference;
//   3. if no node has room the key opens a new level-1 node whose centre is the key itself
//      (the reference draws its new parents from the orphans, indexer/cuda.py:612-635); the
//      new node is attached the same way one level up: nearest level-2 node with a free
//      child slot, else a new level-2 node, ... up to the root level, which simply grows.
// Child counts stay authoritative (the reference over-counts on overflow and repairs the
// counters with an O(N D) rescan after every update, indexer/cuda.py:1233-1298).
//
// state (T, HIRA_MAX_LEVELS + 2) int32: [l] = slots of level l in use (l >= 1; the host keeps
// the maximum over the trees as size[l]), [HIRA_MAX_LEVELS] = keys inserted so far,
// [HIRA_MAX_LEVELS + 1] = error flag (1: a level ran out of capacity; the key was dropped).
// [0] (trees of two or more levels): every level-1 node with a lower index is full -- a lower
// bound that the search for a node with room starts from and raises as it learns more (0 is
// always valid; whoever lowers a count of a level-1 node from outside must lower it too).
#include <algorithm>
#include <chrono>

#include "rows.h"
#include "threshold_kernel.h"

namespace hira {

constexpr int kUpdThreads = 256;  // of a workgroup that takes key after key
constexpr int kWinThreads = 512;  // of one that takes a window (the functions of both: NT)

struct UpdateParams {
    void* keys;
    void* values;
    int32_t* perm;
    void* centers[HIRA_MAX_LEVELS];
    float* radii[HIRA_MAX_LEVELS];
    int32_t* counts[HIRA_MAX_LEVELS];
    int32_t cap[HIRA_MAX_LEVELS];
    int32_t num_levels, bf, dim, vdim, layout;  // layout: of the centers
    int32_t key_layout;
    int8_t* keys8;        // HIRA_TILE16_Q8: the 8-bit shadow of the keys
    const float* kscale;  //   its step per tree and channel
    float* keps;          //   largest error, in steps, among the keys of each level-1 node
    const void* new_keys;    // (T, m, D)
    const void* new_values;  // (T, m, Dv) or NULL
    int32_t m;
    int32_t* state;
    int32_t stage_values;  // windows: the values' rows have room in LDS too
};

// The kernels' arguments lie in six 64-byte lines of memory: all of them asked for at once (touch_kernel_arguments
// of search.h, for its kernels' nine): a window of 64 keys 21 -> 19.7 us, a single key 7.6 -> 7.2.
__device__ __forceinline__ void touch_update_arguments() {
    static_assert(sizeof(UpdateParams) > 5 * 64 + 4 && sizeof(UpdateParams) <= 6 * 64, "one load per 64-byte line of the arguments");
    auto ka = __builtin_amdgcn_kernarg_segment_ptr();
    uint32_t d0, d1, d2, d3, d4, d5;
    asm volatile(
        "s_load_dword %0, %6, 0x0\n\t"
        "s_load_dword %1, %6, 0x40\n\t"
        "s_load_dword %2, %6, 0x80\n\t"
        "s_load_dword %3, %6, 0xc0\n\t"
        "s_load_dword %4, %6, 0x100\n\t"
        "s_load_dword %5, %6, 0x140\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&s"(d0), "=&s"(d1), "=&s"(d2), "=&s"(d3), "=&s"(d4), "=&s"(d5)
        : "s"(ka)
        : "memory");
}

// Rows of a key sample that new keys of the same call take the place of, in workgroups behind the trees':
// dst[t][slot[i]] = new_keys[t][from[i]].  They share nothing with the append, and a launch of their own costs
// the host and the GPU more than they do (a token that goes into the index at once, 2 trees of 64 bf16 columns:
// 6.9 us for the append and, behind a gap of 1.2, 2.0 for the sample; together 7.0).  The pairs travel with the
// arguments.
constexpr int kSamplePairs = 32;
struct SampleRows {
    uint4* dst;
    int32_t trees, chunks, rows_per_tree, n;  // trees: the workgroups that append
    int32_t slot[kSamplePairs], from[kSamplePairs];
};

template <int NT>
__device__ __forceinline__ void replace_sample(const UpdateParams& p, const SampleRows& r) {
    const int i = ((int)blockIdx.x - r.trees) * NT + (int)threadIdx.x;
    if (i >= r.trees * r.n * r.chunks) return;
    const int row = i / r.chunks, c = i - row * r.chunks;  // row: tree * n + pair
    const int t = row / r.n, k = row - t * r.n;
    r.dst[((size_t)t * r.rows_per_tree + r.slot[k]) * r.chunks + c] =
        reinterpret_cast<const uint4*>(p.new_keys)[((size_t)t * p.m + r.from[k]) * r.chunks + c];
}

// a bound must survive the fp32 rounding of the sums that produced it
__device__ __forceinline__ float pad_up(float r) { return r > 0.0f ? r * (1.0f + 4.0f * 1.1920929e-7f) + 1e-30f : r; }

// Nearest node of level l (among nodes first .. used - 1; the ones before `first` are known to
// be full) with a free child slot; -1 if none.  Waves take stretches of 64 nodes in turn; a full
// node costs one count read.  Ties go to the lowest id.  *not_full (if given) receives the lowest
// index from `first` on whose node is not full (`used` if there is none).
constexpr int kCountsInFlight = 16;  // reads of child counts a lane has in flight
template <typename T, int NT>
__device__ __forceinline__ int nearest_with_room(const UpdateParams& p, int tree, int l, int first, int used,
                                 const float* x, float* red_f, int* red_i, int* not_full,
                                 int* count_of = nullptr, float* dist2_of = nullptr,
                                 float* radius_of = nullptr) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int D = p.dim;
    const size_t base = (size_t)tree * p.cap[l];
    const int32_t* cnt = p.counts[l] + base;
    float best = INFINITY;
    int arg = -1, argc = 0;  // the best node so far and its child count
    float argr = 0.0f;       // (its radius, asked for with the centre)
    int low = used;  // lowest index of a node that is not full, among those I have seen
    for (int nb = (first & ~63) + wave * 64; nb < used; nb += kCountsInFlight * NT) {
        // the reads of the child counts in flight together (a wave's nodes still come in
        // increasing order): one trip to memory for 16 NT nodes
        int c4[kCountsInFlight];
#pragma unroll
        for (int u = 0; u < kCountsInFlight; ++u) {
            const int n = nb + u * NT + lane;
            c4[u] = n < used ? cnt[n] : p.bf;
        }
#pragma unroll
        for (int u = 0; u < kCountsInFlight; ++u) {
            if (nb + u * NT >= used) break;  // uniform
            if (c4[u] < p.bf) low = min(low, nb + u * NT + lane);
            // a node in use with a free slot; count 0 marks a pad slot, which is not a node yet
            unsigned long long bal = __ballot(c4[u] > 0 && c4[u] < p.bf);
            while (bal != 0ull) {  // uniform in the wave
                const int src = __ffsll((long long)bal) - 1;
                const int node = nb + u * NT + src;
                const int node_c = __shfl(c4[u], src, 64);
                bal &= bal - 1ull;
                float ss = 0.0f;
                const float rad = radius_of != nullptr ? p.radii[l][base + node] : 0.0f;
                for (int j = lane; j < D; j += 64) {
                    const float df = x[j] - load_elem<T>(p.centers[l], base * D + elem_index(p.layout, D, (size_t)node, j));
                    ss += df * df;
                }
                ss = wave_sum(ss);
                if (ss < best) {
                    best = ss;
                    arg = node;
                    argc = node_c;
                    argr = rad;
                }
            }
        }
    }
    __syncthreads();
    if (not_full != nullptr) {  // uniform
        low = wave_min(low);
        if (lane == 0) red_i[wave] = low;
        __syncthreads();
        if (threadIdx.x == 0) {
#pragma unroll
            for (int w = 1; w < NT / 64; ++w) low = min(low, red_i[w]);
            *not_full = max(low, first);
        }
        __syncthreads();
    }
    if (lane == 0) {
        red_f[wave] = best;
        red_i[wave] = arg;
    }
    __syncthreads();
    float b = red_f[0];
    int a = red_i[0], aw_of = 0;
#pragma unroll
    for (int w = 1; w < NT / 64; ++w) {
        const float bw = red_f[w];
        const int aw = red_i[w];
        if (aw >= 0 && (a < 0 || bw < b || (bw == b && aw < a))) {
            b = bw;
            a = aw;
            aw_of = w;
        }
    }
    __syncthreads();
    if (count_of != nullptr) {  // uniform: the child count of the chosen node, as the scan read it
        if (lane == 0) red_i[wave] = argc;
        __syncthreads();
        *count_of = red_i[aw_of];
        __syncthreads();
    }
    if (dist2_of != nullptr) *dist2_of = b;
    if (radius_of != nullptr) {  // uniform
        if (lane == 0) red_f[wave] = argr;
        __syncthreads();
        *radius_of = red_f[aw_of];
        __syncthreads();
    }
    return a;
}

// One key of the window, placed the general way: key i of the tree's new keys.
//   sm: 2 D floats (the key, the centre of a node being attached upwards).
template <typename T, int NT>
__device__ __forceinline__ void update_one_key(const UpdateParams& p, const int tree, const int i, float* sm, float* red_f,
                               int* red_i, float* s_dist, float* s_rad) {
    float* x = sm;              // (D) the new key, fp32
    float* cbuf = sm + p.dim;   // (D) centre of the node being attached upwards
    const int t = threadIdx.x;
    const int D = p.dim, Dv = p.vdim, L = p.num_levels, bf = p.bf;
    int32_t* st = p.state + (size_t)tree * (HIRA_MAX_LEVELS + 2);
    const size_t base0 = (size_t)tree * p.cap[0];

    const size_t src = ((size_t)tree * p.m + i) * D;
    for (int j = t; j < D; j += NT) x[j] = load_elem<T>(p.new_keys, src + j);
    __syncthreads();
    const int position = st[HIRA_MAX_LEVELS];

    long long slot = -1;  // key slot
    int node1 = -1;       // level-1 node that took the key (L >= 2)
    int count1 = 0;       // keys it held before
    if (L == 1) {
        slot = position < p.cap[0] ? position : -1;
    } else {
        node1 = nearest_with_room<T, NT>(p, tree, 1, min(max(st[0], 0), st[1]), st[1], x, red_f, red_i, &st[0],
                                         &count1);
        if (node1 < 0) {
            // ---- open a new level-1 node; attach it upwards -----------------------
            // child_c = centre of the node being attached (the key itself at level 1)
            for (int j = t; j < D; j += NT) cbuf[j] = x[j];
            __syncthreads();
            int lvl = 1;          // level of the node that needs a parent
            int parent = -1;      // node of level lvl+1 that takes it
            int opened_top = 0;   // levels 1..opened_top get a brand-new node
            // find the lowest level that has a parent with room
            while (true) {
                if (lvl == L - 1) {  // the root level grows
                    parent = -1;
                    break;
                }
                parent = nearest_with_room<T, NT>(p, tree, lvl + 1, 0, st[lvl + 1], cbuf, red_f, red_i, nullptr);
                if (parent >= 0) break;
                ++lvl;
            }
            opened_top = lvl;
            // index of the new node at level opened_top
            long long idx;
            if (parent >= 0) {
                idx = (long long)parent * bf + p.counts[opened_top + 1][(size_t)tree * p.cap[opened_top + 1] + parent];
            } else {
                idx = st[opened_top];
            }
            // every new node below it is the first child of the new node above
            bool fits = true;
            long long id = idx;
            for (int l = opened_top; l >= 1; --l) {
                if (id >= p.cap[l]) fits = false;
                id *= bf;
            }
            if (id >= p.cap[0]) fits = false;
            __syncthreads();  // everybody has read the counters the writes below change
            if (!fits) {
                if (t == 0) st[HIRA_MAX_LEVELS + 1] = 1;
                __syncthreads();
                return;  // uniform: the key is dropped, the host sees the flag
            }
            id = idx;
            for (int l = opened_top; l >= 1; --l) {
                const size_t bl = (size_t)tree * p.cap[l];
                for (int j = t; j < D; j += NT)
                    store_elem<T>(p.centers[l], bl * D + elem_index(p.layout, D, (size_t)id, j), x[j]);
                if (t == 0) {
                    p.radii[l][bl + id] = 0.0f;
                    p.counts[l][bl + id] = (l == 1) ? 0 : 1;  // level 1 gets its key below
                    if (id + 1 > st[l]) st[l] = (int)(id + 1);
                }
                id *= bf;
            }
            if (t == 0 && parent >= 0)
                p.counts[opened_top + 1][(size_t)tree * p.cap[opened_top + 1] + parent] += 1;
            __syncthreads();
            node1 = (int)(id / bf);  // the new level-1 node (id is now its first key slot)
            count1 = 0;
        }
        // the key takes the next slot of node1
        // (a node found by the scan: the count the scan read; a node just opened: none)
        const size_t b1 = (size_t)tree * p.cap[1];
        const int c = count1;
        slot = (long long)node1 * bf + c;
        __syncthreads();
        if (t == 0) p.counts[1][b1 + node1] = c + 1;
    }
    if (slot < 0 || slot >= p.cap[0]) {
        if (t == 0) st[HIRA_MAX_LEVELS + 1] = 1;
        __syncthreads();
        return;
    }
    // ---- write key, value, perm -------------------------------------------------------
    {
        const T* dummy = nullptr;
        (void)dummy;
        for (int j = t; j < D; j += NT)
            store_elem<T>(p.keys, base0 * D + elem_index(p.key_layout, D, (size_t)slot, j), x[j]);
        if (p.keys8 != nullptr) {
            // the key's 8-bit shadow with the tree's steps; a component beyond +-127 steps
            // clips, and the node's error bound then covers it
            float worst = 0.0f;
            for (int j = t; j < D; j += NT) {
                const float u = x[j] / p.kscale[(size_t)tree * D + j];
                const float r = fminf(fmaxf(rintf(u), -127.0f), 127.0f);
                worst = fmaxf(worst, fabsf(u - r));
                p.keys8[base0 * D + shadow_index(D, (size_t)slot, j)] = (int8_t)(int)r;
            }
            worst = wave_max(worst);
            if ((t & 63) == 0) red_f[t >> 6] = worst;
            __syncthreads();
            if (t == 0) {
                float* e = p.keps + (size_t)tree * p.cap[1] + node1;
                float w = red_f[0];
#pragma unroll
                for (int i = 1; i < NT / 64; ++i) w = fmaxf(w, red_f[i]);
                // a node that just opened holds no other key: its bound starts here
                const bool fresh = count1 == 0;
                *e = fresh ? w : fmaxf(*e, w);
            }
            __syncthreads();
        }
        if (p.new_values && p.values) {
            const size_t vs = ((size_t)tree * p.m + i) * Dv;
            for (int j = t; j < Dv; j += NT)
                store_elem<T>(p.values, (base0 + slot) * Dv + j, load_elem<T>(p.new_values, vs + j));
        }
        if (t == 0) {
            p.perm[base0 + slot] = position;
            st[HIRA_MAX_LEVELS] = position + 1;
            if (L == 1 && slot + 1 > st[0]) st[0] = (int)(slot + 1);
        }
    }
    // ---- radii: the leaf parent covers the key, every ancestor covers its child.  The
    // distances of all levels are taken at once (a wave per level), then one thread walks
    // the chain R_l = max(R_l, d_l + R_{l-1}). ---------------------------------------------
    if (L >= 2) {
        const int lane = t & 63;
        for (int l = 1 + (t >> 6); l < L; l += NT / 64) {  // uniform in the wave
            size_t child = (size_t)node1;  // node of level l - 1 on the key's path (l >= 2)
            for (int i = 2; i < l; ++i) child /= (size_t)bf;
            const size_t node = l == 1 ? (size_t)node1 : child / (size_t)bf;
            const size_t bl = (size_t)tree * p.cap[l], bc = (size_t)tree * p.cap[l - 1];
            const float rad_now = p.radii[l][bl + node];  // (asked for with the centres)
            float ss = 0.0f;
            for (int j = lane; j < D; j += 64) {
                const float a =
                    l == 1 ? x[j]
                           : load_elem<T>(p.centers[l - 1], bc * D + elem_index(p.layout, D, child, j));
                const float b = load_elem<T>(p.centers[l], bl * D + elem_index(p.layout, D, node, j));
                ss += (a - b) * (a - b);
            }
            ss = wave_sum(ss);
            if (lane == 0) {
                s_dist[l] = sqrtf(ss);
                s_rad[l] = rad_now;
            }
        }
        __syncthreads();
        if (t == 0) {
            size_t node = (size_t)node1;
            float r_child = 0.0f;
            for (int l = 1; l < L; ++l) {
                const float rn = fmaxf(s_rad[l], pad_up(s_dist[l] + r_child));
                if (rn != s_rad[l]) p.radii[l][(size_t)tree * p.cap[l] + node] = rn;
                r_child = rn;
                node /= (size_t)bf;
            }
        }
    }
    __syncthreads();
}

template <typename T>
__global__ __launch_bounds__(kUpdThreads) void k_update(const UpdateParams p, const SampleRows sample) {
    extern __shared__ float sm[];
    __shared__ float red_f[4];
    __shared__ int red_i[4];
    __shared__ float s_dist[HIRA_MAX_LEVELS], s_rad[HIRA_MAX_LEVELS];
    touch_update_arguments();
    if ((int)blockIdx.x >= sample.trees) {  // uniform in the workgroup
        replace_sample<kUpdThreads>(p, sample);
        return;
    }
    for (int i = 0; i < p.m; ++i)
        update_one_key<T, kUpdThreads>(p, (int)blockIdx.x, i, sm, red_f, red_i, s_dist, s_rad);
}

// An append of a few keys per tree and the thresholds of a decode step in one launch: the first
// `trees` workgroups append (their first kUpdThreads threads; the others leave at once, and a
// barrier counts only the waves still there), the ones behind them take a head each.  The two
// halves share nothing: the sample is not touched by the append.
template <typename T, int E>
__global__ __launch_bounds__(kTauThreads) void k_update_threshold(
    const UpdateParams p, const int trees, const T* __restrict__ samples, const int S,
    const T* __restrict__ q, const int32_t* __restrict__ tree_q_off,
    const int32_t* __restrict__ tree_q_heads, const int group_size, const int method, const int k,
    float* __restrict__ tau) {
    extern __shared__ float sm[];
    __shared__ float red_f[4];
    __shared__ int red_i[4];
    __shared__ float s_dist[HIRA_MAX_LEVELS], s_rad[HIRA_MAX_LEVELS];
    if ((int)blockIdx.x < trees) {  // uniform in the workgroup
        if (threadIdx.x >= kUpdThreads) return;
        for (int i = 0; i < p.m; ++i)
            update_one_key<T, kUpdThreads>(p, (int)blockIdx.x, i, sm, red_f, red_i, s_dist, s_rad);
        return;
    }
    threshold_block<T, E>(samples, S, p.dim, q, tree_q_off, tree_q_heads, group_size, trees, method, k,
                          tau, (int)blockIdx.x - trees);
}

// ---- windows of several keys ---------------------------------------------------------------
// Placing a key the general way costs a handful of dependent trips to memory (child counts,
// the centres of the nodes with room, the ancestors' centres and radii): 4-5 us a key, one key
// after the other.  But the nodes with room are few -- the tail nodes opened by earlier appends,
// what a rebuilt subtree left free -- and between two keys of a window only the window itself
// changes them.  So a workgroup that has a window to place lists them ONCE in LDS (ids, child
// counts, centres, radii, and for every ancestor on their paths its radius and the distance
// between consecutive centres, which never changes) and takes the window 64 keys at a time:
//   distances  of all 64 keys to all candidates, by all waves, into a table in LDS;
//   choice     wave 0, a candidate a lane, key after key: the smallest distance among the lanes
//              whose node has room (ties: the lowest id, as the general way) -- one row of the
//              table, a minimum over the wave, a count, which is all that has to happen one key after
//              the other;
//   rows       of the 64 keys to their slots, 16 bytes a thread.
// What bounds it is latency in one workgroup a tree (its waves wait 69 % of their cycles).  A launch, 8 trees
// of 128 bf16 columns: with 45 nodes to list, 39 us for 4 keys, 42 for 16, 49 for 32, 57 for 64 (48, 52, 60, 87); with one
// node, full after 32 keys, and then another: 12 us for 4, 14 for 32, 20 for 64, 34 for 128, 66 for 255 (16, 21, 33, 59
// and 119 when a key that opens a node looked for its parent in memory, the distances to the new node were taken of
// keys that it has no room for, the 8-bit shadow was written a byte at a time, and the general way was a call, around which
// values lay in scratch memory: 4 us of any launch).  256 threads instead of 512: 13, 15, 21, 37, 76.
// Radii wait until the list is given up: R = max over the keys of what each asks for, and that
// grows with the distance, so the largest distance a candidate saw gives the radius that key by
// key would have reached, to the last bit, and so up the levels.  A key that finds all candidates
// full opens a node, which becomes the list.  A key that has no finite distance to any candidate opens
// one too, but the others still have room: it ends its chunk, and the nodes with room are listed anew.
// A tree with more nodes with room than the list holds goes the general way altogether.  Same
// placement, slots and radii as key by key (the replaced kernels:
// kernels/triton_update_kernels.py:85-123 nearest centre for a whole window at once, :126-235 slots,
// :238-326 radii).
constexpr int kCandMax = 48;
constexpr int kWinKeys = 64;  // keys of a window taken together
// COLS, below: columns of a row a lane holds, at most.  Rows of fp32, and of bf16 up to 256, take four;
// wider ones five (320 columns): 8 trees x 64 keys of 288 columns, which went key by key, 358 -> 61 us.
// Five for all rows would cost those of 128 columns 0.8 us a launch.
constexpr int kWinColsMax = 5;
constexpr size_t kWinLds = 144 * 1024;  // dynamic LDS of a workgroup, at most (256 fp32 columns: 142 KiB; 320
                                        // bf16 columns: 135)
// Level-2 nodes with room, listed like those of level 1, so that a key that opens a node finds its parent without a
// trip to memory.  More than the list holds, or more nodes to look through than one trip reads: no list.
template <typename T>
constexpr int kParents = 64 / (int)sizeof(T);
constexpr int kParentsMax = 32, kParentCounts = 2;  // (counts a thread reads)

struct WindowLds {
    int n;                                  // candidates listed (may exceed kCandMax: then unusable)
    int low_empty;                          // lowest level-1 slot from `first` on that is no node yet
    int id[kCandMax];                       // level-1 node
    int cnt[kCandMax];                      // its child count (bf: full by now)
    int cnt0[kCandMax];                     // its child count as memory has it
    float rad[kCandMax];                    // its radius, as memory has it
    float far[kCandMax];                    // largest squared distance of a key it took
    int anc_id[HIRA_MAX_LEVELS][kCandMax];      // [l][c]: c's ancestor at level l
    int anc_rep[HIRA_MAX_LEVELS][kCandMax];     // [l][c]: the first candidate with the same ancestor at level l
    float anc_rad[HIRA_MAX_LEVELS][kCandMax];   // [l][rep]: that ancestor's radius
    float anc_step[HIRA_MAX_LEVELS][kCandMax];  // [l][c]: distance between c's ancestors at levels l-1 and l
    int n2;                                 // level-2 nodes listed (more than kParents: no list)
    int id2[kParentsMax], cnt2[kParentsMax];
    float d2[kParentsMax];                  // squared distances of a key to them
};

// level-l ancestor of level-1 node `node1` (l >= 1)
__device__ __forceinline__ size_t ancestor_of(size_t node1, int l, int bf) {
    for (int i = 1; i < l; ++i) node1 /= (size_t)bf;
    return node1;
}

// Reads the tree's level-1 nodes with room into LDS, and those of level 2.  cen: (kCandMax, D) floats, par:
// (kParents, D).  Returns false (uniform) when there are more of level 1 than the list holds.
template <typename T, int NT>
__device__ __forceinline__ bool window_candidates(const UpdateParams& p, const int tree, const int st0, const int st1,
                                                  const int st2, WindowLds& w, float* cen, T* par) {
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int D = p.dim, L = p.num_levels, bf = p.bf;
    const int used = st1, first = min(max(st0, 0), used);
    const int used2 = L > 2 ? st2 : 0;
    const bool look2 = used2 <= kParentCounts * NT;
    const size_t b1 = (size_t)tree * p.cap[1];
    if (t == 0) {
        w.n = 0;
        w.low_empty = used;
        w.n2 = look2 ? 0 : kParents<T> + 1;
    }
    int c2[kParentCounts];  // (on their way beside level 1's)
#pragma unroll
    for (int u = 0; u < kParentCounts; ++u) {
        const int n = u * NT + t;
        c2[u] = look2 && n < used2 ? p.counts[2][(size_t)tree * p.cap[2] + n] : bf;
    }
    __syncthreads();
    for (int nb = first & ~63; nb < used; nb += NT) {  // uniform
        const int n = nb + t;
        const int c = (n >= first && n < used) ? p.counts[1][b1 + n] : bf;
        if (c <= 0) atomicMin(&w.low_empty, n);
        // a node in use with a free slot; count 0 marks a pad slot, which is not a node yet
        const bool room = c > 0 && c < bf;
        const unsigned long long bal = __ballot(room);
        int at = 0;
        if (lane == 0 && bal != 0ull) at = atomicAdd(&w.n, __popcll(bal));
        at = __shfl(at, 0, 64) + __popcll(bal & ((1ull << lane) - 1ull));
        if (room && at < kCandMax) {
            w.id[at] = n;
            w.cnt[at] = w.cnt0[at] = c;
            w.far[at] = -1.0f;
        }
    }
#pragma unroll
    for (int u = 0; u < kParentCounts; ++u)
        if (c2[u] > 0 && c2[u] < bf) {
            const int at = atomicAdd(&w.n2, 1);
            if (at < kParents<T>) {
                w.id2[at] = u * NT + t;
                w.cnt2[at] = c2[u];
            }
        }
    __syncthreads();
    const int nc = w.n, n2 = w.n2 <= kParents<T> ? w.n2 : 0;
    if (nc > kCandMax) return false;
    for (int e = t; e < n2 * D; e += NT)
        store_elem<T>(par, e, load_elem<T>(p.centers[2], (size_t)tree * p.cap[2] * D + elem_index(p.layout, D, (size_t)w.id2[e / D], e % D)));
    // (the order in which the waves listed their nodes does not matter: ties between candidates
    // are decided by the node's id)
    for (int c = wave; c < nc; c += NT / 64) {  // uniform in the wave
        const size_t node = (size_t)w.id[c];
        for (int j = lane; j < D; j += 64)
            cen[(size_t)c * D + j] = load_elem<T>(p.centers[1], b1 * D + elem_index(p.layout, D, node, j));
        if (lane == 0) w.rad[c] = p.radii[1][b1 + node];
        for (int l = 2; l < L; ++l) {
            const size_t child = ancestor_of(node, l - 1, bf), anc = child / (size_t)bf;
            const size_t bl = (size_t)tree * p.cap[l], bc = (size_t)tree * p.cap[l - 1];
            float ss = 0.0f;
            for (int j = lane; j < D; j += 64) {
                const float a = load_elem<T>(p.centers[l - 1], bc * D + elem_index(p.layout, D, child, j));
                const float b = load_elem<T>(p.centers[l], bl * D + elem_index(p.layout, D, anc, j));
                ss += (a - b) * (a - b);
            }
            ss = wave_sum(ss);
            if (lane == 0) {
                w.anc_id[l][c] = (int)anc;
                w.anc_step[l][c] = sqrtf(ss);
                w.anc_rad[l][c] = p.radii[l][bl + anc];  // (read where c is its ancestor's first candidate)
            }
        }
    }
    __syncthreads();
    for (int k = t; k < nc * HIRA_MAX_LEVELS; k += NT) {
        const int c = k % nc, l = k / nc;
        if (l < 2 || l >= L) continue;
        const int anc = w.anc_id[l][c];
        int rep = c;
        for (int o = 0; o < c; ++o)
            if (w.anc_id[l][o] == anc) {
                rep = o;
                break;
            }
        w.anc_rep[l][c] = rep;
    }
    __syncthreads();
    return true;
}

// the value that lane ^ BIT holds, by moves that need no trip through LDS (16, 32: the sum with it)
template <int BIT>
__device__ __forceinline__ float win_partner(float v) {
    if constexpr (BIT == 1) return dpp_move<0xB1>(v);                   // quad [1,0,3,2]
    else if constexpr (BIT == 2) return dpp_move<0x4E>(v);              // quad [2,3,0,1]
    else if constexpr (BIT == 4) return dpp_move<0x1B>(dpp_move<0x141>(v));  // halves of 8 mirrored, quads mirrored
    else return dpp_move<0x128>(v);                                     // 8: row rotated by 8
}
template <int BIT>
__device__ __forceinline__ float win_sum_across(float v) {
    const auto r = BIT == 32 ? __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false)
                             : __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Squared distances of keys [k0, k1) of the chunk (rows in LDS) to all candidates:
// table[k * kCandMax + c].  A wave takes eight keys at a time, its lanes a column (of every 64)
// each, and goes through the candidates: the eight sums over the lanes halve in number with every
// one of the first three steps (lanes with the bit set go on with the other half).  The additions are those of a butterfly of lane ^ 1, ^ 2,
// ..., ^ 32, in that order: the general way's, to the last bit.
template <typename T, int COLS, int NT>
__device__ __forceinline__ void window_distances(const int D, const WindowLds& w, const float* cen, const T* rows,
                                 const int k0, const int k1, float* table) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int nc = w.n;
    if (nc == 0) return;
    const bool b0 = lane & 1, b1 = lane & 2, b2 = lane & 4;
    const int mine = (b0 ? 4 : 0) + (b1 ? 2 : 0) + (b2 ? 1 : 0);  // the key (of eight) I end up with
    for (int k = k0 + wave * 8; k < k1; k += NT / 64 * 8) {  // uniform in the wave
        float x[8][COLS];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const size_t src = (size_t)min(k + u, k1 - 1) * D;
#pragma unroll
            for (int i = 0; i < COLS; ++i)
                if (i * 64 < D) {  // (uniform)
                    const float xi = load_elem<T>(rows, src + min(i * 64 + lane, D - 1));
                    x[u][i] = i * 64 + lane < D ? xi : 0.0f;
                }
        }
        for (int c = 0; c < nc; ++c) {  // uniform
            float v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = 0.0f;
#pragma unroll
            for (int i = 0; i < COLS; ++i)
                if (i * 64 < D) {  // uniform
                    const float ci = cen[(size_t)c * D + min(i * 64 + lane, D - 1)];
                    const float cj = i * 64 + lane < D ? ci : 0.0f;
#pragma unroll
                    for (int u = 0; u < 8; ++u) {
                        const float df = x[u][i] - cj;
                        v[u] += df * df;
                    }
                }
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = (b0 ? v[u + 4] : v[u]) + win_partner<1>(b0 ? v[u] : v[u + 4]);
#pragma unroll
            for (int u = 0; u < 2; ++u) v[u] = (b1 ? v[u + 2] : v[u]) + win_partner<2>(b1 ? v[u] : v[u + 2]);
            float s = (b2 ? v[1] : v[0]) + win_partner<4>(b2 ? v[0] : v[1]);
            s += win_partner<8>(s);
            s = win_sum_across<16>(s);
            s = win_sum_across<32>(s);
            if (lane < 8 && k + mine < k1) table[(k + mine) * kCandMax + c] = s;
        }
    }
}

__device__ __forceinline__ float win_min(float v) {  // over the wave, the same in every lane
    v = fminf(v, win_partner<1>(v));
    v = fminf(v, win_partner<2>(v));
    v = fminf(v, dpp_move<0x141>(v));  // (any lane of the other four will do)
    v = fminf(v, win_partner<8>(v));
    auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fminf(__uint_as_float(r[0]), __uint_as_float(r[1]));
    r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fminf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// The list is given up: child counts and radii of the candidates that took keys, and their
// ancestors' radii, go to memory.  By wave 0, a candidate a lane.
__device__ __forceinline__ void window_flush(const UpdateParams& p, const int tree, WindowLds& w) {
    const int c = threadIdx.x, L = p.num_levels;
    if (c >= 64) return;
    const bool took = c < w.n && w.cnt[c] != w.cnt0[c];
    float r = 0.0f;
    if (took) {
        const size_t at = (size_t)tree * p.cap[1] + w.id[c];
        p.counts[1][at] = w.cnt[c];
        r = fmaxf(w.rad[c], pad_up(sqrtf(w.far[c])));
        if (r != w.rad[c]) p.radii[1][at] = r;
    }
    for (int l = 2; l < L; ++l) {
        int rep = 0;
        float have = 0.0f;
        if (took) {
            rep = w.anc_rep[l][c];
            have = w.anc_rad[l][rep];
        }
        __builtin_amdgcn_wave_barrier();
        // (radii are -inf or not negative: their bits order as signed integers)
        if (took) atomicMax(reinterpret_cast<int*>(&w.anc_rad[l][rep]), __float_as_int(pad_up(w.anc_step[l][c] + r)));
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
        if (took) {
            r = w.anc_rad[l][rep];
            if (r != have) p.radii[l][(size_t)tree * p.cap[l] + w.anc_id[l][c]] = r;  // (the same from all of them)
        }
    }
}

// Key i of the tree's window opens a level-1 node centred on itself, no node having room: what
// update_one_key does in that case, in the trips to memory that it cannot do without (the child
// counts of the level above, the centres and radii of the nodes there with room, the path above the
// chosen one), the key and the level sizes (s_used) being in LDS.  Returns the node (-1: dropped for
// lack of capacity); x (LDS) then holds the key in fp32, s_dist[l] the distance between the node's
// ancestors at levels l - 1 and l, s_rad[l] the radius of the latter.
template <typename T, int NT>
__device__ __forceinline__ int open_node(const UpdateParams& p, const int tree, const int i,
                                                 const int position, int* s_used, const T* key, float* x,
                                                 float* red_f, int* red_i, float* s_dist, float* s_rad) {
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int D = p.dim, Dv = p.vdim, L = p.num_levels, bf = p.bf;
    int32_t* st = p.state + (size_t)tree * (HIRA_MAX_LEVELS + 2);
    const size_t base0 = (size_t)tree * p.cap[0];
    for (int j = t; j < D; j += NT) x[j] = load_elem<T>(key, j);
    __syncthreads();
    int top = 1;  // levels 1 .. top get a new node
    int parent = -1, pcount = 0;
    float pdist = 0.0f, prad = 0.0f;
    for (; top < L - 1; ++top) {  // uniform
        parent = nearest_with_room<T, NT>(p, tree, top + 1, 0, s_used[top + 1], x, red_f, red_i, nullptr, &pcount, &pdist,
                                      &prad);
        if (parent >= 0) break;
    }
    const long long idx = parent >= 0 ? (long long)parent * bf + pcount : s_used[top];
    bool fits = true;  // every new node below is the first child of the new node above
    long long id = idx;
    for (int l = top; l >= 1; --l) {
        if (id >= p.cap[l]) fits = false;
        id *= bf;
    }
    if (id >= p.cap[0]) fits = false;
    __syncthreads();  // (everybody has read the sizes)
    if (!fits) {
        if (t == 0) st[HIRA_MAX_LEVELS + 1] = 1;
        __syncthreads();
        return -1;  // uniform
    }
    // the path above the new nodes: radii, and the distances between centres (a wave per level)
    for (int l = top + 1 + wave; l < L; l += NT / 64) {  // uniform in the wave
        float d = sqrtf(pdist), rad_now = prad;
        if (l > top + 1) {
            const size_t node = ancestor_of((size_t)parent, l - top, bf);
            rad_now = p.radii[l][(size_t)tree * p.cap[l] + node];
            const size_t child = ancestor_of((size_t)parent, l - top - 1, bf);
            const size_t bl = (size_t)tree * p.cap[l], bc = (size_t)tree * p.cap[l - 1];
            float ss = 0.0f;
            for (int j = lane; j < D; j += 64) {
                const float a = load_elem<T>(p.centers[l - 1], bc * D + elem_index(p.layout, D, child, j));
                const float b = load_elem<T>(p.centers[l], bl * D + elem_index(p.layout, D, node, j));
                ss += (a - b) * (a - b);
            }
            ss = wave_sum(ss);
            d = sqrtf(ss);
        }
        if (lane == 0) {
            s_dist[l] = d;
            s_rad[l] = rad_now;
        }
    }
    // the new nodes, the key, its value
    id = idx;
    for (int l = top; l >= 1; --l) {
        const size_t bl = (size_t)tree * p.cap[l];
        for (int j = t; j < D; j += NT)
            store_elem<T>(p.centers[l], bl * D + elem_index(p.layout, D, (size_t)id, j), x[j]);
        if (t == 0) {
            p.radii[l][bl + id] = 0.0f;
            p.counts[l][bl + id] = 1;
            if (id + 1 > s_used[l]) s_used[l] = st[l] = (int)(id + 1);
            s_dist[l] = s_rad[l] = 0.0f;
        }
        id *= bf;
    }
    const size_t slot = (size_t)id;
    const int node1 = (int)(id / bf);
    for (int j = t; j < D; j += NT)
        store_elem<T>(p.keys, base0 * D + elem_index(p.key_layout, D, slot, j), x[j]);
    if (p.new_values && p.values)
        for (int j = t; j < Dv; j += NT)
            store_elem<T>(p.values, (base0 + slot) * Dv + j, load_elem<T>(p.new_values, ((size_t)tree * p.m + i) * Dv + j));
    float worst = 0.0f;
    if (p.keys8 != nullptr) {
        for (int j = t; j < D; j += NT) {
            const float u = x[j] / p.kscale[(size_t)tree * D + j];
            const float r = fminf(fmaxf(rintf(u), -127.0f), 127.0f);
            worst = fmaxf(worst, fabsf(u - r));
            p.keys8[base0 * D + shadow_index(D, slot, j)] = (int8_t)(int)r;
        }
        worst = wave_max(worst);
        if (lane == 0) red_f[wave] = worst;
    }
    __syncthreads();
    if (t == 0) {
        if (p.keys8 != nullptr) {  // (the node holds no other key: its bound starts here)
            float w = red_f[0];
#pragma unroll
            for (int i = 1; i < NT / 64; ++i) w = fmaxf(w, red_f[i]);
            p.keps[(size_t)tree * p.cap[1] + node1] = w;
        }
        p.perm[base0 + slot] = position;
        st[HIRA_MAX_LEVELS] = position + 1;
        if (parent >= 0) p.counts[top + 1][(size_t)tree * p.cap[top + 1] + parent] = pcount + 1;
        float r_child = 0.0f;
        for (int l = top + 1; l < L; ++l) {
            const float rn = fmaxf(s_rad[l], pad_up(s_dist[l] + r_child));
            if (rn != s_rad[l]) p.radii[l][(size_t)tree * p.cap[l] + ancestor_of((size_t)parent, l - top, bf)] = rn;
            s_rad[l] = r_child = rn;
        }
    }
    __syncthreads();
    return node1;
}

// All that is left of a chunk, keys [k, nk), once no listed node has room: from there on a key opens a node, the
// bf - 1 behind it fill that one, whatever their distance, and the next opens another.  So everything is known but
// the parents, and what was a chain of openings (parent, distances to the new node, choice: 4.6 us each) is one pass:
// the openers' distances to the listed level-2 nodes and everybody's to its opener at once, the parents one after
// the other by one wave, the paths above them together.  A window of 64 keys, two openings, 18.5 -> 12.3 us (with what the other waves do beside wave 0).
// The new nodes then stand in the list as candidates do, take their counts and radii to memory as they do, and the
// last one stays as the list.  The keys' rows go the way of all others (s_slot).  Returns the first key that is
// left (k: none was placed): at one that no listed parent takes, whose node's slot lies behind the capacity, or
// whose distance is no finite number.
template <typename T, int NT>
__device__ __forceinline__ int open_run(const UpdateParams& p, const int tree, int* s_used, int* s_slot, int* s_stop, const T* rows,
                                        const T* par, WindowLds& w, float* cen, float* table, const int k, const int nk) {
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int D = p.dim, L = p.num_levels, bf = p.bf, n2 = w.n2;
    const size_t b1 = (size_t)tree * p.cap[1];
    const int most = min((nk - k + bf - 1) / bf, kCandMax);  // openers: keys k, k + bf, ...
    const int end = min(nk, k + most * bf);
    float* far = table + kCandMax * kParentsMax;  // (kWinKeys) squared distances to the openers
    // (the additions are those of a butterfly of lane ^ 1, ^ 2, ..., ^ 32, the general way's)
    auto total = [&](float ss) {
        ss += win_partner<1>(ss);
        ss += win_partner<2>(ss);
        ss += win_partner<4>(ss);
        ss += win_partner<8>(ss);
        ss = win_sum_across<16>(ss);
        return win_sum_across<32>(ss);
    };
    auto apart = [&](const T* x, const T* y) {
        float ss = 0.0f;
        for (int j = lane; j < D; j += 64) {
            const float df = load_elem<T>(x, j) - load_elem<T>(y, j);
            ss += df * df;
        }
        return ss;
    };
    // (numbers below a few thousand: the float quotients are exact)
    const float inv_bf = 1.0f / (float)bf, inv_n2 = 1.0f / (float)max(n2, 1);
    auto over = [](int x, float inv) { return (int)(((float)x + 0.5f) * inv); };
    // (wave 0 comes from taking the list before to memory, and asks for the parents' radii meanwhile)
    constexpr int NW = NT / 64 - 1;
    float rad2 = 0.0f;
    if (wave == 0 && lane < n2) rad2 = p.radii[2][(size_t)tree * p.cap[2] + w.id2[min(lane, kParentsMax - 1)]];
    for (int e = wave - 1; e < most * n2 && wave > 0; e += NW) {  // uniform in the wave
        const int i = over(e, inv_n2), c = e - i * n2;
        const float ss = total(apart(rows + (size_t)(k + i * bf) * D, par + (size_t)c * D));
        if (lane == 0) table[i * kParentsMax + c] = ss;
    }
    for (int q0 = k + wave - 1; q0 < end && wave > 0; q0 += NW * 5) {  // uniform in the wave; five keys at a time
        float ss[5];
#pragma unroll
        for (int u = 0; u < 5; ++u) {
            const int q = min(q0 + u * NW, end - 1);
            ss[u] = apart(rows + (size_t)q * D, rows + (size_t)(k + over(q - k, inv_bf) * bf) * D);
        }
#pragma unroll
        for (int u = 0; u < 5; ++u) {
            const int q = q0 + u * NW;
            const float d = total(ss[u]);
            if (lane == 0 && q < end) far[q - k] = over(q - k, inv_bf) * bf == q - k ? 0.0f : d;
        }
    }
    __syncthreads();
    if (wave == 0) {
        int cnt2 = lane < n2 ? w.cnt2[lane] : bf;
        const int id2 = lane < n2 ? w.id2[min(lane, kParentsMax - 1)] : 0x7fffffff, had2 = cnt2;
        const int grp = over(lane, inv_bf);  // of key k + lane
        const float mine = lane < end - k ? far[lane] : 0.0f;
        const unsigned long long bad = __ballot(!(mine < INFINITY));
        int stop = bad != 0ull ? k + __ffsll((long long)bad) - 1 : end;
        int n = 0, used = s_used[1];
        for (; n < most && k + n * bf < stop; ++n) {
            const float have = lane < n2 && cnt2 < bf ? table[n * kParentsMax + min(lane, kParentsMax - 1)] : INFINITY;
            const float d = have < INFINITY ? have : INFINITY;
            const float best = win_min(d);
            if (best == INFINITY) break;
            unsigned long long who = __ballot(d == best);
            if (who & (who - 1ull)) {  // ties: the lowest node
                int low = d == best ? id2 : 0x7fffffff;
                low = wave_min(low);
                who = __ballot(d == best && id2 == low);
            }
            const int c = __ffsll((long long)who) - 1;
            const int parent = __builtin_amdgcn_readlane(id2, c);
            const long long idx = (long long)parent * bf + __builtin_amdgcn_readlane(cnt2, c);
            if (idx >= p.cap[1] || idx * bf >= p.cap[0]) break;
            if (lane == c) ++cnt2;
            used = max(used, (int)(idx + 1));
            if (lane == 0) {
                w.id[n] = (int)idx;
                w.anc_id[2][n] = parent;
                w.anc_step[2][n] = sqrtf(best);
                w.anc_rad[2][n] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(rad2), c));
            }
        }
        stop = min(stop, k + n * bf);
        if (lane < n) {
            w.cnt[lane] = min(bf, stop - k - lane * bf);
            w.cnt0[lane] = 0;  // (memory has neither count nor radius of it)
            w.rad[lane] = -INFINITY;
            w.far[lane] = 0.0f;
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
        if (lane < stop - k) {
            s_slot[k + lane] = w.id[grp] * bf + (lane - grp * bf);
            atomicMax(reinterpret_cast<int*>(&w.far[grp]), __float_as_int(mine));  // (not negative: ordered as integers)
        }
        if (lane < n2 && cnt2 != had2) {
            w.cnt2[lane] = cnt2;
            p.counts[2][(size_t)tree * p.cap[2] + id2] = cnt2;
        }
        if (lane == 0) {
            if (used != s_used[1]) s_used[1] = p.state[(size_t)tree * (HIRA_MAX_LEVELS + 2) + 1] = used;
            w.n = n;
            *s_stop = stop;
        }
    }
    __syncthreads();
    const int n = w.n, stop = *s_stop;
    if (n == 0) return k;  // uniform
    for (int i = wave - 1; i < n && wave > 0; i += NW)  // uniform in the wave
        for (int j = lane; j < D; j += 64) {
            const float x = load_elem<T>(rows, (size_t)(k + i * bf) * D + j);
            store_elem<T>(p.centers[1], b1 * D + elem_index(p.layout, D, (size_t)w.id[i], j), x);
            if (i == n - 1) cen[j] = x;
        }
    if (p.keps != nullptr && t < n) p.keps[b1 + w.id[t]] = 0.0f;  // (its keys' rows raise it)
    for (int e = wave; e < n * (L - 3); e += NT / 64) {  // the paths above level 2: a wave per node and level
        const int i = e % n, l = 3 + e / n;
        const size_t parent = (size_t)w.anc_id[2][i], node = ancestor_of(parent, l - 1, bf);
        const size_t bl = (size_t)tree * p.cap[l];
        const float rad_now = p.radii[l][bl + node];
        const size_t child = ancestor_of(parent, l - 2, bf), bc = (size_t)tree * p.cap[l - 1];
        float ss = 0.0f;
        for (int j = lane; j < D; j += 64) {
            const float a = load_elem<T>(p.centers[l - 1], bc * D + elem_index(p.layout, D, child, j));
            const float b = load_elem<T>(p.centers[l], bl * D + elem_index(p.layout, D, node, j));
            ss += (a - b) * (a - b);
        }
        ss = wave_sum(ss);
        if (lane == 0) {
            w.anc_id[l][i] = (int)node;
            w.anc_step[l][i] = sqrtf(ss);
            w.anc_rad[l][i] = rad_now;
        }
    }
    if (L > 3) __syncthreads();  // uniform
    if (wave == 0) {
        for (int l = 2; l < L; ++l)
            if (lane < n) {
                const int anc = w.anc_id[l][lane];
                int first = lane;
                for (int o = lane - 1; o >= 0; --o) first = w.anc_id[l][o] == anc ? o : first;
                w.anc_rep[l][lane] = first;
            }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
        window_flush(p, tree, w);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
        if (lane == 0) {  // the last one is the list
            const int c = n - 1;
            w.n = 1;
            w.id[0] = w.id[c];
            w.cnt[0] = w.cnt0[0] = w.cnt[c];
            w.rad[0] = pad_up(sqrtf(w.far[c]));
            w.far[0] = -1.0f;
            for (int l = 2; l < L; ++l) {
                w.anc_id[l][0] = w.anc_id[l][c];
                w.anc_step[l][0] = w.anc_step[l][c];
                w.anc_rad[l][0] = w.anc_rad[l][w.anc_rep[l][c]];
                w.anc_rep[l][0] = 0;
            }
        }
    }
    __syncthreads();
    return stop;
}

template <typename T, int COLS>
__global__ __launch_bounds__(kWinThreads) void k_update_window(const UpdateParams p, const SampleRows sample) {
    // 2 D floats of the general way, kCandMax centres, the table of distances, kParents centres, a chunk of key rows
    extern __shared__ __attribute__((aligned(16))) float sm[];
    constexpr int NT = kWinThreads;
    __shared__ float red_f[NT / 64];
    __shared__ int red_i[NT / 64];
    __shared__ float s_dist[HIRA_MAX_LEVELS], s_rad[HIRA_MAX_LEVELS];
    __shared__ WindowLds w;
    __shared__ int s_slot[kWinKeys];  // where the chunk's keys went (-1: placed the general way, or dropped)
    __shared__ int s_done;            // keys of the chunk dealt with so far
    __shared__ bool s_room;           // a listed node has room
    __shared__ int s_used[HIRA_MAX_LEVELS];  // slots in use per level
    touch_update_arguments();
    if ((int)blockIdx.x >= sample.trees) {  // uniform in the workgroup
        replace_sample<kWinThreads>(p, sample);
        return;
    }
    constexpr int EPL = Elem<T>::kPerChunk;
    const int tree = blockIdx.x;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int D = p.dim, Dv = p.vdim, L = p.num_levels, bf = p.bf;
    float* cen = sm + 2 * (size_t)D;
    float* table = cen + (size_t)kCandMax * D;
    T* par = reinterpret_cast<T*>(table + (size_t)kCandMax * kWinKeys);
    T* rows = par + (size_t)kParents<T> * D;  // (kWinKeys, D): the chunk's keys
    uint4* vals = p.stage_values ? reinterpret_cast<uint4*>(rows + (size_t)kWinKeys * D) : nullptr;  // its values
    int32_t* st = p.state + (size_t)tree * (HIRA_MAX_LEVELS + 2);
    const size_t base0 = (size_t)tree * p.cap[0], b1 = (size_t)tree * p.cap[1];
    const bool with_values = p.new_values != nullptr && p.values != nullptr;
    const int kc = D / EPL;
    auto stage = [&](int i0) {  // the rows of the chunk that starts at key i0 into LDS
        const int nk = min(kWinKeys, p.m - i0);
        const uint4* src = reinterpret_cast<const uint4*>(reinterpret_cast<const T*>(p.new_keys) +
                                                          ((size_t)tree * p.m + i0) * D);
        const uint4* vsrc = vals == nullptr ? nullptr
                                            : reinterpret_cast<const uint4*>(reinterpret_cast<const T*>(p.new_values) +
                                                                             ((size_t)tree * p.m + i0) * Dv);
        typedef uint32_t vec4 __attribute__((ext_vector_type(4)));  // (an array of uint4 stays in memory here)
        constexpr int SU = 2048 / NT;
        const int nc = nk * kc, nv = vals == nullptr ? 0 : nk * (Dv / EPL);
        for (int e0 = t; e0 < nc + nv; e0 += SU * NT) {
            vec4 raw[SU];
#pragma unroll
            for (int u = 0; u < SU; ++u) {
                const int e = min(e0 + u * NT, nc + nv - 1);
                raw[u] = *reinterpret_cast<const vec4*>(e < nc ? src + e : vsrc + (e - nc));
            }
#pragma unroll
            for (int u = 0; u < SU; ++u) {
                const int e = e0 + u * NT;
                if (e < nc) reinterpret_cast<vec4*>(rows)[e] = raw[u];
                else if (e < nc + nv) reinterpret_cast<vec4*>(vals)[e - nc] = raw[u];
            }
        }
    };
    int position = st[HIRA_MAX_LEVELS];  // of the next key (every thread carries it along)
    // (the state is asked for with the first rows, not behind them)
    const int st0 = st[0], st1 = st[1], st2 = st[2], my_used = t < HIRA_MAX_LEVELS ? st[t] : 0;
    stage(0);
    if (t >= 1 && t < L) s_used[t] = my_used;
    int i0 = 0;
    bool flushed = false;  // (wave 0's)
    bool general = !window_candidates<T, NT>(p, tree, st0, st1, st2, w, cen, par);  // uniform: what is left goes the general way
    while (i0 < p.m && !general) {  // uniform
        int nk = min(kWinKeys, p.m - i0);
        bool list_anew = false;  // behind this chunk
        const int position0 = position;
        if (i0 > 0) {
            stage(i0);  // (behind the barrier that ends the chunk before: nobody needs its rows any more)
            __syncthreads();
        }
        window_distances<T, COLS, NT>(D, w, cen, rows, 0, nk, table);
        for (int k = 0; k < nk;) {  // uniform
            __syncthreads();
            if (wave == 0) {
                const int n = w.n;
                int cnt = lane < n ? w.cnt[lane] : bf;
                const int id = lane < n ? w.id[lane] : 0x7fffffff;
                const int cl = min(lane, kCandMax - 1);
                float far = lane < n ? w.far[lane] : -1.0f;
                float next = table[k * kCandMax + cl];
                int kk = k;
                for (; kk < nk; ++kk) {
                    // a single node with room takes the keys that follow until it is full: a key a lane
                    const unsigned long long room = __ballot(cnt < bf);
                    if (room != 0ull && (room & (room - 1ull)) == 0ull) {
                        const int c = __ffsll((long long)room) - 1;
                        const int have = __builtin_amdgcn_readlane(cnt, c), node = __builtin_amdgcn_readlane(id, c);
                        const int take = min(bf - have, nk - kk);
                        const float d = lane < take ? table[(kk + lane) * kCandMax + c] : 0.0f;
                        if (__ballot(!(d < INFINITY)) == 0ull) {
                            if (lane < take) s_slot[kk + lane] = node * bf + have + lane;
                            const float most = -win_min(-d);
                            if (lane == c) {
                                cnt += take;
                                far = fmaxf(far, most);
                            }
                            kk += take - 1;
                            next = table[min(kk + 1, nk - 1) * kCandMax + cl];
                            continue;
                        }
                    }
                    const float d = cnt < bf ? next : INFINITY;
                    next = table[min(kk + 1, nk - 1) * kCandMax + cl];
                    const float best = win_min(d);
                    if (best == INFINITY) break;  // no node has room
                    unsigned long long who = __ballot(d == best);
                    if (who & (who - 1ull)) {  // ties: the lowest node
                        int low = d == best ? id : 0x7fffffff;
                        low = wave_min(low);
                        who = __ballot(d == best && id == low);
                    }
                    if (lane == __ffsll((long long)who) - 1) {
                        s_slot[kk] = id * bf + cnt;
                        ++cnt;
                        far = fmaxf(far, d);
                    }
                }
                if (lane < n) {
                    w.cnt[lane] = cnt;
                    w.far[lane] = far;
                }
                const bool room = __ballot(cnt < bf) != 0ull;
                if (lane == 0) {
                    s_done = kk;
                    s_room = room;
                    if (kk < nk) s_slot[kk] = -1;
                }
            }
            __syncthreads();
            const int kd = s_done;
            position += kd - k;
            k = kd;
            if (k < nk) {
                // key k found no node with room, or none at a distance that is a finite number: it opens one
                list_anew = s_room;
                window_flush(p, tree, w);
                const T* key = rows + (size_t)k * D;
                if (!list_anew && L > 2 && w.n2 <= kParents<T>) {  // uniform
                    const int k1 = open_run<T, NT>(p, tree, s_used, s_slot, &s_done, rows, par, w, cen, table, k, nk);
                    if (k1 > k) {
                        position += k1 - k;
                        k = k1;
                        if (k < nk) window_distances<T, COLS, NT>(D, w, cen, rows, k, nk, table);
                        continue;
                    }
                }
                {
                    // (with no room left in the list a node of level 2 is opened too, the only one there with room then)
                    bool none2 = w.n2 <= kParents<T>;
                    for (int e = 0; none2 && e < w.n2; ++e) none2 = w.cnt2[e] >= bf;
                    const int node = open_node<T, NT>(p, tree, i0 + k, position, s_used, key, sm, red_f, red_i, s_dist, s_rad);
                    if (node >= 0) ++position;
                    if (list_anew) {  // uniform
                        nk = k + 1;
                        break;
                    }
                    // (all listed nodes are full: the new one is the whole list from here on)
                    if (t == 0) {
                        w.n = node >= 0 ? 1 : 0;
                        w.id[0] = node;
                        w.cnt[0] = w.cnt0[0] = 1;
                        w.rad[0] = s_rad[1];
                        w.far[0] = -1.0f;
                        for (int l = 2; l < L; ++l) {
                            w.anc_id[l][0] = (int)ancestor_of((size_t)max(node, 0), l, bf);
                            w.anc_rep[l][0] = 0;
                            w.anc_step[l][0] = s_dist[l];
                            w.anc_rad[l][0] = s_rad[l];
                        }
                        w.n2 = none2 && node >= 0 ? 1 : kParents<T> + 1;
                        w.id2[0] = node / bf;
                        w.cnt2[0] = 1;
                    }
                    for (int j = t; j < D; j += NT) {  // (its centre is the key)
                        cen[j] = sm[j];
                        par[j] = key[j];
                    }
                    __syncthreads();
                }
                ++k;
                // (of the keys that it has room for: those behind them find it full, whatever the distance)
                window_distances<T, COLS, NT>(D, w, cen, rows, k, min(nk, k + bf - 1), table);
            }
        }
        // ---- the rows of the keys placed from the list, 16 bytes a thread -----------------------
        if (p.keys8 != nullptr) {  // thread 0's bounds of nodes opened here, ahead of the maxima that raise them
            if (wave == 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
        }
        float step[16];  // of a chunk of the 8-bit shadow: a thread's columns are the same for all its keys
        const int sc = D / 16, my_chunk = t % max(sc, 1);
        if (p.keys8 != nullptr)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float4 v = reinterpret_cast<const float4*>(p.kscale + (size_t)tree * D + my_chunk * 16)[q];
                step[q * 4] = v.x, step[q * 4 + 1] = v.y, step[q * 4 + 2] = v.z, step[q * 4 + 3] = v.w;
            }
        const bool v_chunks = with_values && Dv % EPL == 0;
        const int vc = v_chunks ? Dv / EPL : 0, per = kc + vc;
        // (behind the last chunk wave 0 takes the list to memory meanwhile)
        const bool last = i0 + nk >= p.m && !list_anew;  // uniform
        const int rt = last ? t - 64 : t, rn = last ? NT - 64 : NT;
        if (last && wave == 0) {
            window_flush(p, tree, w);
            flushed = true;
        }
        constexpr int RU = 4;  // chunks a thread has in flight
        const float inv_per = 1.0f / (float)per;  // (at most 64 x 128 chunks: the float quotient is exact)
        for (int e0 = rt; e0 < nk * per && rt >= 0; e0 += RU * rn) {
            uint4 raw[RU];
            T* dst[RU];
#pragma unroll
            for (int u = 0; u < RU; ++u) {
                const int e = min(e0 + u * rn, nk * per - 1);
                const int q = (int)(((float)e + 0.5f) * inv_per), c = e - q * per, slot = s_slot[q];
                const size_t r = (size_t)tree * p.m + i0 + q;
                const bool key = c < kc;
                if (key) raw[u] = reinterpret_cast<const uint4*>(rows)[q * kc + c];
                else if (vals != nullptr) raw[u] = vals[q * vc + c - kc];
                else raw[u] = load_chunk<T>(p.new_values, r * Dv, c - kc);
                dst[u] = slot < 0 || e0 + u * rn >= nk * per
                             ? nullptr
                             : (key ? reinterpret_cast<T*>(p.keys) + base0 * D + elem_index(p.key_layout, D, (size_t)slot, c * EPL)
                                    : reinterpret_cast<T*>(p.values) + (base0 + slot) * Dv + (c - kc) * EPL);
            }
#pragma unroll
            for (int u = 0; u < RU; ++u)
                if (dst[u] != nullptr) *reinterpret_cast<uint4*>(dst[u]) = raw[u];
        }
        if (with_values && !v_chunks)  // (value rows that are not made of chunks)
            for (int e = t; e < nk * Dv; e += NT) {
                const int q = e / Dv, j = e - q * Dv;
                if (s_slot[q] >= 0)
                    store_elem<T>(p.values, (base0 + s_slot[q]) * Dv + j,
                                  load_elem<T>(p.new_values, ((size_t)tree * p.m + i0 + q) * Dv + j));
            }
        // (positions: the chunk's keys in order, without those that were dropped -- which can only
        // be keys that found no room, so every key before the first dropped one has its plain place)
        if (wave == 0 && lane < nk) {
            const int slot = s_slot[lane];
            if (slot >= 0) p.perm[base0 + slot] = position0 + lane;
        }
        if (p.keys8 != nullptr) {
            // the keys' 8-bit shadow with the tree's steps; a component beyond +-127 steps clips,
            // and the node's error bound then covers it.  Sixteen columns a thread, 4 or 8 threads a key.
            for (int e0 = 0; e0 < nk * sc; e0 += NT) {  // uniform
                const int q = min((e0 + t) / sc, nk - 1), slot = e0 + t < nk * sc ? s_slot[q] : -1;
                float worst = 0.0f;
                uint32_t out[4];
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    out[g] = 0;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float u = load_elem<T>(rows, (size_t)q * D + my_chunk * 16 + g * 4 + e) / step[g * 4 + e];
                        const float k8 = fminf(fmaxf(rintf(u), -127.0f), 127.0f);
                        worst = fmaxf(worst, fabsf(u - k8));
                        out[g] |= (uint32_t)(uint8_t)(int8_t)(int)k8 << (8 * e);
                    }
                }
                worst = fmaxf(worst, win_partner<1>(worst));
                worst = fmaxf(worst, win_partner<2>(worst));
                if (sc > 4) worst = fmaxf(worst, win_partner<4>(worst));  // uniform
                if (slot >= 0) {
                    *reinterpret_cast<uint4*>(p.keys8 + base0 * D + shadow_index(D, (size_t)slot, my_chunk * 16)) =
                        make_uint4(out[0], out[1], out[2], out[3]);
                    if (my_chunk == 0) atomicMax(reinterpret_cast<int*>(p.keps + b1 + slot / bf), __float_as_int(worst));
                }
            }
        }
        i0 += nk;
        if (list_anew) {  // uniform
            __syncthreads();
            general = !window_candidates<T, NT>(p, tree, st[0], st[1], st[2], w, cen, par);
        }
        if (i0 < p.m) __syncthreads();
    }
    if (general) {
        if (t == 0) st[HIRA_MAX_LEVELS] = position;
        __syncthreads();
        for (; i0 < p.m; ++i0) update_one_key<T, NT>(p, tree, i0, sm, red_f, red_i, s_dist, s_rad);
        return;
    }
    if (!flushed) window_flush(p, tree, w);
    if (wave == 0) {
        // the bound of the next search for room: the lowest listed node that still has some, or
        // the lowest slot that was no node when the list was made
        int low = lane < w.n && w.cnt[lane] < bf ? w.id[lane] : 0x7fffffff;
        low = wave_min(low);
        if (lane == 0) {
            st[0] = min(low, min(w.low_empty, s_used[1]));
            st[HIRA_MAX_LEVELS] = position;
        }
    }
}

}  // namespace hira

using namespace hira;

// hira_update's checks and the kernels' arguments; *window: the launch takes the window kernel
static int update_arguments(const HiraTree* tree, const void* new_keys, const void* new_values,
                            int32_t m, int32_t* state, UpdateParams* out, bool* window,
                            size_t* smem, size_t* smem_w) {
    HIRA_CHECK_ARG(tree != nullptr && new_keys != nullptr && state != nullptr,
                   "tree / new_keys / state missing");
    HIRA_CHECK_ARG(tree->dtype == HIRA_F32 || tree->dtype == HIRA_BF16, "dtype %d", tree->dtype);
    HIRA_CHECK_ARG(tree->num_levels >= 1 && tree->num_levels <= HIRA_MAX_LEVELS, "num_levels %d",
                   tree->num_levels);
    HIRA_CHECK_ARG(tree->bf >= 1 && tree->bf <= 64, "branching factor %d", tree->bf);
    HIRA_CHECK_ARG(m >= 0, "m = %d", m);
    HIRA_CHECK_ARG(tree->keys && tree->perm, "keys / perm missing");
    HIRA_CHECK_ARG((new_values == nullptr) || tree->values != nullptr,
                   "values given but the index holds none");
    UpdateParams& p = *out;
    memset(&p, 0, sizeof(p));
    *window = false;
    *smem = *smem_w = 0;
    if (m == 0) return HIRA_OK;  // nothing to append: the callers launch nothing for it
    p.keys = tree->keys;
    p.values = tree->values;
    p.perm = tree->perm;
    for (int l = 0; l < HIRA_MAX_LEVELS; ++l) {
        p.centers[l] = tree->centers[l];
        p.radii[l] = tree->radii[l];
        p.counts[l] = tree->counts[l];
        p.cap[l] = tree->cap[l];
    }
    for (int l = 1; l < tree->num_levels; ++l)
        HIRA_CHECK_ARG(p.centers[l] && p.radii[l] && p.counts[l], "level %d arrays missing", l);
    p.num_levels = tree->num_levels;
    p.bf = tree->bf;
    p.dim = tree->dim;
    p.vdim = tree->vdim;
    p.layout = center_layout_of(tree->layout);
    p.key_layout = key_layout_of(tree->layout);
    if (tree->layout == HIRA_TILE16_Q8) {
        HIRA_CHECK_ARG(tree->keys8 && tree->kscale && tree->keps && tree->num_levels >= 2,
                       "keys8 / kscale / keps missing");
        p.keys8 = tree->keys8;
        p.kscale = tree->kscale;
        p.keps = tree->keps;
    }
    p.new_keys = new_keys;
    p.new_values = new_values;
    p.m = m;
    p.state = state;
    *smem = 2 * (size_t)tree->dim * sizeof(float);
    // windows of a few keys and more: the nodes with room are listed in LDS (where they fit: 48 centres
    // of up to 256 columns, bf16 320, and those of level 2 beside the table of distances and a chunk of rows)
    *smem_w = *smem + (size_t)kCandMax * (tree->dim + kWinKeys) * sizeof(float) + (size_t)64 * tree->dim +
              (size_t)kWinKeys * tree->dim * (tree->dtype == HIRA_F32 ? 4 : 2);
    *window = m >= 4 && tree->num_levels >= 2 && tree->dim <= 64 * (tree->dtype == HIRA_F32 ? 4 : kWinColsMax) && *smem_w <= kWinLds;
    const size_t vrow = (size_t)tree->vdim * (tree->dtype == HIRA_F32 ? 4 : 2);
    if (new_values != nullptr && vrow % 16 == 0 && *smem_w + kWinKeys * vrow <= kWinLds) {
        p.stage_values = 1;
        *smem_w += kWinKeys * vrow;
    }
    return HIRA_OK;
}

// workgroups: one a tree, and as many as the sample's rows take
static unsigned update_grid(const SampleRows& r, int threads) {
    return (unsigned)(r.trees + (r.trees * r.n * r.chunks + threads - 1) / threads);
}

// The window kernel's LDS, its own lists beside the dynamic part, can exceed what a launch gets
// without asking: asked for once per kernel and device.
template <typename T, int COLS>
static int launch_update_window(const UpdateParams& p, const SampleRows& sample, size_t smem, hipStream_t s) {
    constexpr int kMaxDevices = 64;
    static int asked[kMaxDevices];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices)
        return fail(HIRA_ELAUNCH, "update: no current device");
    if (__atomic_load_n(&asked[dev], __ATOMIC_RELAXED) == 0) {
        if (hipFuncSetAttribute(reinterpret_cast<const void*>(&k_update_window<T, COLS>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)kWinLds) != hipSuccess)
            return fail(HIRA_ELAUNCH, "update: %zu bytes of LDS refused", kWinLds);
        __atomic_store_n(&asked[dev], 1, __ATOMIC_RELAXED);
    }
    hipLaunchKernelGGL((k_update_window<T, COLS>), dim3(update_grid(sample, kWinThreads)), dim3(kWinThreads), smem, s, p,
                       sample);
    return HIRA_OK;
}

namespace hira {
struct StateRow {
    int32_t v[HIRA_MAX_LEVELS + 2];
};
__global__ void k_update_state(int32_t* state, const StateRow row, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) state[i] = row.v[i % (HIRA_MAX_LEVELS + 2)];
}
}  // namespace hira

/* see include/hira_hip.h */
extern "C" int hira_update_state(const HiraTree* tree, int32_t num_keys, int32_t* state, void* stream) {
    HIRA_CHECK_ARG(tree && state && tree->num_trees >= 1 && tree->num_levels >= 1 &&
                       tree->num_levels <= HIRA_MAX_LEVELS,
                   "hira_update_state: tree / state");
    StateRow row;
    memset(&row, 0, sizeof(row));
    for (int l = tree->num_levels == 1 ? 0 : 1; l < tree->num_levels; ++l) row.v[l] = tree->size[l];
    row.v[HIRA_MAX_LEVELS] = num_keys;
    const int n = tree->num_trees * (HIRA_MAX_LEVELS + 2);
    hipLaunchKernelGGL(k_update_state, dim3((n + 255) / 256), dim3(256), 0, reinterpret_cast<hipStream_t>(stream),
                       state, row, n);
    HIRA_CHECK_LAUNCH("hira_update_state");
    return HIRA_OK;
}

static int update_launch(const HiraTree* tree, const UpdateParams& p, const SampleRows& sample, bool window, size_t smem,
                         size_t smem_w, hipStream_t s) {
    if (window) {
        const int rc = tree->dtype == HIRA_F32
                           ? launch_update_window<float, 4>(p, sample, smem_w, s)
                           : tree->dim <= 256 ? launch_update_window<bf16_t, 4>(p, sample, smem_w, s)
                                              : launch_update_window<bf16_t, kWinColsMax>(p, sample, smem_w, s);
        if (rc != HIRA_OK) return rc;
    } else {
        const dim3 grid(update_grid(sample, kUpdThreads)), block(kUpdThreads);
        if (tree->dtype == HIRA_F32) hipLaunchKernelGGL(k_update<float>, grid, block, smem, s, p, sample);
        else hipLaunchKernelGGL(k_update<bf16_t>, grid, block, smem, s, p, sample);
    }
    HIRA_CHECK_LAUNCH("update kernel");
    return HIRA_OK;
}

/* see include/hira_hip.h */
extern "C" int hira_update(const HiraTree* tree, const void* new_keys, const void* new_values,
                           int32_t m, int32_t* state, void* stream) {
    return hira_update_sample(tree, new_keys, new_values, m, state, nullptr, 0, nullptr, nullptr, 0, stream);
}

/* see include/hira_hip.h */
extern "C" int hira_update_sample(const HiraTree* tree, const void* new_keys, const void* new_values, int32_t m,
                                  int32_t* state, void* sample, int32_t rows_per_tree, const int32_t* slot_host,
                                  const int32_t* from_host, int32_t n, void* stream) {
    UpdateParams p;
    bool window;
    size_t smem, smem_w;
    if (const int rc = update_arguments(tree, new_keys, new_values, m, state, &p, &window, &smem, &smem_w))
        return rc;
    SampleRows r;
    memset(&r, 0, sizeof(r));
    r.trees = tree->num_trees;
    HIRA_CHECK_ARG(n >= 0 && (n == 0 || (sample && slot_host && from_host)), "hira_update_sample: null argument");
    for (int i = 0; i < n; ++i)
        HIRA_CHECK_ARG(slot_host[i] >= 0 && slot_host[i] < rows_per_tree && from_host[i] >= 0 && from_host[i] < m,
                       "hira_update_sample: row %d from %d", slot_host[i], from_host[i]);
    const int row = tree->dim * (tree->dtype == HIRA_F32 ? 4 : 2);
    // (the launch takes a few rows, whole and aligned, each slot once; otherwise a launch of their own behind it)
    const bool along = n > 0 && n <= kSamplePairs && row % 16 == 0 && (((uintptr_t)sample | (uintptr_t)new_keys) & 15) == 0 &&
                       (int64_t)tree->num_trees * n * (row / 16) < (int64_t)1 << 31;
    if (along) {
        r.dst = static_cast<uint4*>(sample);
        r.chunks = row / 16;
        r.rows_per_tree = rows_per_tree;
        r.n = n;
        memcpy(r.slot, slot_host, n * sizeof(int32_t));
        memcpy(r.from, from_host, n * sizeof(int32_t));
    }
    if (m > 0)
        if (const int rc = update_launch(tree, p, r, window, smem, smem_w, reinterpret_cast<hipStream_t>(stream))) return rc;
    if (n > 0 && !along)
        return hira_replace_rows(sample, tree->dtype, tree->dim, tree->num_trees, rows_per_tree, new_keys, m, m, slot_host,
                                 from_host, n, stream);
    return HIRA_OK;
}

namespace hira {
// The state rows to the host that waits for them.  Value and ticket are one store of eight bytes, so nothing has to be
// ordered before it (a fence of the system's scope writes the L2 back, some 10 us).
__global__ __launch_bounds__(256) void k_tell_host(const int32_t* state, uint64_t* rows, uint32_t ticket, int n) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n)
        __hip_atomic_store(rows + i, ((uint64_t)ticket << 32) | (uint32_t)state[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
}  // namespace hira

// A launch behind the append's writes the rows into host memory, which the host watches: what ran before on the stream
// is over when they are there, as behind a copy that is waited for.  8 trees, windows of 64 keys, a call: 25 us; with
// the runtime's wait for the stream instead of the watching 28, a copy to the host and its wait 31; with rows that the
// append's launch writes itself 21, but then the caller goes on while that launch still runs.
// The host watches for as long as an append takes behind little else on its stream, then it leaves the waiting to the
// runtime.
constexpr std::chrono::microseconds kWatch(500);

/* see include/hira_hip.h */
extern "C" int hira_read_state(const HiraTree* tree, const int32_t* state, uint64_t* host_rows, uint32_t ticket, int32_t* most,
                               void* stream) {
    HIRA_CHECK_ARG(tree && state && host_rows && most && tree->num_trees >= 1, "hira_read_state: null argument");
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &capturing) != hipSuccess || capturing != hipStreamCaptureStatusNone) {
        (void)hipGetLastError();  // (refused here: not an error of the next call's)
        return fail(HIRA_ELAUNCH, "hira_read_state: a stream under capture cannot be waited for");
    }
    void* rows = nullptr;
    if (hipHostGetDevicePointer(&rows, host_rows, 0) != hipSuccess) {
        (void)hipGetLastError();
        return fail(HIRA_EINVAL, "hira_read_state: the rows do not lie in pinned host memory");
    }
    const int n = tree->num_trees * (HIRA_MAX_LEVELS + 2);
    hipLaunchKernelGGL(k_tell_host, dim3((n + 255) / 256), dim3(256), 0, s, state, static_cast<uint64_t*>(rows), ticket, n);
    HIRA_CHECK_LAUNCH("hira_read_state");
    for (int i = 0; i < HIRA_MAX_LEVELS + 2; ++i) most[i] = INT32_MIN;
    const auto begin = std::chrono::steady_clock::now();
    bool waited = false;
    for (int i = 0; i < n; ++i) {
        uint64_t v;
        for (int spins = 1; (uint32_t)((v = __atomic_load_n(host_rows + i, __ATOMIC_RELAXED)) >> 32) != ticket; ++spins) {
            if (waited) return fail(HIRA_ELAUNCH, "hira_read_state: the stream has ended without the rows");
            if (spins % 64 == 0 && std::chrono::steady_clock::now() - begin > kWatch) {
                if (hipStreamSynchronize(s) != hipSuccess) return fail(HIRA_ELAUNCH, "hira_read_state: the stream failed");
                waited = true;
            }
        }
        int32_t& to = most[i % (HIRA_MAX_LEVELS + 2)];
        to = std::max(to, (int32_t)(uint32_t)v);
    }
    __atomic_thread_fence(__ATOMIC_ACQUIRE);
    return HIRA_OK;
}

namespace hira {
template <typename T>
static void launch_update_threshold(int e, const UpdateParams& p, const HiraTree* tree, size_t smem,
                                    hipStream_t s, const void* samples, int S, const HiraQuery* qu,
                                    int method, int k, float* tau) {
    const T* x = static_cast<const T*>(samples);
    const T* q = static_cast<const T*>(qu->q);
    const dim3 grid(tree->num_trees + qu->num_q_heads), block(kTauThreads);
#define HIRA_UT_LAUNCH(E)                                                                         \
    hipLaunchKernelGGL((k_update_threshold<T, E>), grid, block, smem, s, p, tree->num_trees, x, S, \
                       q, qu->tree_q_off, qu->tree_q_heads, qu->group_size, method, k, tau)
    if (e == 1) HIRA_UT_LAUNCH(1);
    else if (e == 2) HIRA_UT_LAUNCH(2);
    else HIRA_UT_LAUNCH(4);
#undef HIRA_UT_LAUNCH
}
}  // namespace hira

/* see include/hira_hip.h */
extern "C" int hira_update_threshold(const HiraTree* tree, const void* new_keys,
                                     const void* new_values, int32_t m, int32_t* state,
                                     const void* samples, int32_t num_samples,
                                     const HiraQuery* query, int32_t method, int32_t k,
                                     float* tau_out, void* stream) {
    UpdateParams p;
    bool window;
    size_t smem, smem_w;
    if (const int rc = update_arguments(tree, new_keys, new_values, m, state, &p, &window, &smem, &smem_w))
        return rc;
    if (const int rc = check_threshold_arguments(samples, tree->dtype, tree->num_trees, num_samples,
                                                 tree->dim, query, method, k, tau_out))
        return rc;
    if (m == 0 || window) {
        // nothing to append, or a window that takes the window kernel: the two launches
        if (const int rc = hira_update(tree, new_keys, new_values, m, state, stream)) return rc;
        return hira_threshold(samples, tree->dtype, tree->num_trees, num_samples, tree->dim, query,
                              method, k, tau_out, stream);
    }
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    const int e = threshold_sort_registers(num_samples);
    if (tree->dtype == HIRA_F32)
        launch_update_threshold<float>(e, p, tree, smem, s, samples, num_samples, query, method, k, tau_out);
    else
        launch_update_threshold<bf16_t>(e, p, tree, smem, s, samples, num_samples, query, method, k, tau_out);
    HIRA_CHECK_LAUNCH("update + threshold kernel");
    return HIRA_OK;
}
