// 8-bit shadow of the keys (layout HIRA_TILE16_Q8): one step per tree and channel, the keys
// rounded to whole steps in [-127, 127] and stored in tiles of 16 rows x 64 columns, and per
// level-1 node the largest rounding (or clipping) error, in steps, among its keys.  The search
// scans the shadow first: with k = kscale * (k8 + e), |e| <= keps, a score obeys
//   |q.k - sum_j (q_j kscale_j) k8_j| <= keps * sum_j |q_j kscale_j|,
// so a key whose 8-bit score plus that bound stays below the threshold cannot be selected and
// its bf16 row is never fetched.  The reference keeps fp32 keys only (indexer/cuda.py:365-368);
// this is what halves the bytes of the leaf scan without touching the selected set.
#include "rows.h"

namespace hira {

constexpr int kQuantThreads = 256;
constexpr float kMinStep = 1e-30f;  // a channel that is zero in every key

// largest finite magnitude per channel.  A thread reads 16 bytes of a row (eight channels), a
// workgroup 256 / (D / 8) rows a step, eight steps in flight; its maxima join kscale (zeroed before)
// through integer atomic maxima -- the bits of non-negative floats order like unsigned integers,
// and a maximum does not depend on the order of arrival.  Bound by the read of the keys: 8 x 131072
// rows of 256 bytes 40 us, 6.7 TB/s (with two bytes a lane and one step in flight 212 us).
__global__ __launch_bounds__(kQuantThreads) void k_absmax(const uint16_t* keys, size_t tree_stride,
                                                          int rows, int D, float* kscale) {
    constexpr int U = 8;
    const int t = blockIdx.y;
    const int cpr = D / 8, per = kQuantThreads / cpr, c = threadIdx.x % cpr, r0 = threadIdx.x / cpr;
    float m[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) m[e] = 0.0f;
    if (r0 < per)
        for (int r = blockIdx.x * per * U + r0; r < rows; r += gridDim.x * per * U) {
            uint4 raw[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {  // (past the end: the last row again)
                const int row = min(r + u * per, rows - 1);
                raw[u] = *reinterpret_cast<const uint4*>(keys + ((size_t)t * tree_stride + row) * D + c * 8);
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                float f[8];
                unpack<bf16_t>(raw[u], f);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float a = fabsf(f[e]);
                    m[e] = a < INFINITY && a > m[e] ? a : m[e];
                }
            }
        }
    __shared__ float sm[kQuantThreads * 8];
#pragma unroll
    for (int e = 0; e < 8; ++e) sm[threadIdx.x * 8 + e] = m[e];  // (row r0 of D numbers: r0 * D + c * 8 + e)
    __syncthreads();
    for (int j = threadIdx.x; j < D; j += kQuantThreads) {
        float best = 0.0f;
        for (int k = 0; k < per; ++k) best = fmaxf(best, sm[k * D + j]);
        if (best > 0.0f) atomicMax(reinterpret_cast<unsigned*>(kscale) + (size_t)t * D + j, __float_as_uint(best));
    }
}

__global__ void k_zero_f32(float* p, size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0.0f;
}

// n steps of D channels a tree; absmax: `copies` maxima a channel, (n / D, copies, D)
__global__ void k_step_from_absmax(float* kscale, const float* absmax, int copies, int D, size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float* at = absmax + i / D * copies * D + i % D;
    float m = 0.0f;
    for (int c0 = 0; c0 < copies; c0 += 16) {  // (16 on their way: one after the other, 32 copies were 10 us)
        float v[16];
#pragma unroll
        for (int c = 0; c < 16; ++c) v[c] = at[(size_t)min(c0 + c, copies - 1) * D];
#pragma unroll
        for (int c = 0; c < 16; ++c) m = fmaxf(m, v[c]);
    }
    kscale[i] = fmaxf(m / 127.0f, kMinStep);
}

// a / b, given the reciprocal of b rounded to nearest: the product with it, and the remainder, which a fused
// multiply-add gives exactly, divided the same way (P. Markstein's correction; a division instruction sequence takes
// twice as many).  What is no finite number stays what the product is.
__device__ __forceinline__ float quotient(float a, float b, float reciprocal) {
    const float q = a * reciprocal;
    const float corrected = fmaf(fmaf(-q, b, a), reciprocal, q);
    return fabsf(q) < INFINITY ? corrected : q;
}

// one wave per level-1 node: its bf key slots -> shadow bytes, error bound of the node.  A lane takes
// 16 bytes of a row (eight channels: eight bytes of one chunk of the shadow), D / 8 lanes a row, four
// steps of rows in flight.  Bound by the bytes moved, three per channel, and the arithmetic: 8 x 131072 rows
// of 128 channels 75 us, 5.4 TB/s (with a division per component 95 us; with a channel a lane, a row after the other
// and bytes stored one by one 265 us).
constexpr int kQuantWaves = kQuantThreads / 64;

__global__ __launch_bounds__(kQuantThreads) void k_quantize(const uint16_t* keys, int8_t* keys8, const float* kscale,
                                                            const int32_t* perm, float* keps, size_t cap0,
                                                            size_t cap1, int node_first, int nodes, int bf, int D) {
    constexpr int U = 4;
    const int t = blockIdx.y, lane = threadIdx.x & 63;
    const int i_node = blockIdx.x * kQuantWaves + (int)(threadIdx.x >> 6);
    if (i_node >= nodes) return;  // (the whole wave; no barrier below)
    const int node = node_first + i_node;
    const int cpr = D / 8, groups = 64 / cpr, rg = lane / cpr, c = lane % cpr;
    const size_t base = (size_t)t * cap0;
    float step[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) step[e] = kscale[(size_t)t * D + c * 8 + e];
    float inverse[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) inverse[e] = 1.0f / step[e];
    float worst = 0.0f;
    if (rg < groups)
        for (int i0 = rg; i0 < bf; i0 += groups * U) {
            uint4 raw[U];
            int at[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const size_t slot = (size_t)node * bf + min(i0 + u * groups, bf - 1);
                raw[u] = *reinterpret_cast<const uint4*>(keys + (base + slot) * D + c * 8);
                at[u] = perm[base + slot];
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (i0 + u * groups >= bf) break;
                float f[8];
                unpack<bf16_t>(raw[u], f);
                uint32_t out[2] = {0u, 0u};
                if (at[u] >= 0) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const float v = quotient(f[e], step[e], inverse[e]);
                        const float r = fminf(fmaxf(rintf(v), -127.0f), 127.0f);
                        worst = fmaxf(worst, fabsf(v - r));
                        out[e >> 2] |= ((uint32_t)(int)r & 0xffu) << (8 * (e & 3));
                    }
                }
                const size_t slot = (size_t)node * bf + i0 + u * groups;
                *reinterpret_cast<uint2*>(keys8 + base * D + shadow_index(D, slot, c * 8)) = make_uint2(out[0], out[1]);
            }
        }
    worst = wave_max(worst);
    if (lane == 0) keps[(size_t)t * cap1 + node] = worst;
}

static void quantize_nodes(const HiraTree* tree, int node_first, int nodes, hipStream_t s) {
    hipLaunchKernelGGL(k_quantize, dim3((nodes + kQuantWaves - 1) / kQuantWaves, tree->num_trees), dim3(kQuantThreads), 0, s,
                       reinterpret_cast<const uint16_t*>(tree->keys), tree->keys8, tree->kscale, tree->perm, tree->keps,
                       (size_t)tree->cap[0], (size_t)tree->cap[1], node_first, nodes, tree->bf, tree->dim);
}

int quantize_with(const HiraTree* tree, const float* absmax, int copies, hipStream_t s) {
    const size_t n = (size_t)tree->num_trees * tree->dim;
    hipLaunchKernelGGL(k_step_from_absmax, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, tree->kscale, absmax, copies,
                       tree->dim, n);
    quantize_nodes(tree, 0, tree->size[1], s);
    HIRA_CHECK_LAUNCH("quantize kernel");
    return HIRA_OK;
}

}  // namespace hira

using namespace hira;

/* see include/hira_hip.h */
extern "C" int hira_quantize(const HiraTree* tree, int32_t slot_first, int32_t slot_count,
                             int32_t recompute_scale, void* stream) {
    HIRA_CHECK_ARG(tree != nullptr && tree->layout == HIRA_TILE16_Q8,
                   "hira_quantize needs an index in the layout with an 8-bit shadow");
    HIRA_CHECK_ARG(tree->dtype == HIRA_BF16 && tree->dim % 64 == 0 && tree->dim <= 256 &&
                       tree->num_levels >= 2,
                   "8-bit shadow: bf16 rows of 64, 128, 192 or 256 columns, at least two levels");
    HIRA_CHECK_ARG(tree->keys && tree->perm && tree->keys8 && tree->kscale && tree->keps,
                   "keys / perm / keys8 / kscale / keps missing");
    const int bf = tree->bf;
    HIRA_CHECK_ARG(slot_first >= 0 && slot_count >= 0 && slot_first % bf == 0 && slot_count % bf == 0 &&
                       (int64_t)slot_first + slot_count <= tree->cap[0] &&
                       ((int64_t)slot_first + slot_count) / bf <= tree->cap[1],
                   "slots [%d, +%d): whole level-1 nodes inside the capacity", slot_first, slot_count);
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    const int D = tree->dim, T = tree->num_trees;
    const uint16_t* keys = reinterpret_cast<const uint16_t*>(tree->keys);
    if (recompute_scale) {
        HIRA_CHECK_ARG(slot_first == 0 && slot_count >= tree->size[0],
                       "new steps need the shadow of every key recomputed");
        const int rows = tree->size[0];
        const size_t n = (size_t)T * D;
        int parts = (rows + 1023) / 1024;
        if (parts > 128) parts = 128;
        if (parts < 1) parts = 1;
        hipLaunchKernelGGL(k_zero_f32, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, tree->kscale, n);
        if (rows > 0)
            hipLaunchKernelGGL(k_absmax, dim3(parts, T), dim3(kQuantThreads), 0, s, keys,
                               (size_t)tree->cap[0], rows, D, tree->kscale);
        hipLaunchKernelGGL(k_step_from_absmax, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s,
                           tree->kscale, tree->kscale, 1, D, n);
    }
    if (slot_count == 0) return HIRA_OK;
    quantize_nodes(tree, slot_first / bf, slot_count / bf, s);
    HIRA_CHECK_LAUNCH("quantize kernel");
    return HIRA_OK;
}
