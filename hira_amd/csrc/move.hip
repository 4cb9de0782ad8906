// Rows and whole arrays moved in one launch each: what the cache layer and the indexer do beside
// the search and would otherwise do with a tensor operation per array.
//   hira_enqueue       the new keys and values of a decode step into the queue
//   hira_replace_rows  a few rows of every tree's key sample replaced by new keys
//   hira_fill_arrays   the level arrays of an index into larger ones, or their padding alone
// All three are bound by their launch at the sizes of a decode step (a few KiB), so what counts is
// that there is one of them: a token's two row copies were two launches (3.0 us each on the GPU
// and about as much on the host), growing an index of three levels was eighteen.
#include "common.hip.h"

namespace hira {

constexpr int kMoveThreads = 256;

__global__ __launch_bounds__(kMoveThreads) void k_enqueue(uint4* qk, uint4* qv, int cap, int at,
                                                          int m, int kc, int vc, const uint4* k,
                                                          const uint4* v, int total) {
    const int i = blockIdx.x * kMoveThreads + threadIdx.x;
    if (i >= total) return;
    const int per = kc + vc, row = i / per, c = i - row * per;  // row: tree * m + new row
    const int t = row / m, r = row - t * m;
    const size_t dst = (size_t)t * cap + at + r;
    if (c < kc) qk[dst * kc + c] = k[(size_t)row * kc + c];
    else qv[dst * vc + (c - kc)] = v[(size_t)row * vc + (c - kc)];
}

// (replaced rows travel with the kernel's arguments: a few for a token, many for a whole sample)
template <int N>
struct RowPairs {
    int32_t slot[N], from[N];
};
constexpr int kFewPairs = 32, kManyPairs = 448;

template <int N>
__global__ __launch_bounds__(kMoveThreads) void k_replace_rows(uint4* rows, int chunks,
                                                               int rows_per_tree, const uint4* from,
                                                               int from_stride, const RowPairs<N> pairs,
                                                               int n, int total) {
    const int i = blockIdx.x * kMoveThreads + threadIdx.x;
    if (i >= total) return;
    const int row = i / chunks, c = i - row * chunks;  // row: tree * n + pair
    const int t = row / n, p = row - t * n;
    rows[((size_t)t * rows_per_tree + pairs.slot[p]) * chunks + c] =
        from[((size_t)t * from_stride + pairs.from[p]) * chunks + c];
}

// Every array is walked as one stretch of num_trees x stride bytes, kStretch a workgroup: bytes
// below `copy` of a tree come from the source, bytes from `from` on become the fill word, what
// lies between is left alone.  Word = 16 bytes where an array's numbers allow it, else 4.
constexpr int kMaxArrays = 32;
constexpr int kStretch = 32 * 1024;
struct ArrayList {
    struct One {
        char* dst;
        const char* src;
        unsigned long long dst_stride, src_stride, copy, from;
        uint32_t fill;
        int32_t wide;
        uint32_t first_block;  // workgroups of the arrays before this one
        uint32_t pad_;
    } a[kMaxArrays];
    int32_t n;
};

template <typename W>
__device__ __forceinline__ void move_stretch(const ArrayList::One& a, unsigned long long begin,
                                             unsigned long long end, W fill) {
    // (one division a thread; from then on the place inside the tree is carried along)
    unsigned long long o = begin + (unsigned long long)threadIdx.x * sizeof(W);
    unsigned long long t = o / a.dst_stride, r = o - t * a.dst_stride;
    for (; o < end; o += kMoveThreads * sizeof(W)) {
        while (r >= a.dst_stride) {
            r -= a.dst_stride;
            ++t;
        }
        if (r < a.copy)
            *reinterpret_cast<W*>(a.dst + o) = *reinterpret_cast<const W*>(a.src + t * a.src_stride + r);
        else if (r >= a.from)
            *reinterpret_cast<W*>(a.dst + o) = fill;
        r += kMoveThreads * sizeof(W);
    }
}

__global__ __launch_bounds__(kMoveThreads) void k_fill_arrays(const ArrayList list, int trees) {
    int i = 0;
    while (i + 1 < list.n && list.a[i + 1].first_block <= blockIdx.x) ++i;  // uniform
    const ArrayList::One& a = list.a[i];
    const unsigned long long begin = (unsigned long long)(blockIdx.x - a.first_block) * kStretch;
    const unsigned long long all = a.dst_stride * (unsigned long long)trees;
    const unsigned long long end = begin + kStretch < all ? begin + kStretch : all;
    if (a.wide) move_stretch<uint4>(a, begin, end, make_uint4(a.fill, a.fill, a.fill, a.fill));
    else move_stretch<uint32_t>(a, begin, end, a.fill);
}

}  // namespace hira

using namespace hira;

static int row_chunks(int32_t dtype, int32_t width) {  // 16-byte chunks of a row; -1: not whole ones
    const int bytes = width * (dtype == HIRA_F32 ? 4 : 2);
    return width >= 0 && bytes % 16 == 0 ? bytes / 16 : -1;
}

static bool aligned16(const void* a, const void* b) {  // (the kernels move 16 bytes a lane)
    return (((uintptr_t)a | (uintptr_t)b) & 15) == 0;
}

/* see include/hira_hip.h */
extern "C" int hira_enqueue(void* queue_keys, void* queue_values, int32_t dtype, int32_t num_trees,
                            int32_t cap, int32_t at, int32_t m, int32_t dim, int32_t vdim,
                            const void* new_keys, const void* new_values, void* stream) {
    HIRA_CHECK_ARG(dtype == HIRA_F32 || dtype == HIRA_BF16, "hira_enqueue: dtype %d", dtype);
    const int kc = row_chunks(dtype, dim), vc = row_chunks(dtype, vdim);
    HIRA_CHECK_ARG(kc >= 1 && vc >= 0, "hira_enqueue: dim %d / vdim %d: rows must be a multiple of 16 bytes",
                   dim, vdim);
    HIRA_CHECK_ARG(num_trees >= 1 && m >= 0 && at >= 0 && (int64_t)at + m <= cap,
                   "hira_enqueue: rows %d .. %d of %d", at, at + m, cap);
    HIRA_CHECK_ARG(queue_keys && new_keys && (vc == 0 || (queue_values && new_values)),
                   "hira_enqueue: null argument");
    HIRA_CHECK_ARG(aligned16(queue_keys, new_keys) && (vc == 0 || aligned16(queue_values, new_values)),
                   "hira_enqueue: rows must be 16-byte aligned");
    const int64_t total = (int64_t)num_trees * m * (kc + vc);
    HIRA_CHECK_ARG(total < (int64_t)1 << 31, "hira_enqueue: too many rows at once");
    if (total == 0) return HIRA_OK;
    hipLaunchKernelGGL(k_enqueue, dim3((unsigned)((total + kMoveThreads - 1) / kMoveThreads)),
                       dim3(kMoveThreads), 0, reinterpret_cast<hipStream_t>(stream),
                       static_cast<uint4*>(queue_keys), static_cast<uint4*>(queue_values), cap, at, m, kc,
                       vc, static_cast<const uint4*>(new_keys), static_cast<const uint4*>(new_values),
                       (int)total);
    HIRA_CHECK_LAUNCH("hira_enqueue");
    return HIRA_OK;
}

template <int N>
static void replace_some(void* rows, int chunks, int num_trees, int rows_per_tree, const void* from,
                         int from_stride, const int32_t* slot_host, const int32_t* from_host, int c,
                         void* stream) {
    RowPairs<N> pairs;
    memset(&pairs, 0, sizeof(pairs));
    memcpy(pairs.slot, slot_host, c * sizeof(int32_t));
    memcpy(pairs.from, from_host, c * sizeof(int32_t));
    const int total = num_trees * c * chunks;
    hipLaunchKernelGGL((k_replace_rows<N>), dim3((total + kMoveThreads - 1) / kMoveThreads), dim3(kMoveThreads), 0,
                       reinterpret_cast<hipStream_t>(stream), static_cast<uint4*>(rows), chunks, rows_per_tree,
                       static_cast<const uint4*>(from), from_stride, pairs, c, total);
}

/* see include/hira_hip.h */
extern "C" int hira_replace_rows(void* rows, int32_t dtype, int32_t dim, int32_t num_trees,
                                 int32_t rows_per_tree, const void* from, int32_t from_rows,
                                 int32_t from_stride, const int32_t* slot_host, const int32_t* from_host,
                                 int32_t n, void* stream) {
    HIRA_CHECK_ARG(dtype == HIRA_F32 || dtype == HIRA_BF16, "hira_replace_rows: dtype %d", dtype);
    const int chunks = row_chunks(dtype, dim);
    HIRA_CHECK_ARG(chunks >= 1, "hira_replace_rows: dim %d: rows must be a multiple of 16 bytes", dim);
    HIRA_CHECK_ARG(num_trees >= 1 && n >= 0 && from_rows <= from_stride, "hira_replace_rows: bad counts");
    HIRA_CHECK_ARG(n == 0 || (rows && from && slot_host && from_host), "hira_replace_rows: null argument");
    HIRA_CHECK_ARG(n == 0 || aligned16(rows, from), "hira_replace_rows: rows must be 16-byte aligned");
    for (int i = 0; i < n; ++i)
        HIRA_CHECK_ARG(slot_host[i] >= 0 && slot_host[i] < rows_per_tree && from_host[i] >= 0 &&
                           from_host[i] < from_rows,
                       "hira_replace_rows: row %d from %d", slot_host[i], from_host[i]);
    HIRA_CHECK_ARG((int64_t)num_trees * kManyPairs * chunks < (int64_t)1 << 31, "hira_replace_rows: too many trees");
    for (int i0 = 0; i0 < n;) {
        const int left = n - i0;
        if (left <= kFewPairs)
            replace_some<kFewPairs>(rows, chunks, num_trees, rows_per_tree, from, from_stride, slot_host + i0,
                                    from_host + i0, left, stream);
        else
            replace_some<kManyPairs>(rows, chunks, num_trees, rows_per_tree, from, from_stride, slot_host + i0,
                                     from_host + i0, left < kManyPairs ? left : kManyPairs, stream);
        i0 += left <= kFewPairs ? left : kManyPairs;
    }
    HIRA_CHECK_LAUNCH("hira_replace_rows");
    return HIRA_OK;
}

/* see include/hira_hip.h */
extern "C" int hira_fill_arrays(const HiraArray* arrays_host, int32_t n, int32_t num_trees, void* stream) {
    HIRA_CHECK_ARG(n >= 0 && n <= kMaxArrays && num_trees >= 1 && (n == 0 || arrays_host),
                   "hira_fill_arrays: %d arrays (at most %d) of %d trees", n, kMaxArrays, num_trees);
    ArrayList list;
    memset(&list, 0, sizeof(list));
    uint64_t blocks = 0;
    for (int i = 0; i < n; ++i) {
        const HiraArray& h = arrays_host[i];
        HIRA_CHECK_ARG(h.dst && h.dst_stride > 0 && h.copy_bytes >= 0 && h.fill_from >= h.copy_bytes &&
                           h.copy_bytes <= h.dst_stride,
                       "hira_fill_arrays: array %d", i);
        HIRA_CHECK_ARG(h.copy_bytes == 0 || (h.src && h.copy_bytes <= h.src_stride),
                       "hira_fill_arrays: array %d copies %lld bytes of rows of %lld", i,
                       (long long)h.copy_bytes, (long long)h.src_stride);
        const uint64_t all = (uint64_t)h.dst | (uint64_t)h.src | (uint64_t)h.dst_stride |
                             (uint64_t)h.src_stride | (uint64_t)h.copy_bytes | (uint64_t)h.fill_from;
        HIRA_CHECK_ARG(all % 4 == 0, "hira_fill_arrays: array %d is not made of whole words", i);
        ArrayList::One& o = list.a[list.n++];
        o.dst = static_cast<char*>(h.dst);
        o.src = static_cast<const char*>(h.src);
        o.dst_stride = (uint64_t)h.dst_stride;
        o.src_stride = (uint64_t)h.src_stride;
        o.copy = (uint64_t)h.copy_bytes;
        o.from = (uint64_t)h.fill_from;
        o.fill = h.fill;
        o.wide = all % 16 == 0;
        o.first_block = (uint32_t)blocks;
        blocks += ((uint64_t)h.dst_stride * num_trees + kStretch - 1) / kStretch;
    }
    HIRA_CHECK_ARG(blocks < (uint64_t)1 << 31, "hira_fill_arrays: arrays too large");
    if (blocks == 0) return HIRA_OK;
    hipLaunchKernelGGL(k_fill_arrays, dim3((unsigned)blocks), dim3(kMoveThreads), 0,
                       reinterpret_cast<hipStream_t>(stream), list, num_trees);
    HIRA_CHECK_LAUNCH("hira_fill_arrays");
    return HIRA_OK;
}
