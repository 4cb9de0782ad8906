// Shared device helpers for the gfx950 kernels: 16-byte row chunks, wave64 cross-lane
// reductions, error reporting for the C ABI.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include "../../include/hira_hip.h"

namespace hira {

constexpr int kWave = 64;
constexpr float kLog2e = 1.4426950408889634f;

// ---- error text (thread local, returned by hira_last_error) -------------------------
char* error_buffer();
int fail(int code, const char* fmt, ...);

#define HIRA_CHECK_ARG(cond, ...)                              \
    do {                                                       \
        if (!(cond)) return ::hira::fail(HIRA_EINVAL, __VA_ARGS__); \
    } while (0)

#define HIRA_CHECK_LAUNCH(what)                                                        \
    do {                                                                               \
        hipError_t e_ = hipGetLastError();                                             \
        if (e_ != hipSuccess)                                                          \
            return ::hira::fail(HIRA_ELAUNCH, "%s: %s", what, hipGetErrorString(e_));  \
    } while (0)

// ---- storage types -------------------------------------------------------------------
struct bf16_t {
    uint16_t bits;
};

template <typename T>
struct Elem;
template <>
struct Elem<float> {
    static constexpr int kPerChunk = 4;  // elements in one 16-byte chunk
};
template <>
struct Elem<bf16_t> {
    static constexpr int kPerChunk = 8;
};

__device__ __forceinline__ float bf16_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }

// Round-to-nearest-even fp32 -> bf16 (NaN kept quiet), by the instruction that does two of them: the same bits as by
// shifts and additions for each of the 2^32 numbers, where those take eight instructions each.
__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
    typedef __attribute__((ext_vector_type(2))) float f32x2;
    typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
}
__device__ __forceinline__ uint16_t f32_to_bf16_bits(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }
__device__ __host__ __forceinline__ float bf16_bits_to_f32(uint16_t b) {
    union {
        float f;
        uint32_t u;
    } v;
    v.u = ((uint32_t)b) << 16;
    return v.f;
}

// Unpack one 16-byte chunk into fp32 lanes.
template <typename T>
__device__ __forceinline__ void unpack(const uint4& raw, float (&f)[Elem<T>::kPerChunk]);
template <>
__device__ __forceinline__ void unpack<float>(const uint4& raw, float (&f)[4]) {
    f[0] = __uint_as_float(raw.x);
    f[1] = __uint_as_float(raw.y);
    f[2] = __uint_as_float(raw.z);
    f[3] = __uint_as_float(raw.w);
}
template <>
__device__ __forceinline__ void unpack<bf16_t>(const uint4& raw, float (&f)[8]) {
    f[0] = bf16_lo(raw.x);
    f[1] = bf16_hi(raw.x);
    f[2] = bf16_lo(raw.y);
    f[3] = bf16_hi(raw.y);
    f[4] = bf16_lo(raw.z);
    f[5] = bf16_hi(raw.z);
    f[6] = bf16_lo(raw.w);
    f[7] = bf16_hi(raw.w);
}

// 16-byte load of chunk `ch` of the row that starts at element `row_elems` of `base`.
template <typename T>
__device__ __forceinline__ uint4 load_chunk(const void* base, size_t row_elems, int ch) {
    const T* p = reinterpret_cast<const T*>(base) + row_elems + (size_t)ch * Elem<T>::kPerChunk;
    return *reinterpret_cast<const uint4*>(p);
}

// ---- cross-lane ----------------------------------------------------------------------
// By moves of the data path: __shfl goes through the LDS crossbar, some hundred cycles a step, in chains that
// nothing else fills.  Before and after: attention over 4 trees x 5003 rows of 80 fp32 12.4 -> 11.8 us, 1111 keys of
// 64 bf16 in five levels 12.9 -> 11.2, a decode step of 8 trees x 32768 keys 19.25 -> 18.85.
template <int CTRL, typename V>
__device__ __forceinline__ V dpp_move(V v) {
    static_assert(sizeof(V) == 4, "a lane's register");
    return __builtin_bit_cast(V, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}

// op(mine, lane ^ BIT's) for an op that does not mind the order; whole waves only.  Rows of 16 and halves
// trade places by a swap that leaves both values in either.
template <int BIT, typename V, typename Op>
__device__ __forceinline__ V xor_with(V v, Op op) {
    if constexpr (BIT >= 16) {
        const auto r = BIT == 32 ? __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, v), __builtin_bit_cast(uint32_t, v), false, false)
                                 : __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, v), __builtin_bit_cast(uint32_t, v), false, false);
        return op(__builtin_bit_cast(V, (uint32_t)r[0]), __builtin_bit_cast(V, (uint32_t)r[1]));
    } else if constexpr (BIT == 8) {
        return op(v, dpp_move<0x128>(v));  // row rotated by 8
    } else if constexpr (BIT == 4) {
        return op(v, dpp_move<0x1B>(dpp_move<0x141>(v)));  // halves of a row mirrored, quads mirrored
    } else {
        return op(v, dpp_move<BIT == 2 ? 0x4E : 0xB1>(v));  // quads
    }
}
struct OpSum {
    template <typename V>
    __device__ __forceinline__ V operator()(V a, V b) const { return a + b; }
};
struct OpMax {
    __device__ __forceinline__ float operator()(float a, float b) const { return fmaxf(a, b); }
};
struct OpMin {
    __device__ __forceinline__ int operator()(int a, int b) const { return min(a, b); }
};

// over the lanes that differ in bits FROM .. TO / 2 (a butterfly: lane ^ FROM first), the same in all of them
template <int FROM, int TO, typename V, typename Op>
__device__ __forceinline__ V lanes_fold(V v, Op op) {
    if constexpr (FROM < TO) return lanes_fold<FROM * 2, TO>(xor_with<FROM>(v, op), op);
    else return v;
}

// Sum over each aligned group of LANES consecutive lanes; every lane gets the group sum.
template <int LANES>
__device__ __forceinline__ float group_sum(float v) {
    // (from 4 on a mirror will do: the lanes it pairs hold the same sums as lane ^ 4, lane ^ 8.  16 and 32 by the
    // crossbar: many such sums are under way at once where this is called, and a swap takes three instructions --
    // 8 trees x 32768 rows of 128 fp32 43.8 us, with swaps 44.8)
    if (LANES >= 2) v += dpp_move<0xB1>(v);
    if (LANES >= 4) v += dpp_move<0x4E>(v);
    if (LANES >= 8) v += dpp_move<0x141>(v);
    if (LANES >= 16) v += dpp_move<0x140>(v);
    if (LANES >= 32) v += __shfl_xor(v, 16, 64);
    if (LANES >= 64) v += __shfl_xor(v, 32, 64);
    return v;
}
// over the wave, the additions of the same butterfly
__device__ __forceinline__ float wave_sum(float v) { return lanes_fold<16, 64>(group_sum<16>(v), OpSum{}); }

// sum over each aligned group of `lpr` lanes (uniform), in the order of group_sum<lpr>
__device__ __forceinline__ float group_sum_of(float v, int lpr) {
    if (lpr >= 2) v += dpp_move<0xB1>(v);
    if (lpr >= 4) v += dpp_move<0x4E>(v);
    if (lpr >= 8) v += dpp_move<0x141>(v);
    if (lpr >= 16) v += dpp_move<0x140>(v);
    if (lpr >= 32) v = xor_with<16>(v, OpSum{});
    if (lpr >= 64) v = xor_with<32>(v, OpSum{});
    return v;
}

// Reductions ACROSS the 64/LANES groups of a wave (lanes with equal lane % LANES).
template <int LANES>
__device__ __forceinline__ float cross_group_max(float v) {
    return lanes_fold<LANES, 64>(v, OpMax{});
}
template <int LANES>
__device__ __forceinline__ float cross_group_sum(float v) {
    return lanes_fold<LANES, 64>(v, OpSum{});
}
// the same for a number of lanes that the compiler does not know (uniform, a power of two)
template <typename V, typename Op>
__device__ __forceinline__ V cross_group(V v, int lanes, Op op) {
    if (lanes <= 1) v = xor_with<1>(v, op);
    if (lanes <= 2) v = xor_with<2>(v, op);
    if (lanes <= 4) v = xor_with<4>(v, op);
    if (lanes <= 8) v = xor_with<8>(v, op);
    if (lanes <= 16) v = xor_with<16>(v, op);
    if (lanes <= 32) v = xor_with<32>(v, op);
    return v;
}

__device__ __forceinline__ float wave_max(float v) { return lanes_fold<1, 64>(v, OpMax{}); }
__device__ __forceinline__ int wave_min(int v) { return lanes_fold<1, 64>(v, OpMin{}); }

__device__ __forceinline__ int lane_id() { return threadIdx.x & 63; }

}  // namespace hira
