// Element-wise access to key / centre / value rows in either storage type.
#pragma once

#include "search.h"

namespace hira {

template <typename T>
__device__ __forceinline__ float load_elem(const void* base, size_t i);
template <>
__device__ __forceinline__ float load_elem<float>(const void* base, size_t i) {
    return reinterpret_cast<const float*>(base)[i];
}
template <>
__device__ __forceinline__ float load_elem<bf16_t>(const void* base, size_t i) {
    return bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(base)[i]);
}
template <typename T>
__device__ __forceinline__ void store_elem(void* base, size_t i, float v);
template <>
__device__ __forceinline__ void store_elem<float>(void* base, size_t i, float v) {
    reinterpret_cast<float*>(base)[i] = v;
}
template <>
__device__ __forceinline__ void store_elem<bf16_t>(void* base, size_t i, float v) {
    reinterpret_cast<uint16_t*>(base)[i] = f32_to_bf16_bits(v);
}
// a 16-byte chunk, from element i (a multiple of the chunk's elements) on
__device__ __forceinline__ void store_chunk_of(float* to, const float (&v)[4]) {
    *reinterpret_cast<float4*>(to) = make_float4(v[0], v[1], v[2], v[3]);
}
__device__ __forceinline__ void store_chunk_of(uint16_t* to, const float (&v)[8]) {
    *reinterpret_cast<uint4*>(to) = make_uint4(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]), pack_bf16(v[4], v[5]), pack_bf16(v[6], v[7]));
}
template <typename T>
__device__ __forceinline__ void store_chunk(void* base, size_t i, const float (&v)[Elem<T>::kPerChunk]) {
    if constexpr (Elem<T>::kPerChunk == 4) store_chunk_of(reinterpret_cast<float*>(base) + i, v);
    else store_chunk_of(reinterpret_cast<uint16_t*>(base) + i, v);
}
template <typename T>
__device__ __forceinline__ float round_to(float v);
template <>
__device__ __forceinline__ float round_to<float>(float v) {
    return v;
}
template <>
__device__ __forceinline__ float round_to<bf16_t>(float v) {
    return bf16_bits_to_f32(f32_to_bf16_bits(v));
}

}  // namespace hira
