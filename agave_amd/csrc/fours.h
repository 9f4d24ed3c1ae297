// Four neighbouring elements of a row as floats, for the 32-bit kernels.
#pragma once
#include "common.h"

typedef float f32x4_t __attribute__((ext_vector_type(4)));

// Elements k .. k+3 of a row; what lies at or behind K is 0.  VEC: K is a multiple of 4 and every row is
// aligned to four elements, so the four are there or not together.
template <bool VEC, typename T> __device__ __forceinline__ f32x4_t ld4(const T* row, int k, int K);
template <> __device__ __forceinline__ f32x4_t ld4<true, float>(const float* row, int k, int K) {
    return k < K ? *(const f32x4_t*)(row + k) : f32x4_t{0.f, 0.f, 0.f, 0.f};
}
template <> __device__ __forceinline__ f32x4_t ld4<true, bf16>(const bf16* row, int k, int K) {
    if (k >= K) return f32x4_t{0.f, 0.f, 0.f, 0.f};
    const uint2 u = *(const uint2*)(row + k);
    return f32x4_t{__builtin_bit_cast(float, u.x << 16), __builtin_bit_cast(float, u.x & 0xffff0000u),
                   __builtin_bit_cast(float, u.y << 16), __builtin_bit_cast(float, u.y & 0xffff0000u)};
}
template <> __device__ __forceinline__ f32x4_t ld4<false, float>(const float* row, int k, int K) {
    f32x4_t v;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = k + e < K ? row[k + e] : 0.f;
    return v;
}
template <> __device__ __forceinline__ f32x4_t ld4<false, bf16>(const bf16* row, int k, int K) {
    f32x4_t v;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = k + e < K ? bf16_to_f32(row[k + e]) : 0.f;
    return v;
}
