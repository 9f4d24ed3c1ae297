// Neighbouring elements of a row as floats.
#pragma once
#include "common.h"

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

// V neighbours, one or four (aligned to as many), from memory and to it.
template <int V, typename T> __device__ __forceinline__ void load_near(const T* p, float* v) {
    static_assert(V == 1 || V == 4, "one or four");
    if constexpr (V == 4) {
        const f32x4_t u = ld4<true>(p, 0, 4);
        v[0] = u[0]; v[1] = u[1]; v[2] = u[2]; v[3] = u[3];
    } else {
        v[0] = ld(p);
    }
}
template <int V> __device__ __forceinline__ void store_near(float* p, const float* v) {
    if constexpr (V == 4) *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
    else *p = v[0];
}
template <int V> __device__ __forceinline__ void store_near(bf16* p, const float* v) {
    if constexpr (V == 4) *reinterpret_cast<uint2*>(p) = make_uint2(f32x2_to_bf16x2(v[0], v[1]), f32x2_to_bf16x2(v[2], v[3]));
    else *p = f32_to_bf16(v[0]);
}
