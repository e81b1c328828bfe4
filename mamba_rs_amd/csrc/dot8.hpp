#pragma once
#include "common.hpp"

namespace mrs {

// 8 products of a 16-byte pair of operand chunks, f32 accumulate (v_dot2_f32_bf16 / v_dot2_f32_f16)
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
template <typename T> struct Dot2;
template <> struct Dot2<bf16_t> {
    __device__ static __forceinline__ float f(uint32_t a, uint32_t b, float c) {
        return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(v2bf, a), __builtin_bit_cast(v2bf, b), c, false);
    }
};
template <> struct Dot2<f16_t> {
    __device__ static __forceinline__ float f(uint32_t a, uint32_t b, float c) {
        return __builtin_amdgcn_fdot2(__builtin_bit_cast(v2h, a), __builtin_bit_cast(v2h, b), c, false);
    }
};
// the products of one 16-byte piece of each operand: 8 elements of a 16-bit type (four v_dot2), 4 of f32
template <typename T> __device__ __forceinline__ float dot8(uint4 a, uint4 b, float c) {
    if constexpr (sizeof(T) == 4) {
        c = fmaf(__uint_as_float(a.x), __uint_as_float(b.x), c); c = fmaf(__uint_as_float(a.y), __uint_as_float(b.y), c);
        c = fmaf(__uint_as_float(a.z), __uint_as_float(b.z), c);
        return fmaf(__uint_as_float(a.w), __uint_as_float(b.w), c);
    } else {
        c = Dot2<T>::f(a.x, b.x, c); c = Dot2<T>::f(a.y, b.y, c); c = Dot2<T>::f(a.z, b.z, c);
        return Dot2<T>::f(a.w, b.w, c);
    }
}

}  // namespace mrs
