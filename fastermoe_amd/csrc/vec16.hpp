// 16-byte vectors of an element type and their conversion from and to float (device code).
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

namespace fmoe {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

template <typename T> struct Vec;  // 16 bytes of T <-> floats
template <> struct Vec<float> {
    static constexpr int N = 4;
    __device__ static void unpack(const u32x4 &v, float (&f)[8]) {
#pragma unroll
        for (int i = 0; i < 4; ++i) f[i] = __uint_as_float(v[i]);
    }
    __device__ static u32x4 pack(const float (&f)[8]) {
        return u32x4{__float_as_uint(f[0]), __float_as_uint(f[1]), __float_as_uint(f[2]), __float_as_uint(f[3])};
    }
};
template <> struct Vec<__bf16> {
    static constexpr int N = 8;
    __device__ static void unpack(const u32x4 &v, float (&f)[8]) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            f[2 * i] = __uint_as_float(v[i] << 16);
            f[2 * i + 1] = __uint_as_float(v[i] & 0xffff0000u);
        }
    }
    __device__ static u32x4 pack(const float (&f)[8]) {
        u32x4 r;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const __bf16 lo = (__bf16)f[2 * i], hi = (__bf16)f[2 * i + 1];
            r[i] = (uint32_t)__builtin_bit_cast(uint16_t, lo) | ((uint32_t)__builtin_bit_cast(uint16_t, hi) << 16);
        }
        return r;
    }
};
template <> struct Vec<_Float16> {
    static constexpr int N = 8;
    __device__ static void unpack(const u32x4 &v, float (&f)[8]) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            f[2 * i] = (float)__builtin_bit_cast(_Float16, (uint16_t)(v[i] & 0xffffu));
            f[2 * i + 1] = (float)__builtin_bit_cast(_Float16, (uint16_t)(v[i] >> 16));
        }
    }
    __device__ static u32x4 pack(const float (&f)[8]) {
        u32x4 r;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const _Float16 lo = (_Float16)f[2 * i], hi = (_Float16)f[2 * i + 1];
            r[i] = (uint32_t)__builtin_bit_cast(uint16_t, lo) | ((uint32_t)__builtin_bit_cast(uint16_t, hi) << 16);
        }
        return r;
    }
};

// The first n of the 16-bit elements at p, which may lie anywhere, zeros after them (8 <= n: all eight); nothing past them is read.
template <typename T> __device__ __forceinline__ u32x4 load_some(const T *p, int64_t n) {
    static_assert(sizeof(T) == 2, "16-bit element types");
    if (n >= 8) {
        u32x4 v;
        __builtin_memcpy(&v, p, 16);
        return v;
    }
    alignas(16) uint16_t e[8] = {};
#pragma unroll
    for (int j = 0; j < 7; ++j)
        if (j < n) e[j] = ((const uint16_t *)p)[j];
    return __builtin_bit_cast(u32x4, e);
}
template <typename T> __device__ __forceinline__ void store_some(T *p, const u32x4 &v, int64_t n) {
    static_assert(sizeof(T) == 2, "16-bit element types");
    if (n >= 8) {
        __builtin_memcpy(p, &v, 16);
        return;
    }
    alignas(16) uint16_t e[8];
    __builtin_memcpy(e, &v, 16);
#pragma unroll
    for (int j = 0; j < 7; ++j)
        if (j < n) ((uint16_t *)p)[j] = e[j];
}

}  // namespace fmoe
