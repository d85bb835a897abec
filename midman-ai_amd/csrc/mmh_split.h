// f32 values as exact sums of three bf16 values, for products on the bf16
// matrix cores (gemm_split.hip says why and how exact; attention_split.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <utility>

namespace mmh {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// Calls f(integral_constant<int, i>) for i = 0..n-1, so that i is a
// compile-time constant in each call (register-slot indices stay static).
template <class F, int... Is>
__device__ __forceinline__ void unroll_seq(F &&f, std::integer_sequence<int, Is...>) {
    (f(std::integral_constant<int, Is>{}), ...);
}

// Operands are lifted by 2^24 before they are split: the lowest bit of any f32
// is then at least 2^-125, so every piece of every value lies in bf16's normal
// range, the smallest subnormal's too. Only values from 2^104 on do not fit
// (they leave infinities), and a product's sums are 2^48 times the true ones.
constexpr float kLift = 0x1p24f, kUnlift = 0x1p-24f, kUnlift2 = 0x1p-48f;

// (bf16(x), bf16(y)), rounded to nearest even. The empty assembly hides where r
// comes from: without it the compiler converts x a second time on its own for
// the remainder. The instruction itself stays the compiler's, which has to keep
// two wait states between it and a matrix instruction that reads r.
__device__ __forceinline__ uint32_t pack_bf16(float x, float y) {
    typedef float floatx2 __attribute__((ext_vector_type(2)));
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    uint32_t r = __builtin_bit_cast(uint32_t, __builtin_convertvector((floatx2){x, y}, bf16x2));
    asm("" : "+v"(r));
    return r;
}

// E values of consecutive k as three pieces of E bf16 each.
template <int E>
__device__ __forceinline__ void split_values(const float (&v)[E], uint32_t (&o)[3][E / 2]) {
#pragma unroll
    for (int i = 0; i < E / 2; ++i) {
        const float x = v[2 * i], y = v[2 * i + 1];
        const uint32_t h = pack_bf16(x, y);
        const float rx = x - __uint_as_float(h << 16), ry = y - __uint_as_float(h & 0xffff0000u);
        const uint32_t m = pack_bf16(rx, ry);
        const float sx = rx - __uint_as_float(m << 16), sy = ry - __uint_as_float(m & 0xffff0000u);
        o[0][i] = h;
        o[1][i] = m;
        o[2][i] = pack_bf16(sx, sy);
    }
}
template <int E>
__device__ __forceinline__ void lift_and_split(const float (&v)[E], uint32_t (&o)[3][E / 2]) {
    float x[E];
#pragma unroll
    for (int e = 0; e < E; ++e) x[e] = v[e] * kLift;
    split_values(x, o);
}

// An address that is the same in every lane, in scalar registers.
__device__ __forceinline__ const float *uniform(const float *ptr) {
    const uint64_t a = reinterpret_cast<uint64_t>(ptr);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)a);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32));
    return reinterpret_cast<const float *>((uint64_t)hi << 32 | lo);
}

}  // namespace mmh
