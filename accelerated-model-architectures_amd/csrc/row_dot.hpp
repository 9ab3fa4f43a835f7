// <a, b> of two rows by one wave: what the router weights' gradient is made of, in the same order wherever it is computed.
#pragma once

#include "common.hpp"

// the whole sum in every lane; two 16-byte chunks of each row in flight per lane; `a` is read once, `b` by k waves
template <typename ET> __device__ __forceinline__ float row_dot(const void *a, const void *b, int H, int lane) {
    const uint16_t *a_row = (const uint16_t *)a, *b_row = (const uint16_t *)b;
    float acc = 0.f;
    auto dot = [&](const u32x4 u, const u32x4 v) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            acc += Elem<ET>::lo(u[q]) * Elem<ET>::lo(v[q]);
            acc += Elem<ET>::hi(u[q]) * Elem<ET>::hi(v[q]);
        }
    };
    auto once = [](const uint16_t *p) { return __builtin_nontemporal_load((const u32x4 *)p); };
    int c = lane * 8;
    for (; c + WAVE * 8 < H; c += 2 * WAVE * 8) {
        const u32x4 a0 = once(a_row + c), a1 = once(a_row + c + WAVE * 8);
        const u32x4 b0 = *(const u32x4 *)(b_row + c), b1 = *(const u32x4 *)(b_row + c + WAVE * 8);
        dot(a0, b0);
        dot(a1, b1);
    }
    if (c < H) dot(once(a_row + c), *(const u32x4 *)(b_row + c));
#pragma unroll
    for (int d = WAVE / 2; d > 0; d >>= 1) acc += __shfl_xor(acc, d);
    return acc;
}

template <> __device__ __forceinline__ float row_dot<float>(const void *a, const void *b, int H, int lane) {
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    float acc = 0.f;
    for (int c = lane * 4; c < H; c += 4 * WAVE) {
        const f32x4 u = *(const f32x4 *)((const float *)a + c), v = *(const f32x4 *)((const float *)b + c);
        acc += u[0] * v[0] + u[1] * v[1] + u[2] * v[2] + u[3] * v[3];
    }
#pragma unroll
    for (int d = WAVE / 2; d > 0; d >>= 1) acc += __shfl_xor(acc, d);
    return acc;
}
