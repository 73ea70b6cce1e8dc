// What the dense attention kernels on bf16 tensors share (dense_attn.hip, dense_row0.hip): elements, dot products of a head's row,
// sums over a wave.
#pragma once
#include "common.h"

namespace tgt {

struct dbf16 { uint16_t x; };

__device__ __forceinline__ short f2bf(float f) {
    const __bf16 b = static_cast<__bf16>(f);
    return __builtin_bit_cast(short, b);
}
__device__ __forceinline__ float bf2f(short s) { return __uint_as_float(((uint32_t)(uint16_t)s) << 16); }
__device__ __forceinline__ float ld1(const float* p) { return *p; }
__device__ __forceinline__ float ld1(const dbf16* p) { return __uint_as_float(((uint32_t)p->x) << 16); }
__device__ __forceinline__ void st1(float* p, float v) { *p = v; }
__device__ __forceinline__ void st1(dbf16* p, float v) { p->x = (uint16_t)f2bf(v); }

__device__ __forceinline__ float round_bf(float x) { return bf2f(f2bf(x)); }
__device__ __forceinline__ float wave_sum(float x) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) x += __shfl_xor(x, off);
    return x;
}
template <int D>
__device__ __forceinline__ float dot_d(const float (&a)[D], const float (&b)[D]) {
    float t = 0.f;
#pragma unroll
    for (int c = 0; c < D; ++c) t = fmaf(a[c], b[c], t);
    return t;
}

}  // namespace tgt
