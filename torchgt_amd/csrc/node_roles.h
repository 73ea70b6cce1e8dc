// What the fused per-node kernels of the two layer families share (node_layer.hip: Graphormer, gt_layer.hip: GT): weights on
// their way to LDS, the two roles of the backward kernels, their partial sums and how they are launched.
#pragma once
#include "node_tile.h"
#include <algorithm>

namespace tgt {
namespace {

constexpr int kVec = 64;      // floats per parameter vector

// N 16-byte vectors from global memory to LDS by all THREADS threads of a workgroup, every load issued before the first write
template <int N, int THREADS> __device__ __forceinline__ void copy_vecs(vec16* dst, const vec16* __restrict__ src) {
    constexpr int R = (N + THREADS - 1) / THREADS;
    vec16 v[R];
#pragma unroll
    for (int i = 0; i < R; ++i) {
        const int at = threadIdx.x + i * THREADS;
        if (N % THREADS == 0 || at < N) v[i] = src[at];
    }
#pragma unroll
    for (int i = 0; i < R; ++i) {
        const int at = threadIdx.x + i * THREADS;
        if (N % THREADS == 0 || at < N) dst[at] = v[i];
    }
}

// A packed weight on its way from memory to LDS through the registers of the four block waves
template <int N> struct WeightsAhead {
    static_assert(N % 256 == 0, "whole vectors per thread");
    vec16 v[N / 256];
    __device__ __forceinline__ void fetch(const vec16* __restrict__ src) {
#pragma unroll
        for (int i = 0; i < N / 256; ++i) v[i] = src[(threadIdx.x & 255) + i * 256];
    }
    __device__ __forceinline__ void put(vec16* dst) const {
#pragma unroll
        for (int i = 0; i < N / 256; ++i) dst[(threadIdx.x & 255) + i * 256] = v[i];
    }
    // the weight at hand to LDS, the next one asked for, and the barrier that says so
    __device__ __forceinline__ void hand_over(vec16* dst, const vec16* __restrict__ src) {
        put(dst);
        fetch(src);
        __syncthreads();
    }
};

// ---- backward: shared pieces ----------------------------------------------------------------------------------------------
// Eight waves, two roles, one of each per SIMD: waves 0 .. 3 ("chain") carry 32 nodes each through the chain of products and
// LayerNorms and leave the planes of both operands of every weight gradient in LDS; waves 4 .. 7 ("blocks") keep one 32 x 32
// block of every weight gradient in registers and add the products over the 128 nodes while the chain is in its next step,
// and hand the chain its packed weights one at a time.  So the matrix work of one role runs beside the vector work of the
// other, and neither has to hold the other's registers (with all waves in both roles, 16 KB of accumulators per wave next to
// the tiles spilled: 106 us for k_node_bwd_post and 55 us for k_node_bwd_pre at 64 K nodes in float32).
constexpr int kChainNodes = 128, kBwdThreads = 512;

template <typename T, int NV = 5> struct BwdLds {
    static constexpr int P = Num<T>::P;
    static constexpr int kW = 2 * P * kPlaneBytes, kStage = kW + kFragVecs<P> * 16, kVecs = kStage + 4 * RowShape<T>::kVecs * 16;
    static constexpr int kBytes = kVecs + NV * kVec * 4;      // NV: parameter vectors
};

// The workgroup's sums to its partial: NM 64 x 64 blocks (registers of the block waves), then NV vectors of 64 (a register
// of each chain wave; added through LDS).
template <int NM, int NV> __device__ __forceinline__ void write_partial(float* __restrict__ mine, const float16_t (&acc)[NM], const float (&col)[NV], float* buf, int wave, int lane) {
    __syncthreads();
    if (wave < 4) {
#pragma unroll
        for (int c = 0; c < NV; ++c) buf[(wave * NV + c) * 64 + lane] = col[c];
    } else {
        const int q = wave - 4, h = lane >> 5;
#pragma unroll
        for (int j = 0; j < NM; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) mine[j * 4096 + (32 * (q >> 1) + 8 * (r >> 2) + 4 * h + (r & 3)) * 64 + 32 * (q & 1) + (lane & 31)] = acc[j][r];
    }
    __syncthreads();
    for (int i = threadIdx.x; i < NV * 64; i += kBwdThreads) mine[NM * 4096 + i] = (buf[i] + buf[NV * 64 + i]) + (buf[2 * NV * 64 + i] + buf[3 * NV * 64 + i]);
}

// Per head of a node (1 / (Z + 1e-6), da . a): what the sparse attention's backward begins with.  da, a: the lane's half of the node.
template <typename T> __device__ __forceinline__ void put_node_side(const Tile& da, const Tile& a, const float* __restrict__ Z0, float* __restrict__ nd0, int heads, int64_t node, int h) {
    float dot[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        dot[k] = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) dot[k] += stored(da.get(8 * k + i), (const T*)nullptr) * a.get(8 * k + i);
    }
    const float* Z = Z0 + node * heads;      // 8, 4 or 2 heads: one, two or four groups of 8 features each
    float2* nd = reinterpret_cast<float2*>(nd0) + node * heads;
    if (heads == 8) {
        const float4 z = *reinterpret_cast<const float4*>(Z + 4 * h);
        float4* o = reinterpret_cast<float4*>(nd + 4 * h);
        o[0] = make_float4(1.f / (z.x + 1e-6f), dot[0], 1.f / (z.y + 1e-6f), dot[1]);
        o[1] = make_float4(1.f / (z.z + 1e-6f), dot[2], 1.f / (z.w + 1e-6f), dot[3]);
    } else if (heads == 4) {
        const float2 z = *reinterpret_cast<const float2*>(Z + 2 * h);
        *reinterpret_cast<float4*>(nd + 2 * h) = make_float4(1.f / (z.x + 1e-6f), dot[0] + dot[1], 1.f / (z.y + 1e-6f), dot[2] + dot[3]);
    } else {
        nd[h] = make_float2(1.f / (Z[h] + 1e-6f), dot[0] + dot[1] + (dot[2] + dot[3]));
    }
}

int bad(const char* who, const char* what) { set_error("%s: %s", who, what); return TGT_ERR_INVALID_ARG; }
// a workgroup of `waves` waves per CU (LDS), fewer when there is less work
int grid_for(int64_t rows, int waves) { return (int)std::max<int64_t>(1, std::min<int64_t>(num_cus(), ((rows + 31) / 32 + waves - 1) / waves)); }

template <typename... Args> int launch(void (*kernel)(Args...), std::atomic<uint64_t>& done, int grid, int threads, int lds, hipStream_t st, Args... args) {
    if (int rc = allow_lds(reinterpret_cast<const void*>(kernel), lds, done)) return rc;
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(threads), lds, st, args...);
    TGT_HIP_CHECK(hipGetLastError());
    return TGT_OK;
}


}  // namespace
}  // namespace tgt
