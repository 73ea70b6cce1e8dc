// What the fused per-node kernels of the two layer families share (node_layer.hip: Graphormer, gt_layer.hip: GT): weights on
// their way to LDS, the two roles of the backward kernels, their partial sums and how they are launched.
#pragma once
#include "node_tile.h"
#include <algorithm>

namespace tgt {
namespace {


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

// N 16-byte vectors from global memory straight to LDS, without registers, by a workgroup of any number of whole waves: everything that a kernel begins with
// is asked for before the first wait.  `landed` waits for what this wave has asked for (its rows, too); the others' follows behind a barrier.
// from: the first thread that takes part, of `threads`.
// With loads to registers and writes to LDS one after the other for vectors and weights, and the rows behind them, a launch began with three
// or four memory round trips in a row: 37605 nodes in float32 had their first rows settled after 18 800 of 46 700 cycles of k_node_fwd, now after 8700 of
// 34 900.  Four and five launches of a model, us before / after: float32 4 K nodes 71 / 62, 37605 115 / 107 (GT 125 / 109); bf16 46 / 42, 81 / 77 (GT 72 / 69).
template <int N> __device__ __forceinline__ void copy_direct(int threads, vec16* dst, const vec16* __restrict__ src, int from = 0) {
    const int wave0 = __builtin_amdgcn_readfirstlane(threadIdx.x & ~63) - from, lane = threadIdx.x & 63;
    for (int at = wave0; at < N; at += threads)
        if (N % 64 == 0 || at + lane < N)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src + at + lane), (__attribute__((address_space(3))) void*)(dst + at), 16, 0, 0);
}
template <int N> __device__ __forceinline__ void copy_direct(int threads, float* dst, const float* __restrict__ src, int from = 0) {      // N floats
    copy_direct<N / 4>(threads, reinterpret_cast<vec16*>(dst), reinterpret_cast<const vec16*>(src), from);
}
__device__ __forceinline__ void landed() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Weights in the place of others that everybody has used, seen by everybody
template <int N> __device__ __forceinline__ void replace_weights(int threads, vec16* dst, const vec16* __restrict__ src) {
    __syncthreads();
    copy_direct<N>(threads, dst, src);
    landed();
    __syncthreads();
}

// A packed weight on its way from memory to LDS through the registers of the block waves (T threads, the last of the workgroup)
template <int N, int T = 256> struct WeightsAhead {
    static_assert(N % T == 0 && (T & (T - 1)) == 0, "whole vectors per thread");
    vec16 v[N / T];
    __device__ __forceinline__ void fetch(const vec16* __restrict__ src) {
#pragma unroll
        for (int i = 0; i < N / T; ++i) v[i] = src[(threadIdx.x & (T - 1)) + i * T];
    }
    __device__ __forceinline__ void put(vec16* dst) const {
#pragma unroll
        for (int i = 0; i < N / T; ++i) dst[(threadIdx.x & (T - 1)) + i * T] = v[i];
    }
    // the weight at hand to LDS, the next one asked for, and the barrier that says so
    __device__ __forceinline__ void hand_over(vec16* dst, const vec16* __restrict__ src) {
        put(dst);
        fetch(src);
        __syncthreads();
    }
};

// ---- backward: shared pieces ----------------------------------------------------------------------------------------------
// Two roles per workgroup: the first CN / R waves ("chain") carry R of its CN nodes each through the chain of products and
// LayerNorms and leave the planes of both operands of every weight gradient in LDS; four more ("blocks") keep one 32 x 32
// block of every weight gradient in registers and add the products over the CN nodes while the chain is in its next step,
// and hand the chain its packed weights one at a time.  So the matrix work of one role runs beside the vector work of the
// other, and neither has to hold the other's registers (with all waves in both roles, 16 KB of accumulators per wave next to
// the tiles spilled: 106 us for k_node_bwd_post and 55 us for k_node_bwd_pre at 64 K nodes in float32).
// With six chain waves of 32 rows there are two block waves of two blocks each: eight waves have 256 registers, nine 168, and
// the chain of k_node_bwd_post would put 161 of them to scratch.
constexpr int kBlockWaves = 4;

template <typename T, int R_, int CN_, int NV = 5, int BW = kBlockWaves> struct Bwd {      // NV: parameter vectors, BW: block waves
    static constexpr int R = R_, CN = CN_, P = Num<T>::P, kChain = CN / R, kBlocks = BW, kThreads = (kChain + BW) * 64, kPlane = CN * 128;
    static constexpr int kW = 2 * P * kPlane, kStage = kW + kFragVecs<P> * 16, kVecs = kStage + kChain * RowShape<T, R>::kVecs * 16;
    static constexpr int kBytes = kVecs + NV * kVec * 4;
    static_assert(kChain * 5 * 64 * 4 <= kW, "the column sums of the chain waves meet where the planes were");
};

// The workgroup's sums to its partial: NM 64 x 64 blocks (registers of the block waves), then NV vectors of 64 (a register
// of each chain wave; added through LDS).
template <typename L, int NM, int NV> __device__ __forceinline__ void write_partial(float* __restrict__ mine, const float16_t (&acc)[NM * (4 / L::kBlocks)], const float (&col)[NV], float* buf, int wave, int lane) {
    constexpr int EACH = 4 / L::kBlocks;
    __syncthreads();
    if (wave < L::kChain) {
#pragma unroll
        for (int c = 0; c < NV; ++c) buf[(wave * NV + c) * 64 + lane] = col[c];
    } else {
        const int h = lane >> 5;
#pragma unroll
        for (int j = 0; j < NM * EACH; ++j) {
            const int q = wave - L::kChain + j % EACH * L::kBlocks;
#pragma unroll
            for (int r = 0; r < 16; ++r) mine[j / EACH * 4096 + (32 * (q >> 1) + 8 * (r >> 2) + 4 * h + (r & 3)) * 64 + 32 * (q & 1) + (lane & 31)] = acc[j][r];
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < NV * 64; i += L::kThreads) {
        float t = 0.f;
#pragma unroll
        for (int c = 0; c < L::kChain; c += 2) t += buf[c * NV * 64 + i] + buf[(c + 1) * NV * 64 + i];
        mine[NM * 4096 + i] = t;
    }
}

// Per head of a node (1 / (Z + 1e-6), da . a): what the sparse attention's backward begins with.  da, a: the lane's share of the node.
// All lanes take part (`in`: whether the node exists).
template <typename T, int R> __device__ __forceinline__ void put_node_side(const TileOf<R>& da, const TileOf<R>& a, const float* __restrict__ Z0, float* __restrict__ nd0, int heads, int64_t node, int g, bool in) {
    float dot[R / 8];
#pragma unroll
    for (int k = 0; k < R / 8; ++k) {
        dot[k] = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) dot[k] += stored(da.get(8 * k + i), (const T*)nullptr) * a.get(8 * k + i);
    }
    if constexpr (R == 16) {      // two heads of 32 features: two lanes each
        if (heads == 2) {
            const float t = dot[0] + dot[1];
            const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(t), __float_as_uint(t), false, false);
            dot[0] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
        }
    }
    if (!in) return;
    const float* Z = Z0 + node * heads;      // 8, 4 or 2 heads: one, two or four groups of 8 features each
    float2* nd = reinterpret_cast<float2*>(nd0) + node * heads;
    if constexpr (R == 16) {
        if (heads == 8) {
            const float2 z = *reinterpret_cast<const float2*>(Z + 2 * g);
            *reinterpret_cast<float4*>(nd + 2 * g) = make_float4(1.f / (z.x + 1e-6f), dot[0], 1.f / (z.y + 1e-6f), dot[1]);
        } else if (heads == 4) nd[g] = make_float2(1.f / (Z[g] + 1e-6f), dot[0] + dot[1]);
        else if ((g & 1) == 0) nd[g >> 1] = make_float2(1.f / (Z[g >> 1] + 1e-6f), dot[0]);
    } else if (heads == 8) {
        const float4 z = *reinterpret_cast<const float4*>(Z + 4 * g);
        float4* o = reinterpret_cast<float4*>(nd + 4 * g);
        o[0] = make_float4(1.f / (z.x + 1e-6f), dot[0], 1.f / (z.y + 1e-6f), dot[1]);
        o[1] = make_float4(1.f / (z.z + 1e-6f), dot[2], 1.f / (z.w + 1e-6f), dot[3]);
    } else if (heads == 4) {
        const float2 z = *reinterpret_cast<const float2*>(Z + 2 * g);
        *reinterpret_cast<float4*>(nd + 2 * g) = make_float4(1.f / (z.x + 1e-6f), dot[0] + dot[1], 1.f / (z.y + 1e-6f), dot[2] + dot[3]);
    } else {
        nd[g] = make_float2(1.f / (Z[g] + 1e-6f), dot[0] + dot[1] + (dot[2] + dot[3]));
    }
}

int bad(const char* who, const char* what) { set_error("%s: %s", who, what); return TGT_ERR_INVALID_ARG; }
int64_t groups_of(int64_t rows, int per) { return std::max<int64_t>(1, (rows + per - 1) / per); }
// Forward: a workgroup per CU (LDS), of as many waves as give every CU one, four to `most` (a workgroup copies the weights of a layer to
// LDS: with fewer waves the copies are more traffic than the rows)
int fwd_waves_for(int64_t rows, int per, int most) { return (int)std::min<int64_t>(most, std::max<int64_t>(4, (groups_of(rows, per) + num_cus() - 1) / num_cus())); }
int fwd_grid(int64_t rows, int per, int waves) { return (int)std::min<int64_t>(num_cus(), groups_of(rows, per * waves)); }

// Backward: nodes of a workgroup's group.  64 while there is a CU for every group of 64 (the chain of a workgroup is what such a launch
// takes), 128 with more: the products of a group run while its chain goes on, and a barrier costs the same for 64 nodes and for 128.
// In between the last round decides: float32 takes about 1.75 times as long for a group of 128 as for one of 64 (37605 nodes, three rounds
// of 64 / two of 128: k_node_bwd_pre 27.4 / 30.4 us, k_node_bwd_post 42.4 / 49.0; 64000, four / two: 35.9 / 33.7, 56.8 / 55.4), bf16 1.45
// times (37605: 18.6 / 17.8, 27.0 / 25.0).  The number of workgroups - and of partial sums - does not depend on the type: it is the same
// for both choices as soon as every CU has a group of 128.
int bwd_workers(int64_t rows) { return (int)std::min<int64_t>(num_cus(), groups_of(rows, rows <= (int64_t)64 * num_cus() ? 64 : 128)); }
bool groups_of_64(int64_t rows, bool f32) {
    const int64_t cus = num_cus();
    if (rows <= 64 * cus) return true;
    if (!f32 || rows < 128 * cus) return false;
    const int64_t r64 = (groups_of(rows, 64) + cus - 1) / cus, r128 = (groups_of(rows, 128) + cus - 1) / cus;
    return 4 * r64 <= 7 * r128;
}

// bf16: 192 nodes where that saves more than a third of the rounds (a round of 192 takes 1.4 times one of 128; from 32769 to 49152 rows
// there is one instead of two).  128 / 192, us: k_node_bwd_pre 33 K rows 14.3 / 11.5, 48000 15.5 / 14.1, 64000 (two rounds of either) 16.0 / 19.3, 300 K
// 54.2 / 53.1; k_node_bwd_post of 33 K rows (same_bits) 27.5 / 22.5; k_readout_bwd 48000 26.3 / 20.8.  Not k_node_bwd_both and k_gt_bwd, which put 66 to 133 registers of sixteen waves to scratch (48000: 33.2 / 45.5,
// 28.0 / 35.0).
bool groups_of_192(int64_t rows) {
    const int64_t cus = num_cus();
    return 3 * ((groups_of(rows, 192) + cus - 1) / cus) < 2 * ((groups_of(rows, 128) + cus - 1) / cus);
}

template <typename... Args> int launch(void (*kernel)(Args...), std::atomic<uint64_t>& done, int grid, int threads, int lds, hipStream_t st, Args... args) {
    if (int rc = allow_lds(reinterpret_cast<const void*>(kernel), lds, done)) return rc;
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(threads), lds, st, args...);
    TGT_HIP_CHECK(hipGetLastError());
    return TGT_OK;
}


}  // namespace
}  // namespace tgt
