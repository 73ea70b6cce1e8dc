// The dense biased attention of query 0 alone: the last layer of the graph-level models.
//
// models/graphormer_graph_level.py:387 reads one row per graph of the last layer's output, the virtual node's.  So the last
// layer's attention is needed for query 0, its output projection and feed-forward block for one row per graph, and in the
// backward only row 0 of dQ and of the bias gradient differs from zero (dK and dV get one term per key); the bias gradient of
// row 0 belongs to the virtual distance.  256 graphs of 129 nodes in bf16: 27 + 84 us of full attention become 6 + 12 us.
//
// One wave per (graph, head), lane = key; the H waves of a workgroup share the node rows of their graph.  bf16 rounds where the
// matrix-core kernels of dense_attn.hip round (scores in tiles of 32 keys with a running maximum, probabilities and dS to bf16),
// float32 is float32 throughout (dense_attn_f32.hip).  Latency bound: a handful of dependent round trips.
#include "dense_dropout.h"
#include "dense_rows.h"
#include <cmath>

namespace tgt {
namespace {

constexpr int kRow0Max = 1024;      // longest sequence (its scores sit in LDS)
constexpr float kLog2e = 1.4426950408889634f;

__device__ __forceinline__ float rounded(float v, const float*) { return v; }
__device__ __forceinline__ float rounded(float v, const dbf16*) { return round_bf(v); }

template <int D> __device__ __forceinline__ void load_vec(const float* p, float (&x)[D]) {
#pragma unroll
    for (int c = 0; c < D; c += 4) {
        const float4 f = *reinterpret_cast<const float4*>(p + c);
        x[c] = f.x; x[c + 1] = f.y; x[c + 2] = f.z; x[c + 3] = f.w;
    }
}
template <int D> __device__ __forceinline__ void load_vec(const dbf16* p, float (&x)[D]) {
#pragma unroll
    for (int c = 0; c < D; c += 8) {
        const uint4 u = *reinterpret_cast<const uint4*>(p + c);
        const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            x[c + 2 * i] = __uint_as_float(w[i] << 16);
            x[c + 2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
        }
    }
}
template <int D> __device__ __forceinline__ void store_vec(float* p, const float (&x)[D]) {
#pragma unroll
    for (int c = 0; c < D; c += 4) *reinterpret_cast<float4*>(p + c) = make_float4(x[c], x[c + 1], x[c + 2], x[c + 3]);
}
template <int D> __device__ __forceinline__ void store_vec(dbf16* p, const float (&x)[D]) {
#pragma unroll
    for (int c = 0; c < D; c += 8) {
        uint32_t w[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            w[i] = (uint32_t)__builtin_bit_cast(uint16_t, static_cast<__bf16>(x[c + 2 * i])) | ((uint32_t)__builtin_bit_cast(uint16_t, static_cast<__bf16>(x[c + 2 * i + 1])) << 16);
        *reinterpret_cast<uint4*>(p + c) = make_uint4(w[0], w[1], w[2], w[3]);
    }
}
__device__ __forceinline__ float exp_of(float x, const float*) { return expf(x); }
__device__ __forceinline__ float exp_of(float x, const dbf16*) { return __builtin_amdgcn_exp2f(x * kLog2e); }

template <typename T> struct Row0Args {
    const T *q, *k, *v, *bias, *s;
    int b, S, H;
    float scale;
    T *a0, *s0;
    float* lse;
    // backward
    const T *da0, *g0;
    T *dq, *dk, *dv, *g;
    float* dvirt;
};

// The score of a key in one expression for forward and backward: the backward's exp(score - lse) is only as good as their last bits
// agree (scores reach the hundreds).  float32: the reference scales the query; bf16: the matrix-core kernels scale the product.
template <typename T, int D> __device__ __forceinline__ void scaled_query(const Row0Args<T>& a, int64_t row, float (&q)[D]) {
    load_vec<D>(a.q + row, q);
    if (sizeof(T) == 4)
#pragma unroll
        for (int c = 0; c < D; ++c) q[c] *= a.scale;
}
template <typename T, int D> __device__ __forceinline__ float score_of(const Row0Args<T>& a, const float (&q)[D], const float (&k)[D], float bias) {
    return sizeof(T) == 2 ? fmaf(dot_d<D>(q, k), a.scale, bias) : dot_d<D>(q, k) + bias;
}

template <typename T, int D, bool DROP> __global__ __launch_bounds__(512) void k_row0_fwd(const Row0Args<T> a, const DropArgs da) {
    extern __shared__ float lds[];
    constexpr bool MATRIX = sizeof(T) == 2;      // rounds like the matrix-core kernels
    const T* tag = nullptr;
    const int g = blockIdx.x, h = threadIdx.x >> 6, lane = threadIdx.x & 63, S = a.S, H = a.H, tiles = (S + 31) / 32;
    float *score = lds + h * (kRow0Max + 2 * (kRow0Max / 32)), *tile_max = score + kRow0Max, *factor = tile_max + kRow0Max / 32;
    const int64_t row = ((int64_t)g * S * H + h) * D, pitch = (int64_t)H * D;
    float q[D];
    scaled_query(a, row, q);
    const T* bias = a.bias ? a.bias + ((int64_t)g * H + h) * S * S : nullptr;
    for (int k0 = 0; k0 < S; k0 += 64) {
        const int key = k0 + lane;
        float sc = -INFINITY;
        if (key < S) {
            float kv[D];
            load_vec<D>(a.k + row + key * pitch, kv);
            const float bv = bias ? ld1(bias + key) : 0.f;
            sc = score_of(a, q, kv, bv);
            score[key] = sc;
        }
        float m = sc;
#pragma unroll
        for (int o = 16; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
        if ((lane & 31) == 0 && k0 + lane < S) tile_max[(k0 + lane) >> 5] = m;
    }
    __syncthreads();
    // running maximum of every tile and what its probabilities are still multiplied with when later tiles raise it
    float top = -INFINITY;
    for (int t = 0; t < tiles; ++t) top = fmaxf(top, tile_max[t]);
    if (MATRIX) {
        float m = -INFINITY;
        for (int t = 0; t < tiles; ++t) {
            const float next = fmaxf(m, tile_max[t]), use = next == -INFINITY ? 0.f : next;
            const float alpha = __builtin_amdgcn_exp2f((m - use) * kLog2e);
            __syncthreads();
            if (lane == 0) { tile_max[t] = use; factor[t] = alpha; }
            __syncthreads();
            m = next;
        }
        if (lane == 0) {
            float f = 1.f;
            for (int t = tiles - 1; t >= 0; --t) { const float alpha = factor[t]; factor[t] = f; f *= alpha; }
        }
        __syncthreads();
    }
    const float use = top == -INFINITY ? 0.f : top;
    const uint32_t rh = DROP ? drop_row_hash(da, g * H + h, 0) : 0u;
    float l = 0.f, o[D];
#pragma unroll
    for (int c = 0; c < D; ++c) o[c] = 0.f;
    for (int key = lane; key < S; key += 64) {
        float vv[D];
        load_vec<D>(a.v + row + key * pitch, vv);
        const float f = MATRIX ? factor[key >> 5] : 1.f;
        const float e = MATRIX ? __builtin_amdgcn_exp2f(fmaf(score[key], kLog2e, -tile_max[key >> 5] * kLog2e)) : expf(score[key] - use);
        const float p = rounded(e, tag);
        l += (D < 32 && !DROP ? p : e) * f;
        const float w = !DROP || drop_keep(da, rh, key) ? p * f : 0.f;
#pragma unroll
        for (int c = 0; c < D; ++c) o[c] = fmaf(w, vv[c], o[c]);
    }
    l = wave_sum(l);
    const float inv = (DROP ? da.inv_keep : 1.f) / l;
#pragma unroll
    for (int c = 0; c < D; ++c) o[c] = wave_sum(o[c]) * inv;
    const int64_t at = ((int64_t)g * H + h) * D;
    if (lane == 0) {
        store_vec<D>(a.a0 + at, o);
        a.lse[g * H + h] = use + logf(l);
    }
    if (lane < D) a.s0[at + lane] = a.s[row + lane];
}

template <typename T, int D, bool DROP> __global__ __launch_bounds__(512) void k_row0_bwd(const Row0Args<T> a, const DropArgs da) {
    const T* tag = nullptr;
    const int g = blockIdx.x, h = threadIdx.x >> 6, lane = threadIdx.x & 63, S = a.S, H = a.H;
    const int64_t row = ((int64_t)g * S * H + h) * D, pitch = (int64_t)H * D, at = ((int64_t)g * H + h) * D;
    float q[D], o[D], gv[D], g0[D], dq[D], none[D];
    scaled_query(a, row, q);
    load_vec<D>(a.a0 + at, o);
    load_vec<D>(a.da0 + at, gv);
    load_vec<D>(a.g0 + at, g0);
#pragma unroll
    for (int c = 0; c < D; ++c) { dq[c] = 0.f; none[c] = 0.f; }
    const float delta = dot_d<D>(o, gv), lse = a.lse[g * H + h];
    const uint32_t rh = DROP ? drop_row_hash(da, g * H + h, 0) : 0u;
    const T* bias = a.bias ? a.bias + ((int64_t)g * H + h) * S * S : nullptr;
    float dv_sum = 0.f;
    for (int key = lane; key < S; key += 64) {
        float kv[D], vv[D];
        load_vec<D>(a.k + row + key * pitch, kv);
        load_vec<D>(a.v + row + key * pitch, vv);
        const float sc = score_of(a, q, kv, bias ? ld1(bias + key) : 0.f);
        const float p = exp_of(sc - lse, tag), ks = !DROP ? 1.f : (drop_keep(da, rh, key) ? da.inv_keep : 0.f);
        const float ds = rounded(p * (dot_d<D>(gv, vv) * ks - delta), tag), pb = rounded(p * ks, tag);
        dv_sum += ds;
#pragma unroll
        for (int c = 0; c < D; ++c) {
            dq[c] = fmaf(ds, kv[c], dq[c]);
            kv[c] = sizeof(T) == 2 ? ds * q[c] * a.scale : ds * q[c];
            vv[c] = pb * gv[c];
        }
        store_vec<D>(a.dk + row + key * pitch, kv);
        store_vec<D>(a.dv + row + key * pitch, vv);
        if (key > 0) {
            store_vec<D>(a.dq + row + key * pitch, none);
            store_vec<D>(a.g + row + key * pitch, none);
        }
    }
#pragma unroll
    for (int c = 0; c < D; ++c) dq[c] = wave_sum(dq[c]) * a.scale;
    dv_sum = wave_sum(dv_sum);
    if (lane == 0) {
        store_vec<D>(a.dq + row, dq);
        store_vec<D>(a.g + row, g0);
        a.dvirt[g * H + h] = dv_sum;
    }
}

// d_virtual[h] += sum over graphs of the above (graphs in order); one wave per head
template <typename T> __global__ __launch_bounds__(64) void k_row0_virtual(const float* __restrict__ dvirt, int b, int H, T* __restrict__ d) {
    float t = 0.f;
    for (int g = threadIdx.x; g < b; g += 64) t += dvirt[g * H + blockIdx.x];
    t = wave_sum(t);
    if (threadIdx.x == 0) st1(d + blockIdx.x, ld1(d + blockIdx.x) + t);
}

int row0_check(const char* who, const void* q, const void* k, const void* v, int b, int S, int H, int d, int dtype, float p_drop) {
    if (!q || !k || !v || b < 1 || S < 1 || H < 1 || (d != 8 && d != 16 && d != 32) || (dtype != TGT_DTYPE_F32 && dtype != TGT_DTYPE_BF16) || !(p_drop >= 0.f && p_drop < 1.f)) {
        set_error("%s: null or bad argument", who);
        return TGT_ERR_INVALID_ARG;
    }
    if (S > kRow0Max || H > 8) {
        set_error("%s: at most %d rows and 8 heads", who, kRow0Max);
        return TGT_ERR_UNSUPPORTED;
    }
    return TGT_OK;
}
template <typename T, int D> int row0_launch(const Row0Args<T>& a, const DropArgs& da, bool drop, bool bwd, hipStream_t st) {
    const size_t lds = bwd ? 0 : sizeof(float) * a.H * (kRow0Max + 2 * (kRow0Max / 32));
    if (bwd) {
        if (drop) hipLaunchKernelGGL((k_row0_bwd<T, D, true>), dim3(a.b), dim3(64 * a.H), 0, st, a, da);
        else hipLaunchKernelGGL((k_row0_bwd<T, D, false>), dim3(a.b), dim3(64 * a.H), 0, st, a, da);
    } else {
        if (drop) hipLaunchKernelGGL((k_row0_fwd<T, D, true>), dim3(a.b), dim3(64 * a.H), lds, st, a, da);
        else hipLaunchKernelGGL((k_row0_fwd<T, D, false>), dim3(a.b), dim3(64 * a.H), lds, st, a, da);
    }
    TGT_HIP_CHECK(hipGetLastError());
    return TGT_OK;
}
template <typename T> int row0(Row0Args<T> a, int d, float p_drop, uint64_t seed, bool bwd, hipStream_t st) {
    a.scale = sqrtf((float)d);      // the reference multiplies q by sqrt(d)
    const DropArgs da = drop_args(p_drop, seed);
    return d == 8 ? row0_launch<T, 8>(a, da, p_drop > 0.f, bwd, st) : d == 16 ? row0_launch<T, 16>(a, da, p_drop > 0.f, bwd, st) : row0_launch<T, 32>(a, da, p_drop > 0.f, bwd, st);
}

}  // namespace
}  // namespace tgt

extern "C" {

int tgt_dense_row0_fwd(const void* d_q, const void* d_k, const void* d_v, const void* d_bias, const void* d_s, int b, int S, int H, int d, int dtype, float p_drop, uint64_t seed,
                       void* d_a0, void* d_s0, float* d_lse, void* stream) {
    using namespace tgt;
    if (int rc = row0_check("tgt_dense_row0_fwd", d_q, d_k, d_v, b, S, H, d, dtype, p_drop)) return rc;
    if (!d_s || !d_a0 || !d_s0 || !d_lse) { set_error("tgt_dense_row0_fwd: null pointer"); return TGT_ERR_INVALID_ARG; }
    KernelTimer t(KS_ROW0_FWD, (hipStream_t)stream);
    const auto run = [&](auto tag) {
        using T = decltype(tag);
        Row0Args<T> a{};
        a.q = (const T*)d_q; a.k = (const T*)d_k; a.v = (const T*)d_v; a.bias = (const T*)d_bias; a.s = (const T*)d_s;
        a.b = b; a.S = S; a.H = H; a.a0 = (T*)d_a0; a.s0 = (T*)d_s0; a.lse = d_lse;
        return row0(a, d, p_drop, seed, false, (hipStream_t)stream);
    };
    return dtype == TGT_DTYPE_F32 ? run(float()) : run(dbf16());
}

int tgt_dense_row0_bwd(const void* d_q, const void* d_k, const void* d_v, const void* d_bias, int b, int S, int H, int d, int dtype, float p_drop, uint64_t seed, const void* d_a0,
                       const float* d_lse, const void* d_da0, const void* d_g0, void* d_dq, void* d_dk, void* d_dv, void* d_g, float* d_dvirt, void* stream) {
    using namespace tgt;
    if (int rc = row0_check("tgt_dense_row0_bwd", d_q, d_k, d_v, b, S, H, d, dtype, p_drop)) return rc;
    if (!d_a0 || !d_lse || !d_da0 || !d_g0 || !d_dq || !d_dk || !d_dv || !d_g || !d_dvirt) { set_error("tgt_dense_row0_bwd: null pointer"); return TGT_ERR_INVALID_ARG; }
    KernelTimer t(KS_ROW0_BWD, (hipStream_t)stream);
    const auto run = [&](auto tag) {
        using T = decltype(tag);
        Row0Args<T> a{};
        a.q = (const T*)d_q; a.k = (const T*)d_k; a.v = (const T*)d_v; a.bias = (const T*)d_bias;
        a.b = b; a.S = S; a.H = H; a.a0 = (T*)d_a0; a.lse = (float*)d_lse; a.da0 = (const T*)d_da0; a.g0 = (const T*)d_g0;
        a.dq = (T*)d_dq; a.dk = (T*)d_dk; a.dv = (T*)d_dv; a.g = (T*)d_g; a.dvirt = d_dvirt;
        return row0(a, d, p_drop, seed, true, (hipStream_t)stream);
    };
    return dtype == TGT_DTYPE_F32 ? run(float()) : run(dbf16());
}

int tgt_dense_row0_virtual(const float* d_dvirt, int b, int H, int dtype, void* d_dvirtual_dist, void* stream) {
    using namespace tgt;
    if (!d_dvirt || b < 1 || H < 1 || !d_dvirtual_dist || (dtype != TGT_DTYPE_F32 && dtype != TGT_DTYPE_BF16)) { set_error("tgt_dense_row0_virtual: null or bad argument"); return TGT_ERR_INVALID_ARG; }
    KernelTimer t(KS_GRAPH_BIAS_BWD, (hipStream_t)stream);
    if (dtype == TGT_DTYPE_F32) hipLaunchKernelGGL((k_row0_virtual<float>), dim3(H), dim3(64), 0, (hipStream_t)stream, d_dvirt, b, H, (float*)d_dvirtual_dist);
    else hipLaunchKernelGGL((k_row0_virtual<dbf16>), dim3(H), dim3(64), 0, (hipStream_t)stream, d_dvirt, b, H, (dbf16*)d_dvirtual_dist);
    TGT_HIP_CHECK(hipGetLastError());
    return TGT_OK;
}

}  // extern "C"
