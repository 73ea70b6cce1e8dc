// Packing of the fused layers' parameters: weights of up to 64 x 64 into the order in which the products read them (both ways), vectors as float32.
// As a launch of its own (node_layer.hip) or beside the first linear of a model (linear_tiles.hip).
#pragma once
#include "node_tile.h"
#include <algorithm>

namespace tgt {
namespace {

constexpr int kPackMats = 96, kPackVecs = 160;
struct PackArgs {
    const void* mat[kPackMats];
    int16_t ld[kPackMats], rows[kPackMats], cols[kPackMats];
    const void* vec[kPackVecs];
    int16_t len[kPackVecs];
    int n_mats, n_vecs, mat0, total_mats, vec0;
    vec16* frags;       // [2][total_mats][kFragVecs]: for y = W x, then for dx = W^T dy
    float* vecs;        // [..][64]
};

// block b of pack_blocks: 512 operand vectors of one (weight, direction), or THREADS / 64 vectors
template <typename T, int THREADS> __device__ __forceinline__ void pack_block(const PackArgs& a, int b) {
    constexpr int P = Num<T>::P;
    if (b >= 2 * a.n_mats) {
        const int i = (b - 2 * a.n_mats) * (THREADS / 64) + threadIdx.x / 64, e = threadIdx.x & 63;
        if (i < a.n_vecs) a.vecs[(a.vec0 + i) * kVec + e] = e < a.len[i] ? as_float(reinterpret_cast<const T*>(a.vec[i])[e]) : 0.f;
        return;
    }
    const int j = b >> 1, back = b & 1;
    const T* W = reinterpret_cast<const T*>(a.mat[j]);
    const int ld = a.ld[j], rows = a.rows[j], cols = a.cols[j];
    const int lane = threadIdx.x & 63;
    float v[512 / THREADS][8];
#pragma unroll
    for (int u = 0; u < 512 / THREADS; ++u) {
        const int sm = (threadIdx.x >> 6) + u * (THREADS / 64), s = sm >> 2, m = sm & 3;
        const int out_f = 16 * gray2((lane >> 2) & 3) + 4 * m + (lane & 3), in0 = 16 * (lane >> 4) + 8 * s;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int o = back ? in0 + i : out_f, k = back ? out_f : in0 + i;
            v[u][i] = o < rows && k < cols ? as_float(W[o * ld + k]) : 0.f;
        }
    }
    vec16* dst = a.frags + ((int64_t)(back ? a.total_mats : 0) + a.mat0 + j) * kFragVecs<P>;
#pragma unroll
    for (int u = 0; u < 512 / THREADS; ++u) {
        const int sm = (threadIdx.x >> 6) + u * (THREADS / 64);
        bf16x8_t p[P];
        to_planes(v[u], p);
#pragma unroll
        for (int q = 0; q < P; ++q) dst[(sm * P + q) * 64 + lane] = __builtin_bit_cast(vec16, p[q]);
    }
}
inline int pack_blocks(const PackArgs& a, int threads) { return 2 * a.n_mats + (a.n_vecs + threads / 64 - 1) / (threads / 64); }

inline int check_pack(const tgt_node_pack_args* a, int dtype) {
    const auto bad = [](const char* what) { set_error("tgt_node_pack: %s", what); return TGT_ERR_INVALID_ARG; };
    if (!a || !a->mats || !a->ld || !a->rows || !a->vecs || !a->lens || a->n_mats < 1 || a->n_vecs < 1 || !a->d_frags || !a->d_vecs ||
        (dtype != TGT_DTYPE_F32 && dtype != TGT_DTYPE_BF16))
        return bad("null or bad argument");
    for (int i = 0; i < a->n_mats; ++i) {
        const int c = a->cols ? a->cols[i] : 64;
        if (!a->mats[i] || a->rows[i] < 1 || a->rows[i] > 64 || c < 1 || c > 64 || a->ld[i] < c || a->ld[i] > 32767) return bad("weights are [1..64, >= 64]");
    }
    for (int i = 0; i < a->n_vecs; ++i)
        if (!a->vecs[i] || a->lens[i] < 1 || a->lens[i] > 64) return bad("vectors have 1 to 64 elements");
    return TGT_OK;
}
// what one launch takes from weight m and vector v on
inline PackArgs pack_args(const tgt_node_pack_args& p, int m, int v) {
    PackArgs a{};
    a.n_mats = std::min(kPackMats, p.n_mats - m); a.n_vecs = std::min(kPackVecs, p.n_vecs - v);
    a.mat0 = m; a.vec0 = v; a.total_mats = p.n_mats;
    a.frags = (vec16*)p.d_frags; a.vecs = p.d_vecs;
    for (int i = 0; i < a.n_mats; ++i) {
        a.mat[i] = p.mats[m + i];
        a.ld[i] = (int16_t)p.ld[m + i]; a.rows[i] = (int16_t)p.rows[m + i]; a.cols[i] = (int16_t)(p.cols ? p.cols[m + i] : 64);
    }
    for (int i = 0; i < a.n_vecs; ++i) { a.vec[i] = p.vecs[v + i]; a.len[i] = (int16_t)p.lens[v + i]; }
    return a;
}

}  // namespace
}  // namespace tgt
