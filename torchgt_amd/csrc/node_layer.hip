// The node-local part of a Graphormer encoder layer (models/graphormer_dist_node_level.py:246-314 and
// models/graphormer_graph_level.py:267-306), hidden and feed-forward width 64, as one forward and two backward kernels.
//
//   forward   [attention rows a, residual stream s] -> s1 = s + a Wo^T + bo;  s' = s1 + W2 gelu(W1 LN2(s1) + b1) + b2
//             and, in the same pass, what the next layer's attention reads: q, k, v = LN1(s') W^T + b - or the class
//             log-probabilities log_softmax(LN(s') Wh^T + bh) behind the last layer
//   backward  k_node_bwd_pre:  dq, dk, dv, ds' (residual) -> ds', gradients of Wq / Wk / Wv and LN1 (and the same for the
//             classes: one weight, d log_softmax in front)
//             k_node_bwd_post: ds' -> ds (residual), da, gradients of Wo, W1, W2 and LN2, and (1 / (Z + eps), da . a) per
//             node and head, which the sparse attention's backward starts from
//
// What bounds them and why this shape.  As one kernel per linear, LayerNorm and activation the part moves 29 rows of 64
// features per node forward and 47 backward through memory; here it moves 6 and 12 (q, k, v, the residual stream and the
// attention rows; the intermediate activations are recomputed in the backward from s and a: two products, against two rows
// written and read).  A wave takes 32 nodes and keeps them in registers through the whole chain (node_tile.h); the waves of
// a workgroup share the packed weights in LDS.  Weight gradients contract over nodes: in the backward kernels four waves carry 32
// nodes each through the chain and put the bf16 planes of both operands into LDS, four others keep one 32 x 32 block of every
// weight gradient each and add the products over these 128 nodes beside it (node_roles.h).
#include "node_roles.h"

namespace tgt {
namespace {

// ---- packing of the parameters ---------------------------------------------------------------------------------------
constexpr int kPackMats = 96, kPackVecs = 160;
struct PackArgs {
    const void* mat[kPackMats];
    int16_t ld[kPackMats], rows[kPackMats];
    const void* vec[kPackVecs];
    int16_t len[kPackVecs];
    int n_mats, n_vecs, mat0, total_mats, vec0;
    vec16* frags;       // [2][total_mats][kFragVecs]: for y = W x, then for dx = W^T dy
    float* vecs;        // [..][64]
};
__device__ __forceinline__ float as_float(float v) { return v; }
__device__ __forceinline__ float as_float(nbf16 v) { return __uint_as_float((uint32_t)v.x << 16); }

// workgroup = one (weight, direction): 512 operand vectors, one per thread; the workgroups behind the weights copy vectors
template <typename T> __global__ __launch_bounds__(512) void k_node_pack(const PackArgs a) {
    constexpr int P = Num<T>::P;
    const int b = blockIdx.x;
    if (b >= 2 * a.n_mats) {
        const int i = (b - 2 * a.n_mats) * 8 + threadIdx.x / 64, e = threadIdx.x & 63;
        if (i < a.n_vecs) a.vecs[(a.vec0 + i) * kVec + e] = e < a.len[i] ? as_float(reinterpret_cast<const T*>(a.vec[i])[e]) : 0.f;
        return;
    }
    const int j = b >> 1, back = b & 1;
    const T* W = reinterpret_cast<const T*>(a.mat[j]);
    const int ld = a.ld[j], rows = a.rows[j];
    const int lane = threadIdx.x & 63, sm = threadIdx.x >> 6, s = sm >> 1, m = sm & 1;
    const int r = lane & 31, out_f = 32 * ((r >> 2) & 1) + 16 * m + 4 * (r >> 3) + (r & 3), in0 = 32 * (lane >> 5) + 8 * s;
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int o = back ? in0 + i : out_f, k = back ? out_f : in0 + i;
        v[i] = o < rows ? as_float(W[o * ld + k]) : 0.f;
    }
    bf16x8_t p[P];
    to_planes(v, p);
    vec16* dst = a.frags + ((int64_t)(back ? a.total_mats : 0) + a.mat0 + j) * kFragVecs<P>;
#pragma unroll
    for (int q = 0; q < P; ++q) dst[(sm * P + q) * 64 + lane] = __builtin_bit_cast(vec16, p[q]);
}

// ---- GELU of a tile of pre-activations (and its slope) ---------------------------------------------------------------------
// SAME (bf16): every sum and rounding as the separate kernels have it - GELU by the device library's error function, products of
// half the depth, the bias behind the products, LayerNorm's sums in their order.  The graph-level models ask for it: they multiply
// queries by sqrt(d), their attention is often all but a choice of one key, and in bf16 a rounding that falls the other way in one
// activation moves every gradient of that graph by a per cent (0.019 of the gradients' norm without, 0.010 with it).
template <typename T, bool SAME> __device__ __forceinline__ float cdf_and_bell(float v, float& bell) {
    float cdf;
    if constexpr (SAME) {
        cdf = 0.5f * (1.f + erff(v * 0.70710678118654752f));
        bell = __expf(-0.5f * v * v);
    } else normal_cdf(v, cdf, bell);
    return cdf;
}
template <typename T, bool SAME> __device__ __forceinline__ void gelu(Tile& u) {
    TGT_EACH(i) {
        const float v = stored(u.get(i), (const T*)nullptr);
        float bell;
        if constexpr (SAME) u.set(i, act_value<false>(v));
        else u.set(i, v * cdf_and_bell<T, SAME>(v, bell));
        if (i % 8 == 7) fence_schedule();
    }
}
template <typename T, bool SAME> __device__ __forceinline__ void gelu(Tile& u, Tile& slope) {
    TGT_EACH(i) {
        const float v = stored(u.get(i), (const T*)nullptr);
        float bell;
        const float cdf = cdf_and_bell<T, SAME>(v, bell);
        u.set(i, v * cdf);
        slope.set(i, cdf + v * bell * 0.39894228040143268f);
        if (i % 8 == 7) fence_schedule();
    }
}

// ---- forward ------------------------------------------------------------------------------------------------------------
enum { NEXT_NONE = 0, NEXT_QKV = 1, NEXT_CLASSES = 2 };

template <typename T, bool SAME> constexpr int fwd_waves() { return sizeof(T) == 4 || SAME ? 8 : 16; }
// bf16 keeps all weights of a launch in LDS for the life of the workgroup; float32 planes of six weights (144 KB) do not
// leave room for the row images, so its two halves take turns (the L2 has them)
template <typename T, bool POST, int NEXT> constexpr int fwd_resident_mats() {
    const int post = POST ? 3 : 0, next = NEXT == NEXT_QKV ? 3 : (NEXT == NEXT_CLASSES ? 1 : 0);
    return sizeof(T) == 4 ? (post > next ? post : next) : post + next;
}
template <typename T, bool SAME, bool POST, int NEXT> constexpr int fwd_lds() {
    return fwd_resident_mats<T, POST, NEXT>() * kFragVecs<Num<T>::P> * 16 + 10 * kVec * 4 + fwd_waves<T, SAME>() * RowShape<T>::kVecs * 16;
}

// Rows of class values.  A wave's 32 rows are 32 C consecutive elements of the [N - tokens, C] array and travel through its
// row image, in words: for bf16 the image starts one element late where the rows begin in the middle of a word.
template <typename T> struct ClassRows {
    static constexpr int kPerWord = 4 / (int)sizeof(T);
    T* img;
    int C, lo, hi;            // elements of the wave's rows that exist: [lo, hi)
    int64_t first, total;     // element of the array the rows start at (negative: token rows), elements of the array
    int shift;
    __device__ __forceinline__ ClassRows(vec16* stage, int64_t row0, int64_t N, int tokens, int classes) {
        C = classes;
        const int64_t r = row0 - tokens, left = N - row0;
        first = r * C; total = (N - tokens) * C;
        lo = r < 0 ? (int)(-r < 32 ? -r : 32) * C : 0;
        hi = (int)(left < 0 ? 0 : (left < 32 ? left : 32)) * C;
        shift = kPerWord == 2 ? (int)(first & 1) : 0;
        img = reinterpret_cast<T*>(stage) + shift;
    }
    __device__ __forceinline__ int words() const { return (hi + shift + kPerWord - 1) / kPerWord; }
    // array -> image; every load is issued before the first is waited for
    __device__ __forceinline__ void load(const T* __restrict__ src, int lane) {
        const int n = words();
        const int64_t w0 = (first - shift) / kPerWord, last = total / kPerWord - 1;
        const uint32_t* p = reinterpret_cast<const uint32_t*>(src);
        uint32_t v[32];
#pragma unroll
        for (int i = 0; i < 32; ++i)
            if (i * 64 < n && last >= 0) {
                int64_t w = w0 + i * 64 + lane;
                w = w < 0 ? 0 : (w > last ? last : w);
                v[i] = p[w];
            }
        wave_sync();
        uint32_t* d = reinterpret_cast<uint32_t*>(img - shift);
#pragma unroll
        for (int i = 0; i < 32; ++i)
            if (i * 64 < n && last >= 0 && i * 64 + lane < n) d[i * 64 + lane] = v[i];
        wave_sync();
        if (kPerWord == 2 && (total & 1) && first + hi == total && hi > lo && lane == 0) img[hi - 1] = src[total - 1];      // half a word at the end
        wave_sync();
    }
    __device__ __forceinline__ void store(T* __restrict__ dst, int lane) const {
        const uint32_t* d = reinterpret_cast<const uint32_t*>(img - shift);
        T* out = dst + first;
        const int n = words();
        for (int w = lane; w < n; w += 64) {
            const int e = w * kPerWord - shift;
            if (e >= lo && e + kPerWord <= hi) *reinterpret_cast<uint32_t*>(out + e) = d[w];
            else {
#pragma unroll
                for (int k = 0; k < kPerWord; ++k)
                    if (e + k >= lo && e + k < hi) out[e + k] = img[e + k];
            }
        }
    }
};
template <typename T> __device__ __forceinline__ T to_elem(float v);
template <> __device__ __forceinline__ float to_elem<float>(float v) { return v; }
template <> __device__ __forceinline__ nbf16 to_elem<nbf16>(float v) { return nbf16{__builtin_bit_cast(uint16_t, static_cast<__bf16>(v))}; }

template <typename T, bool SAME, bool POST, int NEXT>
__global__ __launch_bounds__((fwd_waves<T, SAME>() * 64)) void k_node_fwd(const tgt_node_fwd_args a) {
    constexpr int P = Num<T>::P, NW = fwd_waves<T, SAME>(), THREADS = NW * 64, FV = kFragVecs<P>;
    constexpr bool RESIDENT = sizeof(T) == 2;
    constexpr int NMP = NEXT == NEXT_QKV ? 3 : (NEXT == NEXT_CLASSES ? 1 : 0);
    extern __shared__ __align__(16) unsigned char smem[];
    vec16* w = reinterpret_cast<vec16*>(smem);
    vec16* w_next = w + (RESIDENT && POST ? 3 * FV : 0);
    float* vec = reinterpret_cast<float*>(w + fwd_resident_mats<T, POST, NEXT>() * FV);
    float* vn = vec + 5 * kVec;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h = lane >> 5;
    vec16* stage = reinterpret_cast<vec16*>(vec + 10 * kVec) + wave * RowShape<T>::kVecs;
    const int64_t N = a.rows, tiles = (N + 31) / 32;
    if constexpr (POST) copy_vecs<5 * kVec / 4, THREADS>(reinterpret_cast<vec16*>(vec), reinterpret_cast<const vec16*>(a.v_post));
    if constexpr (NEXT != NEXT_NONE) copy_vecs<(2 + NMP) * kVec / 4, THREADS>(reinterpret_cast<vec16*>(vn), reinterpret_cast<const vec16*>(a.v_next));
    if (RESIDENT) {
        if constexpr (POST) copy_vecs<3 * FV, THREADS>(w, reinterpret_cast<const vec16*>(a.w_post));
        if constexpr (NEXT != NEXT_NONE) copy_vecs<NMP * FV, THREADS>(w_next, reinterpret_cast<const vec16*>(a.w_next));
        __syncthreads();
    }
    for (int64_t t0 = (int64_t)blockIdx.x * NW; t0 < tiles; t0 += (int64_t)gridDim.x * NW) {
        const Rows rows(t0 + wave, N);
        const int64_t row0 = (t0 + wave) * 32;
        const bool active = rows.left > 0;
        Raw<T> raw_a, raw_s;
        if (active) {
            fetch(raw_s, reinterpret_cast<const T*>(a.s_in), rows, lane);
            if (POST) fetch(raw_a, reinterpret_cast<const T*>(a.attn), rows, lane);
        }
        if (!RESIDENT && POST) {
            __syncthreads();
            copy_vecs<3 * FV, THREADS>(w, reinterpret_cast<const vec16*>(a.w_post));
            __syncthreads();
        }
        Tile s;
        if (active) {
            if (!POST && row0 < a.tokens) {      // the global tokens in front of the nodes: from their table, and into the stream
                constexpr int PP = RowShape<T>::kPieces, PER = RowShape<T>::kPer;
#pragma unroll
                for (int i = 0; i < RowShape<T>::kAcc; ++i) {
                    const int64_t r = row0 + i * PER + lane / PP;
                    if (r < a.tokens) {
                        raw_s.v[i] = reinterpret_cast<const vec16*>(a.token)[r * PP + lane % PP];
                        reinterpret_cast<vec16*>(a.s_out)[r * PP + lane % PP] = raw_s.v[i];
                    }
                }
            }
            settle<T, false>(s, raw_s, stage, rows, lane);
            if (POST) {
                Tile x, y;
                settle<T, false>(x, raw_a, stage, rows, lane);
                linear<P, SAME>(y, x, w, vec, lane);
                TGT_EACH(i) s.set(i, s.get(i) + stored(y.get(i), (const T*)nullptr));      // s1 = s + (a Wo^T + bo)
                x = s;
                normalise<SAME>(x, a.eps_post);
                affine(x, x, vec + kVec, vec + 2 * kVec, h);      // y2
                linear<P, SAME>(y, x, w + FV, vec + 3 * kVec, lane);    // u
                gelu<T, SAME>(y);
                linear<P, SAME>(x, y, w + 2 * FV, vec + 4 * kVec, lane);
                TGT_EACH(i) s.set(i, stored(s.get(i), (const T*)nullptr) + stored(x.get(i), (const T*)nullptr));      // s'
                put_rows(reinterpret_cast<T*>(a.s_out), s, stage, rows, lane);
            }
        }
        if constexpr (!RESIDENT && NEXT != NEXT_NONE) {
            __syncthreads();
            copy_vecs<NMP * FV, THREADS>(w, reinterpret_cast<const vec16*>(a.w_next));
            __syncthreads();
        }
        if (NEXT && active) {
            normalise<SAME>(s, a.eps_next);
            affine(s, s, vn, vn + kVec, h);
            if (NEXT == NEXT_QKV) {
#pragma unroll
                for (int j = 0; j < 3; ++j) {
                    Tile y;
                    linear<P, SAME>(y, s, w_next + j * FV, vn + (2 + j) * kVec, lane);
                    put_rows(reinterpret_cast<T*>(j == 0 ? a.q : (j == 1 ? a.k : a.v)), y, stage, rows, lane);
                }
            } else {
                Tile y;
                linear<P, SAME>(y, s, w_next, vn + 2 * kVec, lane);
                const int C = a.classes;
                float lse = 0.f;
                if (!a.linear) {
                    float top = -INFINITY, sum = 0.f;
                    TGT_EACH(i) {      // rounded first: log_softmax reads the logits as a T tensor would hold them
                        y.set(i, stored(y.get(i), (const T*)nullptr));
                        if (32 * h + i < C) top = fmaxf(top, y.get(i));
                    }
                    top = fmaxf(top, __shfl_xor(top, 32, 64));
                    TGT_EACH(i) if (32 * h + i < C) sum += expf(y.get(i) - top);
                    lse = top + logf(both_halves(sum));
                }
                const ClassRows<T> out(stage, row0, N, a.tokens, C);
                wave_sync();
                TGT_EACH(i) if (32 * h + i < C) out.img[(lane & 31) * C + 32 * h + i] = to_elem<T>(y.get(i) - lse);
                wave_sync();
                out.store(reinterpret_cast<T*>(a.logp), lane);
            }
        }
    }
}

// Class gradients of a wave's 32 rows: d logits = d logp - softmax * sum(d logp) (linear: d logits as they come); zero for tokens and past the end.
template <typename T> __device__ __forceinline__ void class_grads(Tile& d, const T* __restrict__ dlogp, const T* __restrict__ logp, bool linear, int C, int tokens, int64_t row0, int64_t N,
                                                                  vec16* stage, int lane) {
    const int n = lane & 31, h = lane >> 5;
    ClassRows<T> rows(stage, row0, N, tokens, C);
    const bool in = n * C >= rows.lo && n * C < rows.hi;
    const T* mine = rows.img + (in ? n * C + 32 * h : 0);
    rows.load(dlogp, lane);
    float sum = 0.f;
    TGT_EACH(i) {
        d.set(i, in && 32 * h + i < C ? as_float(mine[i]) : 0.f);
        sum += d.get(i);
    }
    if (linear) return;
    sum = both_halves(sum);
    rows.load(logp, lane);
    TGT_EACH(i) if (in && 32 * h + i < C) d.set(i, d.get(i) - expf(as_float(mine[i])) * sum);
}

// ---- backward of the part in front of an attention (or of the classes) ------------------------------------------------------
// NORM false (GT): q, k, v are made of the rows s themselves.
template <typename T, bool CLASSES, bool NORM>
__global__ __launch_bounds__(kBwdThreads) void k_node_bwd_pre(const tgt_node_bwd_pre_args a) {
    using L = BwdLds<T>;
    constexpr int P = Num<T>::P, FV = kFragVecs<P>, NM = CLASSES ? 1 : 3;
    extern __shared__ __align__(16) unsigned char smem[];
    unsigned char *p_dy = smem, *p_x = smem + P * kPlaneBytes;
    vec16* w = reinterpret_cast<vec16*>(smem + L::kW);
    float* vec = reinterpret_cast<float*>(smem + L::kVecs);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h = lane >> 5;
    const int64_t N = a.rows, groups = (N + kChainNodes - 1) / kChainNodes;
    if constexpr (NORM) copy_vecs<2 * kVec / 4, kBwdThreads>(reinterpret_cast<vec16*>(vec), reinterpret_cast<const vec16*>(a.v_next));
    __syncthreads();
    float16_t acc[NM];
    float col[NM + 2];
#pragma unroll
    for (int j = 0; j < NM; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[j][r] = 0.f;
#pragma unroll
    for (int j = 0; j < NM + 2; ++j) col[j] = 0.f;
    if (wave < 4) {
        vec16* stage = reinterpret_cast<vec16*>(smem + L::kStage) + wave * RowShape<T>::kVecs;
        const T* src[3] = {reinterpret_cast<const T*>(a.dq), reinterpret_cast<const T*>(a.dk), reinterpret_cast<const T*>(a.dv)};
        const int row = 32 * wave + (lane & 31);
        Raw<T> raw_s, raw_d;
        {
            const Rows rows(4 * (int64_t)blockIdx.x + wave, N);
            fetch(raw_s, reinterpret_cast<const T*>(a.s), rows, lane);
            if (!CLASSES) fetch(raw_d, src[0], rows, lane);
        }
        for (int64_t g0 = blockIdx.x; g0 < groups; g0 += gridDim.x) {
            const Rows rows(4 * g0 + wave, N);
            Tile xhat, dy, d;
            Frags<P> f;
            settle<T, false>(xhat, raw_s, stage, rows, lane);
            float rstd = 1.f;
            if constexpr (NORM) rstd = normalise<false>(xhat, a.eps);
            zero(dy);
#pragma unroll
            for (int j = 0; j < NM; ++j) {
                if (CLASSES) class_grads(d, reinterpret_cast<const T*>(a.dlogp), reinterpret_cast<const T*>(a.logp), a.linear, a.classes, a.tokens, (4 * g0 + wave) * 32, N, stage, lane);
                else {
                    settle<T, true>(d, raw_d, stage, rows, lane);
                    fetch(raw_d, j + 1 < NM ? src[j + 1] : reinterpret_cast<const T*>(a.g_in), rows, lane);
                }
                make_frags(f, d);
                col[j] += column_sums(d, lane);
                __syncthreads();                       // weight j is there; j = 0: the planes are free
                gemm<P>(dy, f, w, lane);               // beside product j - 1 of the block waves
                if (j > 0) __syncthreads();            // product j - 1 is done
                else {
                    Tile y;
                    if constexpr (NORM) affine(y, xhat, vec, vec + kVec, h);
                    else y = xhat;
                    Frags<P> fx;
                    make_frags(fx, y);
                    put_planes<P>(p_x, row, h, fx);
                }
                put_planes<P>(p_dy, row, h, f);
                __syncthreads();                       // planes j are there, weight j has been used
            }
            if (g0 + gridDim.x < groups) fetch(raw_s, reinterpret_cast<const T*>(a.s), Rows(4 * (g0 + gridDim.x) + wave, N), lane);
            TGT_EACH(i) dy.set(i, stored(dy.get(i), (const T*)nullptr));
            if constexpr (NORM) {
                col[NM + 1] += column_sums(dy, lane);
                TGT_EACH(i) d.set(i, dy.get(i) * xhat.get(i));
                col[NM] += column_sums(d, lane);
            }
            if (CLASSES) zero(d);
            else {
                settle<T, true>(d, raw_d, stage, rows, lane);
                if (g0 + gridDim.x < groups) fetch(raw_d, src[0], Rows(4 * (g0 + gridDim.x) + wave, N), lane);
            }
            if constexpr (NORM) ln_back(d, dy, xhat, rstd, vec, h);
            else TGT_EACH(i) d.set(i, d.get(i) + dy.get(i));
            put_rows(reinterpret_cast<T*>(a.g_out), d, stage, rows, lane);
            if (a.d_token && 4 * g0 + wave < (a.tokens + 31) / 32) put_rows(reinterpret_cast<T*>(a.d_token), d, stage, Rows(4 * g0 + wave, a.tokens), lane);
        }
    } else {
        const int q = wave - 4, base_dy = operand_base(q >> 1, lane), base_x = operand_base(q & 1, lane);
        const vec16* weights = reinterpret_cast<const vec16*>(a.w_back);
        WeightsAhead<FV> next;
        next.fetch(weights);
        for (int64_t g0 = blockIdx.x; g0 < groups; g0 += gridDim.x) {
            next.put(w);
            next.fetch(weights + (NM > 1 ? FV : 0));
            __syncthreads();
#pragma unroll
            for (int j = 0; j < NM; ++j) {
                __syncthreads();                       // planes j
                if (j + 1 < NM) {
                    next.put(w);
                    next.fetch(weights + (j + 2 < NM ? j + 2 : 0) * FV);
                    __syncthreads();                   // weight j + 1
                }
                node_product<P>(acc[j], p_dy, p_x, base_dy, base_x);
                if (j + 1 < NM) __syncthreads();       // product j is done
            }
        }
    }
    write_partial<NM, NM + 2>(a.partial + (int64_t)blockIdx.x * (NM * 4096 + (NM + 2) * 64), acc, col, reinterpret_cast<float*>(smem), wave, lane);
}

// ---- backward of the part behind an attention -------------------------------------------------------------------------------
template <typename T, bool SAME>
__global__ __launch_bounds__(kBwdThreads) void k_node_bwd_post(const tgt_node_bwd_post_args a) {
    using L = BwdLds<T>;
    constexpr int P = Num<T>::P, FV = kFragVecs<P>;
    extern __shared__ __align__(16) unsigned char smem[];
    unsigned char *p_dy = smem, *p_x = smem + P * kPlaneBytes;
    vec16* w = reinterpret_cast<vec16*>(smem + L::kW);
    float* vec = reinterpret_cast<float*>(smem + L::kVecs);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), n = lane & 31, h = lane >> 5;
    const int64_t N = a.rows, groups = (N + kChainNodes - 1) / kChainNodes;
    copy_vecs<5 * kVec / 4, kBwdThreads>(reinterpret_cast<vec16*>(vec), reinterpret_cast<const vec16*>(a.v_post));
    __syncthreads();
    float16_t acc[3];       // Wo, W1, W2
    float col[5];           // bo, b1, b2, gamma, beta
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[j][r] = 0.f;
#pragma unroll
    for (int j = 0; j < 5; ++j) col[j] = 0.f;
    if (wave < 4) {
        vec16* stage = reinterpret_cast<vec16*>(smem + L::kStage) + wave * RowShape<T>::kVecs;
        const int row = 32 * wave + n;
        Raw<T> raw_a, raw_s, raw_g;
        {
            const Rows rows(4 * (int64_t)blockIdx.x + wave, N);
            fetch(raw_a, reinterpret_cast<const T*>(a.attn), rows, lane);
            fetch(raw_s, reinterpret_cast<const T*>(a.s), rows, lane);
            fetch(raw_g, reinterpret_cast<const T*>(a.g_in), rows, lane);
        }
        for (int64_t g0 = blockIdx.x; g0 < groups; g0 += gridDim.x) {
            const Rows rows(4 * g0 + wave, N);
            const auto fetch_next = [&]() {
                if (g0 + gridDim.x >= groups) return;
                const Rows ahead(4 * (g0 + gridDim.x) + wave, N);
                fetch(raw_a, reinterpret_cast<const T*>(a.attn), ahead, lane);
                fetch(raw_s, reinterpret_cast<const T*>(a.s), ahead, lane);
                fetch(raw_g, reinterpret_cast<const T*>(a.g_in), ahead, lane);
            };
            Tile g, xhat, slope, t;
            Frags<P> f, fy;      // fy: LayerNorm's output, kept in its one plane for bf16, formed again from xhat for float32
            settle<T, false>(t, raw_a, stage, rows, lane);
            make_frags(f, t);
            settle<T, false>(xhat, raw_s, stage, rows, lane);
            settle<T, true>(g, raw_g, stage, rows, lane);
            col[2] += column_sums(g, lane);
            __syncthreads();                                        // Wo is there; product Wo of the round before is done
            linear<P, SAME>(t, f, w, vec, lane);
            __syncthreads();                                        // Wo has been used
            TGT_EACH(i) xhat.set(i, xhat.get(i) + stored(t.get(i), (const T*)nullptr));      // s1
            t = xhat;
            const MeanRstd stat = row_stats<SAME>(t, a.eps);
            TGT_EACH(i) {      // LayerNorm's output is made of s1, its backward reads s1 as the stream holds it
                t.set(i, (t.get(i) - stat.mean) * stat.rstd);
                xhat.set(i, (stored(xhat.get(i), (const T*)nullptr) - stat.mean) * stat.rstd);
            }
            affine(t, t, vec + kVec, vec + 2 * kVec, h);
            make_frags(fy, t);
            __syncthreads();                                        // W1
            linear<P, SAME>(t, fy, w, vec + 3 * kVec, lane);           // u
            __syncthreads();                                        // W1 has been used
            gelu<T, SAME>(t, slope);
            make_frags(f, t);
            put_planes<P>(p_x, row, h, f);
            make_frags(f, g);
            put_planes<P>(p_dy, row, h, f);
            __syncthreads();                                        // planes of W2; W2^T
            zero(t);
            gemm<P>(t, f, w, lane);                                 // d gelu, beside product W2
            TGT_EACH(i) t.set(i, stored(t.get(i) * slope.get(i), (const T*)nullptr));      // du
            col[1] += column_sums(t, lane);
            make_frags(f, t);
            if (P != 1) {
                forget(xhat);
                affine(t, xhat, vec + kVec, vec + 2 * kVec, h);
            }
            __syncthreads();                                        // product W2 is done, W2^T has been used
            put_planes<P>(p_dy, row, h, f);
            if (P != 1) make_frags(fy, t);
            put_planes<P>(p_x, row, h, fy);
            __syncthreads();                                        // planes of W1; W1^T
            fetch(raw_a, reinterpret_cast<const T*>(a.attn), rows, lane);
            zero(t);
            gemm<P>(t, f, w, lane);                                 // d LN, beside product W1
            TGT_EACH(i) t.set(i, stored(t.get(i), (const T*)nullptr));
            col[4] += column_sums(t, lane);
            ln_back(g, t, xhat, stat.rstd, vec + kVec, h);
            TGT_EACH(i) g.set(i, stored(g.get(i), (const T*)nullptr));
            TGT_EACH(i) t.set(i, t.get(i) * xhat.get(i));
            col[3] += column_sums(t, lane);
            col[0] += column_sums(g, lane);
            put_rows(reinterpret_cast<T*>(a.g_out), g, stage, rows, lane);
            make_frags(f, g);
            settle<T, false>(t, raw_a, stage, rows, lane);
            __syncthreads();                                        // product W1 is done, W1^T has been used
            put_planes<P>(p_dy, row, h, f);
            {
                Frags<P> fx;
                make_frags(fx, t);
                put_planes<P>(p_x, row, h, fx);
            }
            __syncthreads();                                        // planes of Wo; Wo^T
            if (P == 1) fetch_next();      // float32 has the registers only after the products
            zero(g);
            gemm<P>(g, f, w, lane);                                 // da, beside product Wo
            __syncthreads();                                        // Wo^T has been used
            put_rows(reinterpret_cast<T*>(a.d_attn), g, stage, rows, lane);
            if (a.nd && n < rows.left) put_node_side<T>(g, t, a.Z, a.nd, a.heads, rows.first + n, h);
            if (P != 1) fetch_next();
        }
    } else {
        const int q = wave - 4, base_dy = operand_base(q >> 1, lane), base_x = operand_base(q & 1, lane);
        const vec16 *fw = reinterpret_cast<const vec16*>(a.w_post), *bw = reinterpret_cast<const vec16*>(a.w_back);
        WeightsAhead<FV> next;
        next.fetch(fw);
        for (int64_t g0 = blockIdx.x; g0 < groups; g0 += gridDim.x) {
            next.hand_over(w, fw + FV);             // Wo, then on to W1
            __syncthreads();
            next.hand_over(w, bw + 2 * FV);         // W1
            __syncthreads();
            next.hand_over(w, bw + FV);             // W2^T and the planes of W2
            node_product<P>(acc[2], p_dy, p_x, base_dy, base_x);
            __syncthreads();
            next.hand_over(w, bw);                  // W1^T and the planes of W1
            node_product<P>(acc[1], p_dy, p_x, base_dy, base_x);
            __syncthreads();
            next.hand_over(w, fw);                  // Wo^T and the planes of Wo
            node_product<P>(acc[0], p_dy, p_x, base_dy, base_x);
            __syncthreads();
        }
    }
    write_partial<3, 5>(a.partial + (int64_t)blockIdx.x * (3 * 4096 + 5 * 64), acc, col, reinterpret_cast<float*>(smem), wave, lane);
}

// ---- sums of the partials -----------------------------------------------------------------------------------------------
constexpr int kMaxSums = 26, kMaxOut = 8;
struct SumArgs {
    const float* partial[kMaxSums];
    int workers[kMaxSums], n[kMaxSums];
    void* out[kMaxSums][kMaxOut];      // mats x 4096 elements, then vectors of 64 (a null entry is not wanted)
    int16_t mats[kMaxSums], rows[kMaxSums], ld[kMaxSums];   // rows: of the 64 in each matrix and the vectors that follow them (classes)
};
__device__ __forceinline__ void put_elem(float* p, float v) { *p = v; }
__device__ __forceinline__ void put_elem(nbf16* p, float v) { p->x = __builtin_bit_cast(uint16_t, static_cast<__bf16>(v)); }

// 64 consecutive elements x 16 slices of the workers per workgroup: slices in worker order, then the slice sums in order
template <typename T> __global__ __launch_bounds__(1024) void k_node_sums(const SumArgs a) {
    __shared__ float part[16][64];
    const int d = blockIdx.y, n = a.n[d];
    if ((int)blockIdx.x * 64 >= n) return;
    const int el = threadIdx.x & 63, sl = threadIdx.x >> 6, e = blockIdx.x * 64 + el;
    const int w0 = a.workers[d] * sl / 16, w1 = a.workers[d] * (sl + 1) / 16;
    const float* __restrict__ src = a.partial[d] + e;
    float s = 0.f;
    int w = w0;
    for (; w + 8 <= w1; w += 8) {
        float t[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) t[i] = src[(int64_t)(w + i) * n];
#pragma unroll
        for (int i = 0; i < 8; ++i) s += t[i];
    }
    for (; w < w1; ++w) s += src[(int64_t)w * n];
    part[sl][el] = s;
    __syncthreads();
    if (sl == 0) {
        float t = 0.f;
#pragma unroll
        for (int i = 0; i < 16; ++i) t += part[i][el];
        const int mats = a.mats[d], rows = a.rows[d];
        const int seg = e < mats * 4096 ? e >> 12 : mats + ((e - mats * 4096) >> 6), at = e < mats * 4096 ? e & 4095 : (e - mats * 4096) & 63;
        const int limit = seg < mats ? rows * 64 : (seg < 2 * mats ? rows : 64);
        if (a.out[d][seg] && at < limit) put_elem(reinterpret_cast<T*>(a.out[d][seg]) + (seg < mats ? (at >> 6) * a.ld[d] + (at & 63) : at), t);
    }
}

template <typename T, bool SAME, bool POST, int NEXT> int launch_fwd(const tgt_node_fwd_args& a, hipStream_t st) {
    static std::atomic<uint64_t> done{0};
    return launch(&k_node_fwd<T, SAME, POST, NEXT>, done, grid_for(a.rows, fwd_waves<T, SAME>()), fwd_waves<T, SAME>() * 64, fwd_lds<T, SAME, POST, NEXT>(), st, a);
}
template <typename T, bool SAME> int dispatch_fwd(const tgt_node_fwd_args& a, hipStream_t st) {
    if (a.attn) return a.logp ? launch_fwd<T, SAME, true, NEXT_CLASSES>(a, st) : (a.q ? launch_fwd<T, SAME, true, NEXT_QKV>(a, st) : launch_fwd<T, SAME, true, NEXT_NONE>(a, st));
    return launch_fwd<T, SAME, false, NEXT_QKV>(a, st);
}
template <typename T> int dispatch_bwd_pre(const tgt_node_bwd_pre_args& a, int workers, hipStream_t st) {
    static std::atomic<uint64_t> done[3];
    if (a.dlogp) return launch(&k_node_bwd_pre<T, true, true>, done[1], workers, kBwdThreads, BwdLds<T>::kBytes, st, a);
    return a.v_next ? launch(&k_node_bwd_pre<T, false, true>, done[0], workers, kBwdThreads, BwdLds<T>::kBytes, st, a)
                    : launch(&k_node_bwd_pre<T, false, false>, done[2], workers, kBwdThreads, BwdLds<T>::kBytes, st, a);
}
template <typename T, bool SAME> int dispatch_bwd_post(const tgt_node_bwd_post_args& a, int workers, hipStream_t st) {
    static std::atomic<uint64_t> done{0};
    return launch(&k_node_bwd_post<T, SAME>, done, workers, kBwdThreads, BwdLds<T>::kBytes, st, a);
}
bool dtype_ok(int dtype) { return dtype == TGT_DTYPE_F32 || dtype == TGT_DTYPE_BF16; }

}  // namespace
}  // namespace tgt

extern "C" {

int64_t tgt_node_frag_bytes(int n_mats, int dtype) {
    if (n_mats < 0 || !tgt::dtype_ok(dtype)) return -1;
    return 2ll * n_mats * 16 * (dtype == TGT_DTYPE_F32 ? tgt::kFragVecs<3> : tgt::kFragVecs<1>);
}

int tgt_node_pack(const void* const* mats, const int* ld, const int* rows, int n_mats, const void* const* vecs, const int* lens, int n_vecs,
                  int dtype, void* d_frags, float* d_vecs, void* stream) {
    using namespace tgt;
    if (!mats || !ld || !rows || !vecs || !lens || n_mats < 1 || n_vecs < 1 || !d_frags || !d_vecs || !dtype_ok(dtype)) return bad("tgt_node_pack", "null or bad argument");
    for (int i = 0; i < n_mats; ++i)
        if (!mats[i] || rows[i] < 1 || rows[i] > 64 || ld[i] < 64 || ld[i] > 32767) return bad("tgt_node_pack", "weights are [1..64, >= 64]");
    for (int i = 0; i < n_vecs; ++i)
        if (!vecs[i] || lens[i] < 1 || lens[i] > 64) return bad("tgt_node_pack", "vectors have 1 to 64 elements");
    KernelTimer t(KS_NODE_PACK, (hipStream_t)stream);
    for (int m = 0, v = 0; m < n_mats || v < n_vecs;) {
        PackArgs a{};
        a.n_mats = std::min(kPackMats, n_mats - m); a.n_vecs = std::min(kPackVecs, n_vecs - v);
        a.mat0 = m; a.vec0 = v; a.total_mats = n_mats;
        a.frags = (vec16*)d_frags; a.vecs = d_vecs;
        for (int i = 0; i < a.n_mats; ++i) { a.mat[i] = mats[m + i]; a.ld[i] = (int16_t)ld[m + i]; a.rows[i] = (int16_t)rows[m + i]; }
        for (int i = 0; i < a.n_vecs; ++i) { a.vec[i] = vecs[v + i]; a.len[i] = (int16_t)lens[v + i]; }
        const int grid = 2 * a.n_mats + (a.n_vecs + 7) / 8;
        if (dtype == TGT_DTYPE_F32) hipLaunchKernelGGL((k_node_pack<float>), dim3(grid), dim3(512), 0, (hipStream_t)stream, a);
        else hipLaunchKernelGGL((k_node_pack<nbf16>), dim3(grid), dim3(512), 0, (hipStream_t)stream, a);
        TGT_HIP_CHECK(hipGetLastError());
        m += a.n_mats; v += a.n_vecs;
    }
    return TGT_OK;
}

int tgt_node_fwd(const tgt_node_fwd_args* a, void* stream) {
    using namespace tgt;
    if (!a || a->rows < 0 || !dtype_ok(a->dtype) || !a->s_in) return bad("tgt_node_fwd", "null or bad argument");
    if (a->attn ? (!a->s_out || !a->w_post || !a->v_post) : !a->q) return bad("tgt_node_fwd", "attention rows need s_out, w_post, v_post; without them q, k, v are needed");
    if (a->q && (!a->k || !a->v || !a->w_next || !a->v_next || a->logp)) return bad("tgt_node_fwd", "q needs k, v, w_next, v_next and no logp");
    if (a->logp && (!a->attn || !a->w_next || !a->v_next || a->classes < 1 || a->classes > 64)) return bad("tgt_node_fwd", "logp needs attention rows, w_next, v_next and 1 to 64 classes");
    if (a->tokens < 0 || (!a->attn && a->tokens > 0 && (!a->token || !a->s_out))) return bad("tgt_node_fwd", "tokens need their table and s_out");
    if (a->rows == 0) return TGT_OK;
    KernelTimer t(KS_NODE_FWD, (hipStream_t)stream);
    const hipStream_t st = (hipStream_t)stream;
    if (a->dtype == TGT_DTYPE_F32) return dispatch_fwd<float, false>(*a, st);
    return a->same_bits ? dispatch_fwd<nbf16, true>(*a, st) : dispatch_fwd<nbf16, false>(*a, st);
}

int tgt_node_bwd_workers(int64_t rows) { return rows < 0 ? -1 : tgt::grid_for(rows, 4); }

int tgt_node_bwd_pre(const tgt_node_bwd_pre_args* a, void* stream) {
    using namespace tgt;
    if (!a || a->rows < 1 || !dtype_ok(a->dtype) || !a->s || !a->g_out || !a->w_back || (a->dlogp && !a->v_next) || !a->partial) return bad("tgt_node_bwd_pre", "null or bad argument");
    if (a->dlogp ? ((!a->logp && !a->linear) || a->classes < 1 || a->classes > 64 || a->tokens < 0) : (!a->dq || !a->dk || !a->dv || !a->g_in))
        return bad("tgt_node_bwd_pre", "dq, dk, dv, g_in or dlogp, logp and 1 to 64 classes are needed");
    KernelTimer t(KS_NODE_BWD_PRE, (hipStream_t)stream);
    const int workers = grid_for(a->rows, 4);
    return a->dtype == TGT_DTYPE_F32 ? dispatch_bwd_pre<float>(*a, workers, (hipStream_t)stream) : dispatch_bwd_pre<nbf16>(*a, workers, (hipStream_t)stream);
}

int tgt_node_bwd_post(const tgt_node_bwd_post_args* a, void* stream) {
    using namespace tgt;
    if (!a || a->rows < 1 || !dtype_ok(a->dtype) || !a->s || !a->attn || !a->g_in || !a->g_out || !a->d_attn || !a->w_post || !a->w_back || !a->v_post || !a->partial)
        return bad("tgt_node_bwd_post", "null or bad argument");
    if (a->nd && (!a->Z || (a->heads != 8 && a->heads != 4 && a->heads != 2))) return bad("tgt_node_bwd_post", "nd needs Z and 8, 4 or 2 heads");
    KernelTimer t(KS_NODE_BWD_POST, (hipStream_t)stream);
    const hipStream_t st = (hipStream_t)stream;
    const int workers = grid_for(a->rows, 4);
    if (a->dtype == TGT_DTYPE_F32) return dispatch_bwd_post<float, false>(*a, workers, st);
    return a->same_bits ? dispatch_bwd_post<nbf16, true>(*a, workers, st) : dispatch_bwd_post<nbf16, false>(*a, workers, st);
}

int tgt_node_sums(const tgt_node_sum* sums, int count, int dtype, void* stream) {
    using namespace tgt;
    if (!sums || count < 1 || !dtype_ok(dtype)) return bad("tgt_node_sums", "null or bad argument");
    KernelTimer t(KS_NODE_SUMS, (hipStream_t)stream);
    for (int c = 0; c < count; c += kMaxSums) {
        SumArgs a{};
        const int m = std::min(kMaxSums, count - c);
        int longest = 0;
        for (int i = 0; i < m; ++i) {
            const tgt_node_sum& s = sums[c + i];
            if (!s.partial || s.workers < 1 || s.mats < 1 || s.mats > 3 || s.rows < 1 || s.rows > 64 || s.ld < 0 || s.ld > 32767) return bad("tgt_node_sums", "bad descriptor");
            a.partial[i] = s.partial; a.workers[i] = s.workers; a.mats[i] = (int16_t)s.mats; a.rows[i] = (int16_t)s.rows; a.ld[i] = (int16_t)(s.ld ? s.ld : 64);
            a.n[i] = s.mats * 4096 + (s.mats + 2) * 64;
            for (int o = 0; o < 2 * s.mats + 2; ++o) a.out[i][o] = s.out[o];
            longest = std::max(longest, a.n[i]);
        }
        const dim3 grid((unsigned)(longest / 64), (unsigned)m);
        if (dtype == TGT_DTYPE_F32) hipLaunchKernelGGL((k_node_sums<float>), grid, dim3(1024), 0, (hipStream_t)stream, a);
        else hipLaunchKernelGGL((k_node_sums<nbf16>), grid, dim3(1024), 0, (hipStream_t)stream, a);
        TGT_HIP_CHECK(hipGetLastError());
    }
    return TGT_OK;
}

}  // extern "C"
