// Dense biased attention in float32 arithmetic, for float32 callers.
//
// The reference's dense CoreAttention.forward (models/graphormer_graph_level.py:186-214, attn_module.py:99-127)
// computes in float32:  x = (q * sqrt(d)) k^T + attn_bias ; softmax over keys ; dropout ; x v.  The matrix-core
// kernels of dense_attn.hip round their operands to bf16, which costs 2^-8 on logits that the reference's
// q * sqrt(d) makes large; a float32 caller who has not asked for that gets these kernels instead: float32
// products and sums, fp32 softmax with the accurate exponential.  A probability has the rounding of its score, 2^-24 of up to 4.5 d for q and k of
// unit variance, a few times over; against a float64 evaluation the results are off by at most, of the largest value, 5e-6 with 8 features, 6e-6 with 16 and
// 1.6e-5 with 32 (measured at 13 to 256 rows; the tests allow 1e-5, 1e-5 and 2e-5).  Not where a row's dS is the difference of nearly equal numbers in all
// rows that make up a gradient (all weight on one key of two: gradients of 2^-24 of their terms, right in absolute size only).
//
// Up to 256 rows (192 with a head dim of 32) the products go to the float32 matrix instructions (k_dense_f32_mm_*, below), a wave per
// tile of sixteen queries (forward) or keys (backward).  What follows is about the other two kernels, on the vector units.
//
// One workgroup per (graph, head).  Forward: K and V of the head sit in LDS, a thread owns one query row and
// walks the keys with an online softmax; every LDS read of K / V is a broadcast.  A thread that read its own
// bias row from memory would touch a different cache line in every lane, so the bias comes in strips of 32
// keys: the workgroup loads the strip [S queries][32 keys] with coalesced reads into LDS and every thread
// then takes its row from there (and, in the backward, leaves its row of dBias there for a coalesced write).
// Backward: a first walk with thread = query gives dQ and dBias, a second with thread = key gives dK and dV
// (its bias reads are coalesced over the threads as they are); both recompute the probabilities from the
// saved log-sum-exp.
#include "common.h"
#include "dense_dropout.h"
#include <algorithm>

namespace tgt {

constexpr int kF32Block = 256;
constexpr int kF32Chunk = 8;        // keys between two rescalings of the online softmax
constexpr int kF32Strip = 32;       // keys of one bias strip
constexpr int kF32StripLd = 33;     // its row stride in LDS (odd: rows of consecutive queries start in different banks)

// bias[q, k0 .. k0 + 32) for the queries q0 .. q1 - 1 -> strip[q][.] (zeros past the end of a row); coalesced
__device__ __forceinline__ void load_strip(const float* __restrict__ bias_gh, int S, int q0, int q1, int k0,
                                           float* __restrict__ strip) {
    for (int i = threadIdx.x; i < (q1 - q0) * kF32Strip; i += blockDim.x) {
        const int r = q0 + i / kF32Strip, c = i % kF32Strip;
        strip[r * kF32StripLd + c] = (k0 + c < S) ? bias_gh[(int64_t)r * S + k0 + c] : 0.f;
    }
}
__device__ __forceinline__ void store_strip(float* __restrict__ dbias_gh, int S, int q0, int q1, int k0,
                                            const float* __restrict__ strip) {
    for (int i = threadIdx.x; i < (q1 - q0) * kF32Strip; i += blockDim.x) {
        const int r = q0 + i / kF32Strip, c = i % kF32Strip;
        if (k0 + c < S) dbias_gh[(int64_t)r * S + k0 + c] = strip[r * kF32StripLd + c];
    }
}

template <int D>
__device__ __forceinline__ void ld_row(const float* __restrict__ p, float (&x)[D]) {
#pragma unroll
    for (int c = 0; c < D; c += 4) {
        const float4 v = *reinterpret_cast<const float4*>(p + c);
        x[c] = v.x; x[c + 1] = v.y; x[c + 2] = v.z; x[c + 3] = v.w;
    }
}
template <int D>
__device__ __forceinline__ void st_row(float* __restrict__ p, const float (&x)[D], float f) {
#pragma unroll
    for (int c = 0; c < D; c += 4) *reinterpret_cast<float4*>(p + c) = make_float4(x[c] * f, x[c + 1] * f, x[c + 2] * f, x[c + 3] * f);
}
template <int D>
__device__ __forceinline__ float dotf(const float (&a)[D], const float* __restrict__ b) {
    float t = 0.f;
#pragma unroll
    for (int c = 0; c < D; ++c) t = fmaf(a[c], b[c], t);
    return t;
}

// X[g, :, h, :] -> LDS [S][D], optionally scaled
template <int D>
__device__ __forceinline__ void stage_head(const float* __restrict__ X, int g, int h, int S, int H, float f,
                                           float* __restrict__ dst) {
    for (int c = threadIdx.x; c < S * (D / 4); c += blockDim.x) {
        const int row = c / (D / 4), part = c % (D / 4);
        float4 v = *reinterpret_cast<const float4*>(X + (((int64_t)g * S + row) * H + h) * D + part * 4);
        v.x *= f; v.y *= f; v.z *= f; v.w *= f;
        *reinterpret_cast<float4*>(dst + row * D + part * 4) = v;
    }
}

// workgroup -> (graph, head): the H heads of a graph share every line of q/k/v, so they get workgroup ids that
// are congruent modulo 8 (same XCD, same L2) inside a window of 8 * H ids
__device__ __forceinline__ bool pair_of_block(int nb, int H, int& g, int& h) {
    const int win = blockIdx.x / (8 * H), rem = blockIdx.x % (8 * H);
    g = win * 8 + (rem & 7);
    h = rem >> 3;
    return g < nb;
}

template <int D, bool DROP>
__global__ __launch_bounds__(kF32Block) void k_dense_f32_fwd(const float* __restrict__ Q, const float* __restrict__ K,
                                                             const float* __restrict__ V, const float* __restrict__ bias,
                                                             float* __restrict__ out, float* __restrict__ lse, int S, int H,
                                                             float scale, int nb, const DropArgs da) {
    extern __shared__ __align__(16) char smem[];
    float* k_l = reinterpret_cast<float*>(smem);
    float* v_l = k_l + S * D;
    float* strip = v_l + S * D;                      // [S][kF32StripLd]
    int g, h;
    if (!pair_of_block(nb, H, g, h)) return;
    stage_head<D>(K, g, h, S, H, 1.0f, k_l);
    stage_head<D>(V, g, h, S, H, 1.0f, v_l);
    const float* bias_gh = bias ? bias + ((int64_t)g * H + h) * S * S : nullptr;
    // a thread owns query qi = threadIdx.x + 256 * pass; all threads take part in the strip loads of every pass
    for (int q0 = 0; q0 < S; q0 += blockDim.x) {
        const int qi = q0 + threadIdx.x;
        const bool qok = qi < S;
        float qs[D], o[D];
#pragma unroll
        for (int c = 0; c < D; ++c) { qs[c] = 0.f; o[c] = 0.f; }
        if (qok) ld_row<D>(Q + (((int64_t)g * S + qi) * H + h) * D, qs);
#pragma unroll
        for (int c = 0; c < D; ++c) qs[c] *= scale;      // the reference scales q before the product
        const uint32_t rh = DROP ? drop_row_hash(da, g * H + h, qi) : 0u;
        float m = -INFINITY, l = 0.f;
        for (int s0 = 0; s0 < S; s0 += kF32Strip) {
            __syncthreads();                             // K / V staged; the previous strip is consumed
            if (bias_gh) load_strip(bias_gh, S, q0, min(S, q0 + (int)blockDim.x), s0, strip);
            __syncthreads();
            if (!qok) continue;
            const float* brow = strip + qi * kF32StripLd;
#pragma unroll 1
            for (int k0 = s0; k0 < min(S, s0 + kF32Strip); k0 += kF32Chunk) {
                float sc[kF32Chunk], cm = -INFINITY;
#pragma unroll
                for (int j = 0; j < kF32Chunk; ++j) {
                    const int k = k0 + j;
                    sc[j] = -INFINITY;
                    if (k < S) sc[j] = dotf<D>(qs, k_l + k * D) + (bias_gh ? brow[k - s0] : 0.f);
                    cm = fmaxf(cm, sc[j]);
                }
                const float m_new = fmaxf(m, cm);
                const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
                const float alpha = expf(m - m_use);           // m = -inf: 0
                l *= alpha;
#pragma unroll
                for (int c = 0; c < D; ++c) o[c] *= alpha;
#pragma unroll
                for (int j = 0; j < kF32Chunk; ++j) {
                    const int k = k0 + j;
                    if (k < S) {
                        const float p = expf(sc[j] - m_use);
                        l += p;
                        const float pk = (!DROP || drop_keep(da, rh, k)) ? p : 0.f;
                        const float* vr = v_l + k * D;
#pragma unroll
                        for (int c = 0; c < D; ++c) o[c] = fmaf(pk, vr[c], o[c]);
                    }
                }
                m = m_new;
            }
        }
        if (qok) {
            st_row<D>(out + (((int64_t)g * S + qi) * H + h) * D, o, (DROP ? da.inv_keep : 1.0f) / l);
            lse[((int64_t)g * H + h) * S + qi] = (m == -INFINITY ? 0.f : m) + logf(l);
        }
    }
}

template <int D, bool DROP>
__global__ __launch_bounds__(kF32Block) void k_dense_f32_bwd(const float* __restrict__ Q, const float* __restrict__ K,
                                                             const float* __restrict__ V, const float* __restrict__ bias,
                                                             const float* __restrict__ O, const float* __restrict__ lse,
                                                             const float* __restrict__ dO, float* __restrict__ dQ,
                                                             float* __restrict__ dK, float* __restrict__ dV,
                                                             float* __restrict__ dbias, int S, int H, float scale, int nb,
                                                             const DropArgs da) {
    extern __shared__ __align__(16) char smem[];
    float* q_l = reinterpret_cast<float*>(smem);     // q * sqrt(d)
    float* k_l = q_l + S * D;
    float* v_l = k_l + S * D;
    float* g_l = v_l + S * D;                        // dout
    float* lse_l = g_l + S * D;
    float* dd_l = lse_l + S;                         // sum_c dout[q, c] out[q, c]
    float* strip = dd_l + S;                         // [S][kF32StripLd] bias in, dBias out
    int g, h;
    if (!pair_of_block(nb, H, g, h)) return;
    stage_head<D>(Q, g, h, S, H, scale, q_l);
    stage_head<D>(K, g, h, S, H, 1.0f, k_l);
    stage_head<D>(V, g, h, S, H, 1.0f, v_l);
    stage_head<D>(dO, g, h, S, H, 1.0f, g_l);
    for (int i = threadIdx.x; i < S; i += blockDim.x) {
        float ov[D], gv[D];
        ld_row<D>(O + (((int64_t)g * S + i) * H + h) * D, ov);
        ld_row<D>(dO + (((int64_t)g * S + i) * H + h) * D, gv);
        float t = 0.f;
#pragma unroll
        for (int c = 0; c < D; ++c) t = fmaf(ov[c], gv[c], t);
        dd_l[i] = t;
        lse_l[i] = lse[((int64_t)g * H + h) * S + i];
    }
    __syncthreads();
    const float* bias_gh = bias ? bias + ((int64_t)g * H + h) * S * S : nullptr;
    float* dbias_gh = dbias ? dbias + ((int64_t)g * H + h) * S * S : nullptr;
    // thread = query: dQ and the query's row of dBias, strip by strip
    for (int q0 = 0; q0 < S; q0 += blockDim.x) {
        const int qi = q0 + threadIdx.x;
        const bool qok = qi < S;
        float qs[D], gv[D], dq[D];
#pragma unroll
        for (int c = 0; c < D; ++c) { qs[c] = qok ? q_l[qi * D + c] : 0.f; gv[c] = qok ? g_l[qi * D + c] : 0.f; dq[c] = 0.f; }
        const float L = qok ? lse_l[qi] : 0.f, Dq = qok ? dd_l[qi] : 0.f;
        const uint32_t rh = DROP ? drop_row_hash(da, g * H + h, qi) : 0u;
        for (int s0 = 0; s0 < S; s0 += kF32Strip) {
            __syncthreads();                             // the previous strip is written out
            if (bias_gh) load_strip(bias_gh, S, q0, min(S, q0 + (int)blockDim.x), s0, strip);
            __syncthreads();
            if (qok) {
                float* brow = strip + qi * kF32StripLd;
                for (int k = s0; k < min(S, s0 + kF32Strip); ++k) {
                    const float b = bias_gh ? brow[k - s0] : 0.f;
                    const float p = expf(dotf<D>(qs, k_l + k * D) + b - L);
                    const float ks = !DROP ? 1.0f : (drop_keep(da, rh, k) ? da.inv_keep : 0.f);
                    const float dS = p * (dotf<D>(gv, v_l + k * D) * ks - Dq);
                    brow[k - s0] = dS;                   // this thread's own row: the strip now holds dBias
                    const float* kr = k_l + k * D;
#pragma unroll
                    for (int c = 0; c < D; ++c) dq[c] = fmaf(dS, kr[c], dq[c]);
                }
            }
            if (dbias_gh) {
                __syncthreads();
                store_strip(dbias_gh, S, q0, min(S, q0 + (int)blockDim.x), s0, strip);
            }
        }
        if (qok) st_row<D>(dQ + (((int64_t)g * S + qi) * H + h) * D, dq, scale);
    }
    __syncthreads();
    // thread = key: dK and dV (the bias element of (query, key) is read by consecutive threads for one query)
    for (int ki = threadIdx.x; ki < S; ki += blockDim.x) {
        float kv[D], vv[D], dk[D], dv[D];
#pragma unroll
        for (int c = 0; c < D; ++c) { kv[c] = k_l[ki * D + c]; vv[c] = v_l[ki * D + c]; dk[c] = 0.f; dv[c] = 0.f; }
        for (int qq = 0; qq < S; ++qq) {
            const float b = bias_gh ? bias_gh[(int64_t)qq * S + ki] : 0.f;
            const float* qr = q_l + qq * D;
            const float* gr = g_l + qq * D;
            const float p = expf(dotf<D>(kv, qr) + b - lse_l[qq]);
            const float ks = !DROP ? 1.0f : (drop_keep(da, drop_row_hash(da, g * H + h, qq), ki) ? da.inv_keep : 0.f);
            const float dS = p * (dotf<D>(vv, gr) * ks - dd_l[qq]);
            const float pk = p * ks;
#pragma unroll
            for (int c = 0; c < D; ++c) {
                dk[c] = fmaf(dS, qr[c], dk[c]);      // qr holds q * sqrt(d): d s / d k
                dv[c] = fmaf(pk, gr[c], dv[c]);
            }
        }
        st_row<D>(dK + (((int64_t)g * S + ki) * H + h) * D, dk, 1.0f);
        st_row<D>(dV + (((int64_t)g * S + ki) * H + h) * D, dv, 1.0f);
    }
}

// ---- on the matrix instructions ------------------------------------------------------------------------------------------
// v_mfma_f32_16x16x4_f32: A[i][k] and B[k][j] in lane i (j) + 16 k, C[4 g + t][j] in register t of lane j + 16 g; float32 products, the running sum
// rounded no more often than by a chain of fmas.  The contractions over queries and keys take their steps in the order in which C leaves
// them: register t is the B operand of a step over the rows 4 k + t.
//
// With a thread per query row 65 rows kept 65 of 256 threads busy, and every element read the row of K (and V) from LDS twice, once for the
// thread's query and once for its key.  Here a wave has sixteen rows, all of them work, the bias and its gradient go between memory and registers in
// rows of 64 bytes, and the backward forms a probability once.  us, 8 heads of 8, thread per row / this, forward and backward: 256 graphs of
// 13 rows 7.6 / 5.3, 13.5 / 6.9; of 41 16.4 / 12.2, 40.8 / 18.7; of 129 120 / 64, 304 / 128 (bias and gradient alone, 136 MB each, 26 and 53 at
// the rate of a large copy); 64 of 201 101 / 33, 223 / 60; 4 of 129 38 / 12, 87 / 19; heads of 32, 64 of 65 rows 35 / 14, 91 / 27.  (Forward: a lane's four keys
// of the bias in one load wherever they begin; in four, 71 and 39 where it says 65 and 34.)  Errors against 64 bits
// a tenth smaller (256 graphs of 41 rows, of the norm: out 1.29e-7 / 1.40e-7 before, dq 2.1e-7 / 2.2e-7, dbias 1.9e-7 / 2.0e-7).
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));      // 16 bytes that begin at any float
__device__ __forceinline__ f32x4_t mma4(float a, float b, f32x4_t c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
constexpr int kMmTiles = 16;        // tiles of sixteen rows, a wave each
template <int D> struct Mm {
    // row stride in LDS (an odd number of fours: the reads of four features of sixteen rows and of sixteen features of every fourth row both meet every
    // bank once), blocks of sixteen features, steps over them; row stride of a wave's tile (likewise)
    static constexpr int LD = D + 4, DB = (D + 15) / 16, KS = D / 4, TD = 20;
    static int tiles(int S) { return (S + 15) / 16; }
    static int fwd_lds(int S) { return 2 * 16 * tiles(S) * LD * 4; }
    // each: the shares of dQ are added up after every step of queries (two steps' shares in LDS), else all of them at the end
    static int bwd_lds(int S, bool each) {
        const int n = tiles(S), rows = 16 * n;
        static_assert(16 * TD <= 2 * 16 * LD, "the waves' tiles in the place of K and V");
        return (n * (each ? 32 : rows) * D + 2 * rows + 4 * rows * LD) * 4;
    }
    static bool fits(int S) { return S > 0 && tiles(S) <= kMmTiles && bwd_lds(S, true) <= 160 * 1024; }
    // X[g, :, h, :] -> LDS [rows][LD], rows behind S are zero
    static __device__ __forceinline__ void stage(const float* __restrict__ X, int g, int h, int S, int H, float f, float* __restrict__ dst, int rows) {
        for (int c = threadIdx.x; c < rows * KS; c += blockDim.x) {
            const int row = c / KS, part = c % KS;
            float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
            if (row < S) v = *reinterpret_cast<const float4*>(X + (((int64_t)g * S + row) * H + h) * D + part * 4);
            *reinterpret_cast<float4*>(dst + row * LD + part * 4) = make_float4(v.x * f, v.y * f, v.z * f, v.w * f);
        }
    }
};

// Wave w: the queries 16 w ..., a lane's query is its column; 32 keys between two rescalings.
template <int D, bool DROP>
__global__ __launch_bounds__(64 * kMmTiles) void k_dense_f32_mm_fwd(const float* __restrict__ Q, const float* __restrict__ K, const float* __restrict__ V,
                                                                    const float* __restrict__ bias, float* __restrict__ out, float* __restrict__ lse, int S, int H,
                                                                    float scale, int nb, const DropArgs da) {
    using M = Mm<D>;
    constexpr int LD = M::LD, DB = M::DB, KS = M::KS;
    extern __shared__ __align__(16) char smem[];
    const int rows = blockDim.x / 4;
    float *k_l = reinterpret_cast<float*>(smem), *v_l = k_l + rows * LD;
    int g, h;
    if (!pair_of_block(nb, H, g, h)) return;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c = lane & 15, gr = lane >> 4, cd = c % D;
    const int qi = wave * 16 + c, qrow = min(qi, S - 1);
    const float* brow = bias ? bias + (((int64_t)g * H + h) * S + qrow) * S : nullptr;
    // the lane's bias of keys k + 16 u + 4 gr + t
    const auto ask = [&](int k, float (&b)[8]) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int key = k + 16 * u + 4 * gr;
            if (!brow) {
#pragma unroll
                for (int t = 0; t < 4; ++t) b[4 * u + t] = 0.f;
            } else if (k + 16 * u + 16 <= S) {
                const f32x4_any v = *reinterpret_cast<const f32x4_any*>(brow + key);
#pragma unroll
                for (int t = 0; t < 4; ++t) b[4 * u + t] = v[t];
            } else {
#pragma unroll
                for (int t = 0; t < 4; ++t) b[4 * u + t] = brow[min(key + t, S - 1)];
            }
        }
    };
    float next[8], q[KS];
    ask(0, next);
#pragma unroll
    for (int s = 0; s < KS; ++s) q[s] = Q[(((int64_t)g * S + qrow) * H + h) * D + 4 * s + gr] * scale;      // the reference scales q before the product
    M::stage(K, g, h, S, H, 1.0f, k_l, rows);
    M::stage(V, g, h, S, H, 1.0f, v_l, rows);
    __syncthreads();
    const uint32_t rh = DROP ? drop_row_hash(da, g * H + h, qi) : 0u;
    float m = -INFINITY, l = 0.f;
    f32x4_t o[DB];
#pragma unroll
    for (int i = 0; i < DB; ++i) o[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < S; k0 += 32) {
        float sc[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) sc[i] = next[i];
        if (k0 + 32 < S) ask(k0 + 32, next);
        float cm = -INFINITY;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int k = k0 + 16 * u;
            f32x4_t a = {0.f, 0.f, 0.f, 0.f};
            if (k < S) {
#pragma unroll
                for (int s = 0; s < KS; ++s) a = mma4(k_l[(k + c) * LD + 4 * s + gr], q[s], a);
            }
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                sc[4 * u + t] = k + 4 * gr + t < S ? a[t] + sc[4 * u + t] : -INFINITY;
                cm = fmaxf(cm, sc[4 * u + t]);
            }
        }
        cm = fmaxf(cm, __shfl_xor(cm, 16));
        cm = fmaxf(cm, __shfl_xor(cm, 32));
        const float m_new = fmaxf(m, cm), m_use = (m_new == -INFINITY) ? 0.f : m_new;
        const float alpha = expf(m - m_use);           // m = -inf: 0
        l *= alpha;
#pragma unroll
        for (int i = 0; i < DB; ++i) o[i] *= alpha;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int k = k0 + 16 * u;
            if (k >= S) break;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const float p = expf(sc[4 * u + t] - m_use);
                if (k + 4 * gr + t < S) l += p;
                const float pk = k + 4 * gr + t < S && (!DROP || drop_keep(da, rh, k + 4 * gr + t)) ? p : 0.f;
#pragma unroll
                for (int i = 0; i < DB; ++i) o[i] = mma4(v_l[(k + 4 * gr + t) * LD + 16 * i + cd], pk, o[i]);
            }
        }
        m = m_new;
    }
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);
    if (qi >= S) return;
    const float f = (DROP ? da.inv_keep : 1.0f) / l;
#pragma unroll
    for (int i = 0; i < DB; ++i)
        if (D >= 16 || 4 * gr < D)
            *reinterpret_cast<float4*>(out + (((int64_t)g * S + qi) * H + h) * D + 16 * i + 4 * gr) = make_float4(o[i][0] * f, o[i][1] * f, o[i][2] * f, o[i][3] * f);
    if (gr == 0) lse[((int64_t)g * H + h) * S + qi] = (m == -INFINITY ? 0.f : m) + logf(l);
}

// Wave w: the keys 16 w ..., a lane's key is its column, against one tile of queries after the other: dK and dV in registers; dS through a tile in
// LDS of the wave's own, with rows and columns changed, for its share of dQ, which waits in LDS for the others'.  EACH: until the end of the step, behind a
// barrier, where a wave adds the step's shares up, the next one the next step's; else until the end.  All shares are 4 D S bytes a wave and keep other workgroups
// off the CU: to the end where three of them fit it all the same (48 KB), or where there is no more than one for a CU.  us, at the end / EACH: 8 heads of 8, 128
// graphs of 65 rows (27 KB) 21.8 / 23.4, 256 of 129 (70 KB) 128.1 / 128.7, 64 of 201 (129 KB) 65.8 / 59.9, 4 of 129 18.6 / 20.4; heads of 16, 128 of 65 (52 KB)
// 28.6 / 26.7, 200 of 151 177 / 157; of 32, 64 of 65 (98 KB) 35.4 / 27.2.
template <int D, bool DROP, bool EACH>
__global__ __launch_bounds__(64 * kMmTiles) void k_dense_f32_mm_bwd(const float* __restrict__ Q, const float* __restrict__ K, const float* __restrict__ V,
                                                                    const float* __restrict__ bias, const float* __restrict__ O, const float* __restrict__ lse,
                                                                    const float* __restrict__ dO, float* __restrict__ dQ, float* __restrict__ dK, float* __restrict__ dV,
                                                                    float* __restrict__ dbias, int S, int H, float scale, int nb, const DropArgs da) {
    using M = Mm<D>;
    constexpr int LD = M::LD, DB = M::DB, KS = M::KS, TD = M::TD;
    extern __shared__ __align__(16) char smem[];
    const int rows = blockDim.x / 4, waves = blockDim.x / 64;
    float* part = reinterpret_cast<float*>(smem);      // shares of dQ: EACH two steps' [wave][16][D], else [wave][rows][D]
    float* lse_l = part + waves * (EACH ? 32 : rows) * D;
    float* dd_l = lse_l + rows;                        // sum_c dout[q, c] out[q, c]
    float* q_l = dd_l + rows;                          // q * sqrt(d)
    float* g_l = q_l + rows * LD;                      // dout
    float* k_l = g_l + rows * LD;
    float* v_l = k_l + rows * LD;
    int g, h;
    if (!pair_of_block(nb, H, g, h)) return;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c = lane & 15, gr = lane >> 4, cd = c % D;
    float* tile = k_l + wave * 16 * TD;                // when K and V are in registers
    const int ki = wave * 16 + c, kcol = min(ki, S - 1);
    const bool kok = ki < S;
    const int64_t plane = ((int64_t)g * H + h) * S * S;
    const float* bias_gh = bias ? bias + plane : nullptr;
    float* dbias_gh = dbias ? dbias + plane : nullptr;
    const int at0 = 4 * gr * S + kcol, last = (S - 1) * S + kcol;      // the lane's elements of the plane: at0 + (q0 + t) S, its last one
    const auto ask = [&](int q0, float (&b)[4]) {
#pragma unroll
        for (int t = 0; t < 4; ++t) b[t] = bias_gh ? bias_gh[(uint32_t)min(at0 + (q0 + t) * S, last)] : 0.f;
    };
    float next[4];
    ask(0, next);
    M::stage(Q, g, h, S, H, scale, q_l, rows);
    M::stage(K, g, h, S, H, 1.0f, k_l, rows);
    M::stage(V, g, h, S, H, 1.0f, v_l, rows);
    M::stage(dO, g, h, S, H, 1.0f, g_l, rows);
    {
        // dout . out by the steps that give dout . v: where one key has all of a row's weight (out = v) the two cancel bit for bit, as they must
        // (the row's dS is 0).  The wave's rows: the diagonal.
        const int64_t at = (((int64_t)g * S + kcol) * H + h) * D + gr;
        float ov[KS], gv[KS];
#pragma unroll
        for (int s = 0; s < KS; ++s) { ov[s] = O[at + 4 * s]; gv[s] = dO[at + 4 * s]; }
        const float L = lse[((int64_t)g * H + h) * S + kcol];
        f32x4_t dd = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < KS; ++s) dd = mma4(gv[s], ov[s], dd);
        if (gr == c >> 2) {
            const float t = (c & 2) ? ((c & 1) ? dd[3] : dd[2]) : ((c & 1) ? dd[1] : dd[0]);
            dd_l[ki] = kok ? t : 0.f;
            lse_l[ki] = kok ? L : 0.f;
        }
    }
    __syncthreads();
    float kb[KS], vb[KS], ka[4][DB];
#pragma unroll
    for (int s = 0; s < KS; ++s) { kb[s] = k_l[ki * LD + 4 * s + gr]; vb[s] = v_l[ki * LD + 4 * s + gr]; }
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int i = 0; i < DB; ++i) ka[s][i] = k_l[(wave * 16 + 4 * s + gr) * LD + 16 * i + cd];
    f32x4_t dk[DB], dv[DB];
#pragma unroll
    for (int i = 0; i < DB; ++i) dk[i] = dv[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    // dQ of `n` rows from row0 on: the waves' shares in order
    const auto add_up = [&](const float* shares, int apart, int row0, int n, int first, int threads) {
        for (int e = first; e < n * KS; e += threads) {
            f32x4_t t = {0.f, 0.f, 0.f, 0.f};
            for (int w = 0; w < waves; ++w) t += *reinterpret_cast<const f32x4_t*>(&shares[w * apart + 4 * e]);
            *reinterpret_cast<f32x4_t*>(dQ + (((int64_t)g * S + row0 + e / KS) * H + h) * D + e % KS * 4) = t * scale;
        }
    };
    __syncthreads();      // everybody has its K and V
#pragma unroll 1
    for (int q0 = 0; q0 < S; q0 += 16) {
        float b[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) b[t] = next[t];
        if (q0 + 16 < S) ask(q0 + 16, next);
        f32x4_t sc = {0.f, 0.f, 0.f, 0.f}, dp = sc;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            sc = mma4(q_l[(q0 + c) * LD + 4 * s + gr], kb[s], sc);
            dp = mma4(g_l[(q0 + c) * LD + 4 * s + gr], vb[s], dp);
        }
        const int r0 = q0 + 4 * gr;
        const f32x4_t L4 = *reinterpret_cast<const f32x4_t*>(&lse_l[r0]), D4 = *reinterpret_cast<const f32x4_t*>(&dd_l[r0]);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const bool in = kok && r0 + t < S;
            const float p = expf(sc[t] + b[t] - L4[t]);
            const float ks = !DROP ? 1.0f : (drop_keep(da, drop_row_hash(da, g * H + h, r0 + t), ki) ? da.inv_keep : 0.f);
            const float dS = in ? p * (dp[t] * ks - D4[t]) : 0.f, pk = in ? p * ks : 0.f;
            if (dbias_gh && in) dbias_gh[(uint32_t)(at0 + (q0 + t) * S)] = dS;
            tile[(4 * gr + t) * TD + c] = dS;
#pragma unroll
            for (int i = 0; i < DB; ++i) {
                dk[i] = mma4(q_l[(r0 + t) * LD + 16 * i + cd], dS, dk[i]);      // q_l holds q * sqrt(d): d s / d k
                dv[i] = mma4(g_l[(r0 + t) * LD + 16 * i + cd], pk, dv[i]);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        f32x4_t dq[DB];
#pragma unroll
        for (int i = 0; i < DB; ++i) dq[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const float ds = tile[c * TD + 4 * s + gr];
#pragma unroll
            for (int i = 0; i < DB; ++i) dq[i] = mma4(ka[s][i], ds, dq[i]);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        const int step = q0 / 16;
        float* shares = EACH ? part + (step & 1) * waves * 16 * D : part + q0 * D;
        const int apart = (EACH ? 16 : rows) * D;      // from a wave's to the next one's
#pragma unroll
        for (int i = 0; i < DB; ++i)
            if (D >= 16 || 4 * gr < D) *reinterpret_cast<f32x4_t*>(&shares[wave * apart + c * D + 16 * i + 4 * gr]) = dq[i];
        if constexpr (EACH) {
            __syncthreads();      // (the other step's shares have been read: who adds them up comes here afterwards)
            if (wave == step % waves) add_up(shares, apart, q0, min(16, S - q0), lane, 64);
        }
    }
    if constexpr (!EACH) {
        __syncthreads();
        add_up(part, rows * D, 0, S, threadIdx.x, blockDim.x);
    }
    if (kok) {
#pragma unroll
        for (int i = 0; i < DB; ++i)
            if (D >= 16 || 4 * gr < D) {
                const int64_t at = (((int64_t)g * S + ki) * H + h) * D + 16 * i + 4 * gr;
                *reinterpret_cast<f32x4_t*>(dK + at) = dk[i];
                *reinterpret_cast<f32x4_t*>(dV + at) = dv[i];
            }
    }
}

template <int D>
static int launch_f32_mm(const DenseF32Call& c, bool bwd) {
    const float scale = sqrtf((float)D);
    const bool drop = c.p_drop > 0.f;
    const DropArgs da = drop_args(c.p_drop, c.seed);
    const dim3 grid((unsigned)(((c.b + 7) / 8) * 8 * c.H)), block(64 * Mm<D>::tiles(c.S));
    static std::atomic<uint64_t> done[6];
    const int whole = Mm<D>::bwd_lds(c.S, false);
    const bool each = whole > 160 * 1024 || (whole > 48 * 1024 && (int64_t)c.b * c.H > num_cus());
    const int lds = bwd ? (each ? Mm<D>::bwd_lds(c.S, true) : whole) : Mm<D>::fwd_lds(c.S);
    KernelTimer t(bwd ? KS_DENSE_BWD : KS_DENSE_FWD, c.st);
    if (bwd) {
        const auto kernel = each ? (drop ? &k_dense_f32_mm_bwd<D, true, true> : &k_dense_f32_mm_bwd<D, false, true>)
                                 : (drop ? &k_dense_f32_mm_bwd<D, true, false> : &k_dense_f32_mm_bwd<D, false, false>);
        if (int rc = allow_lds(reinterpret_cast<const void*>(kernel), 160 * 1024, done[2 + 2 * each + drop])) return rc;
        hipLaunchKernelGGL(kernel, grid, block, lds, c.st, c.q, c.k, c.v, c.bias, c.out, c.lse, c.dout, c.dq, c.dk, c.dv, c.dbias, c.S, c.H, scale, c.b, da);
    } else {
        const auto kernel = drop ? &k_dense_f32_mm_fwd<D, true> : &k_dense_f32_mm_fwd<D, false>;
        if (int rc = allow_lds(reinterpret_cast<const void*>(kernel), 160 * 1024, done[drop])) return rc;
        hipLaunchKernelGGL(kernel, grid, block, lds, c.st, c.q, c.k, c.v, c.bias, c.o_out, c.o_lse, c.S, c.H, scale, c.b, da);
    }
    TGT_HIP_CHECK(hipGetLastError());
    return TGT_OK;
}

template <int D>
static int launch_f32(const DenseF32Call& c, bool bwd) {
    const int lds_bwd = (4 * c.S * D + 2 * c.S) * 4 + c.S * kF32StripLd * 4;
    const int lds = bwd ? lds_bwd : 2 * c.S * D * 4 + c.S * kF32StripLd * 4;
    if (lds_bwd > 160 * 1024) {      // the forward refuses what its backward could not run
        set_error("dense attention (float32): S=%d with head dim %d needs %d bytes of LDS (limit %d)", c.S, D, lds_bwd, 160 * 1024);
        return TGT_ERR_UNSUPPORTED;
    }
    // (the thread-per-row kernels take what is left: more than 256 rows, or 192 of head dim 32, whose images leave the LDS)
    if (Mm<D>::fits(c.S)) return launch_f32_mm<D>(c, bwd);
    const float scale = sqrtf((float)D);      // the reference MULTIPLIES q by sqrt(d)
    const bool drop = c.p_drop > 0.f;
    const DropArgs da = drop_args(c.p_drop, c.seed);
    const dim3 grid((unsigned)(((c.b + 7) / 8) * 8 * c.H)), block(kF32Block);
    static bool attr_done = false;
    if (!attr_done) {
        const int cap = 160 * 1024;
        TGT_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_dense_f32_fwd<D, false>), hipFuncAttributeMaxDynamicSharedMemorySize, cap));
        TGT_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_dense_f32_fwd<D, true>), hipFuncAttributeMaxDynamicSharedMemorySize, cap));
        TGT_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_dense_f32_bwd<D, false>), hipFuncAttributeMaxDynamicSharedMemorySize, cap));
        TGT_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_dense_f32_bwd<D, true>), hipFuncAttributeMaxDynamicSharedMemorySize, cap));
        attr_done = true;
    }
    if (!bwd) {
        KernelTimer t(KS_DENSE_FWD, c.st);
        if (drop) hipLaunchKernelGGL((k_dense_f32_fwd<D, true>), grid, block, lds, c.st, c.q, c.k, c.v, c.bias, c.o_out, c.o_lse, c.S, c.H, scale, c.b, da);
        else hipLaunchKernelGGL((k_dense_f32_fwd<D, false>), grid, block, lds, c.st, c.q, c.k, c.v, c.bias, c.o_out, c.o_lse, c.S, c.H, scale, c.b, da);
    } else {
        KernelTimer t(KS_DENSE_BWD, c.st);
        if (drop) hipLaunchKernelGGL((k_dense_f32_bwd<D, true>), grid, block, lds, c.st, c.q, c.k, c.v, c.bias, c.out, c.lse, c.dout, c.dq, c.dk, c.dv, c.dbias, c.S, c.H, scale, c.b, da);
        else hipLaunchKernelGGL((k_dense_f32_bwd<D, false>), grid, block, lds, c.st, c.q, c.k, c.v, c.bias, c.out, c.lse, c.dout, c.dq, c.dk, c.dv, c.dbias, c.S, c.H, scale, c.b, da);
    }
    TGT_HIP_CHECK(hipGetLastError());
    return TGT_OK;
}

int dense_attn_f32(const DenseF32Call& c, bool bwd) {
    switch (c.d) {
        case 8: return launch_f32<8>(c, bwd);
        case 16: return launch_f32<16>(c, bwd);
        case 32: return launch_f32<32>(c, bwd);
        default:
            set_error("dense attention: head dim %d not in {8, 16, 32}", c.d);
            return TGT_ERR_UNSUPPORTED;
    }
}

}  // namespace tgt
