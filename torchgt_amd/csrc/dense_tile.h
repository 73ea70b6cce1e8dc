// Building blocks of the dense attention kernels on 32 x 32 score tiles (dense_attn.hip, dense_plane.hip): elements, matrix
// instructions, the heads' images in LDS, the rows of a thin last tile.
#pragma once
#include "dense_rows.h"
#include "dense_dropout.h"

namespace tgt {

typedef short short4_t __attribute__((ext_vector_type(4)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef float float16_t __attribute__((ext_vector_type(16)));

// two / four floats -> bf16 (round to nearest even), two values per conversion instruction
__device__ __forceinline__ uint32_t cvt_pk(float lo, float hi) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    f32x2 x;
    x.x = lo; x.y = hi;
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(x, bf16x2));
}
typedef short short4_pk __attribute__((ext_vector_type(4)));
__device__ __forceinline__ short4_pk pack4(float a, float b, float c, float d) {
    typedef uint32_t u2 __attribute__((ext_vector_type(2)));
    u2 r;
    r.x = cvt_pk(a, b);
    r.y = cvt_pk(c, d);
    return __builtin_bit_cast(short4_pk, r);
}

// four consecutive elements as bf16 bits
__device__ __forceinline__ short4_t ld4(const dbf16* p) {
    return *reinterpret_cast<const short4_t*>(p);
}
__device__ __forceinline__ short4_t ld4(const float* p) {
    const float4_t f = *reinterpret_cast<const float4_t*>(p);
    return pack4(f.x, f.y, f.z, f.w);
}
__device__ __forceinline__ void st4(dbf16* p, float a, float b, float c, float d) {
    *reinterpret_cast<short4_t*>(p) = pack4(a, b, c, d);
}
__device__ __forceinline__ void st4(float* p, float a, float b, float c, float d) {
    float4_t r;
    r.x = a; r.y = b; r.z = c; r.w = d;
    *reinterpret_cast<float4_t*>(p) = r;
}
__device__ __forceinline__ float16_t mfma(short4_t a, short4_t b, float16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ float16_t zero16() {
    float16_t z;
#pragma unroll
    for (int i = 0; i < 16; ++i) z[i] = 0.f;
    return z;
}
__device__ __forceinline__ short4_t zero4() { short4_t z; z.x = 0; z.y = 0; z.z = 0; z.w = 0; return z; }

// LDS images of X[g, :, h, :]: row-major [SP][D] and transposed [D][SP+4] (bf16 bits).
template <int D, int SP> constexpr int rm_elems() { return SP * D; }
template <int D, int SP> constexpr int tr_elems() { return D * (SP + 4); }

// Cooperative load of X[g, :, h, :] into either layout (rows >= S are zero).
template <typename T, int D, int SP>
__device__ __forceinline__ void load_head(const T* __restrict__ X, int g, int h, int S, int H,
                                          short* __restrict__ rm, short* __restrict__ tr) {
    for (int c = threadIdx.x; c < SP * (D / 4); c += blockDim.x) {
        const int row = c / (D / 4), part = c % (D / 4);
        short4_t x = zero4();
        if (row < S) x = ld4(X + (((int64_t)g * S + row) * H + h) * D + part * 4);
        if (rm) *reinterpret_cast<short4_t*>(&rm[row * D + part * 4]) = x;
        if (tr) {
            tr[(part * 4 + 0) * (SP + 4) + row] = x.x;
            tr[(part * 4 + 1) * (SP + 4) + row] = x.y;
            tr[(part * 4 + 2) * (SP + 4) + row] = x.z;
            tr[(part * 4 + 3) * (SP + 4) + row] = x.w;
        }
    }
}

// The keys of a 32-key tile are assigned to the rows of the MFMA A operand in a permuted order,
// row 8j + 4h + t  <->  key 16h + 4j + t, so that in the transposed score tile (lane = query,
// half h = lane / 32) register r of a lane is key 16h + r: sixteen CONSECUTIVE keys per lane,
// which is 32 contiguous bytes of that query's bias row.
__device__ __forceinline__ int key_of_row(int row) { return 16 * ((row >> 2) & 1) + 4 * (row >> 3) + (row & 3); }

// 2^x as the bare hardware instruction (inputs here are <= 0 or row maxima differences; results
// below the normal range flush to zero, which is what a softmax weight of that size is worth)
__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

__device__ __forceinline__ float max3(float a, float b, float c) {
    float d;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "v"(c));
    return d;
}

constexpr float kLog2e = 1.4426950408889634f;

constexpr int kLdsLimit = 160 * 1024;

// ---------------------------------------------------------------------------
// The last tile of a sequence of 32 n + 1 .. 32 n + 4 rows (a virtual node behind a multiple of 32)
// holds one to four rows.  As a matrix tile it would cost its wave as much as a full one, so the wave
// that owns it works on the vector unit instead, lane = key (or query), one row at a time: dot
// products from the LDS images, reductions over the wave.  Probabilities and dS are rounded to bf16
// where the matrix path rounds them.
// ---------------------------------------------------------------------------
__device__ __forceinline__ float wave_max(float x) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) x = fmaxf(x, __shfl_xor(x, off));
    return x;
}
template <int D>
__device__ __forceinline__ void lds_row(const short* __restrict__ rm, int row, float (&x)[D]) {
#pragma unroll
    for (int c = 0; c < D / 4; ++c) {
        const short4_t v = *reinterpret_cast<const short4_t*>(&rm[row * D + 4 * c]);
        x[4 * c + 0] = bf2f(v.x); x[4 * c + 1] = bf2f(v.y); x[4 * c + 2] = bf2f(v.z); x[4 * c + 3] = bf2f(v.w);
    }
}
template <typename T, int D>
__device__ __forceinline__ void store_row(T* __restrict__ p, const float (&x)[D], float f) {
#pragma unroll
    for (int c = 0; c < D; c += 4) st4(p + c, x[c] * f, x[c + 1] * f, x[c + 2] * f, x[c + 3] * f);
}

// forward of the rows first .. first + count - 1 (all keys), by one wave
template <typename T, typename BT, int D, int SP, bool DROP>
__device__ __forceinline__ void thin_rows_fwd(const T* __restrict__ Q, const short* __restrict__ k_rm,
                                              const short* __restrict__ v_tr, const BT* __restrict__ bias_gh, int bstride,
                                              T* __restrict__ out, float* __restrict__ lse, int g, int h, int S, int H,
                                              float scale, int first, int count, int lane, const DropArgs da) {
    constexpr int NC = (SP + 63) / 64;
    for (int tq = 0; tq < count; ++tq) {
        const int qi = first + tq;
        float qv[D];
#pragma unroll
        for (int c = 0; c < D / 4; ++c) {
            const short4_t v = ld4(Q + (((int64_t)g * S + qi) * H + h) * D + 4 * c);
            qv[4 * c + 0] = bf2f(v.x); qv[4 * c + 1] = bf2f(v.y); qv[4 * c + 2] = bf2f(v.z); qv[4 * c + 3] = bf2f(v.w);
        }
        const BT* brow = bias_gh ? bias_gh + (int64_t)qi * bstride : nullptr;
        float sv[NC], mx = -INFINITY;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const int key = c * 64 + lane;
            sv[c] = -INFINITY;
            if (key < S) {
                float kv[D];
                lds_row<D>(k_rm, key, kv);
                sv[c] = fmaf(dot_d<D>(qv, kv), scale, brow ? ld1(brow + key) : 0.f);
            }
            mx = fmaxf(mx, sv[c]);
        }
        mx = wave_max(mx);
        const float m_use = (mx == -INFINITY) ? 0.f : mx;
        float lsum = 0.f, ov[D];
#pragma unroll
        for (int d = 0; d < D; ++d) ov[d] = 0.f;
        const uint32_t rh = DROP ? drop_row_hash(da, g * H + h, qi) : 0u;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const int key = c * 64 + lane;
            if (key < S) {
                const float pb = round_bf(fast_exp2((sv[c] - m_use) * kLog2e));
                lsum += pb;
                const float pk = (!DROP || drop_keep(da, rh, key)) ? pb : 0.f;
#pragma unroll
                for (int d = 0; d < D; ++d) ov[d] = fmaf(pk, bf2f(v_tr[d * (SP + 4) + key]), ov[d]);
            }
        }
        lsum = wave_sum(lsum);
#pragma unroll
        for (int d = 0; d < D; ++d) ov[d] = wave_sum(ov[d]);
        if (lane == 0) {
            store_row<T, D>(out + (((int64_t)g * S + qi) * H + h) * D, ov, (DROP ? da.inv_keep : 1.0f) / lsum);
            lse[((int64_t)g * H + h) * S + qi] = m_use + __logf(lsum);
        }
    }
}

// A call of the dense attention with the bias in memory (the plane kernels: on bf16 tensors)
struct DensePlaneCall {
    const void *q, *k, *v, *bias, *out, *dout;
    const float* lse;
    void *o_out, *dq, *dk, *dv, *dbias;
    float* o_lse;
    int b, S, H, d;
    hipStream_t st;
    float p_drop;          // 0: no dropout
    uint64_t seed;
};

inline int device_cus() {
    static int cus = 0;
    if (cus == 0) {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) == hipSuccess && hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess &&
            n > 0)
            cus = n;
        else
            cus = 256;
    }
    return cus;
}

// dense_plane.hip: the kernels that keep the [S, S] plane of a (graph, head) pair in LDS
template <int D> int dense_plane(const DensePlaneCall& c, bool bwd);

// Its tiles of 32 rows with a wave (or two) of their own: a last one of one to four rows behind others has none
constexpr int plane_tiles(int S) { return S > 32 && S - (S - 1) / 32 * 32 <= 4 ? (S - 1) / 32 : (S + 31) / 32; }
// Its LDS: images of the heads, and the plane behind the bytes that its address lies above a multiple of 16
constexpr int kFlagBytes = 64;      // one word per wave
constexpr int kPlaneAhead = 8;      // words that the forward takes from an element on (`Plane::words`), the last of a plane included
constexpr int plane_bytes(int S) { return (16 + 2 * S * S + 4 * kPlaneAhead + 2 + 15) / 16 * 16; }
constexpr int plane_fwd_lds(int D, int S) {
    const int rows = (S + 31) / 32 * 32;
    return 2 * D * (2 * rows + 4) + kFlagBytes + plane_bytes(S);
}
constexpr int plane_bwd_lds(int D, int S) {
    const int rows = (S + 31) / 32 * 32, thin = S > plane_tiles(S) * 32;
    return 2 * D * (2 * rows + 3 * (rows + 4)) + 8 * rows + kFlagBytes + (thin ? plane_tiles(S) * 8 * D * 4 : 0) + plane_bytes(S);
}

// Whether a call with the bias in memory (or, backward, without one) goes to the plane kernels.  us there against dense_attn.hip's, 8 heads:
// - Rows of a multiple of 32 bytes put the lanes' rows on the same LDS banks: S = 64, 128, 160 forward 29.8, 69.8, 46.5 against 17.9, 23.6, 22.6;
//   backward 27, 67, 75 against 22, 43, 55 (head dim 8; with more products per element the conflicts weigh less: 16 with S = 80, 96, 160
//   43.5, 49, 82 against 58, 56, 99, S = 64, 128 30, 70 against 32, 65, and at 32 all 1.1 to 1.7 times faster; forward at 32, S = 80,
//   144, 176 29.6, 46, 52 against 54.7, 65, 44).
// - Forward, few rows: the general kernel's walk takes as long for them as for 32, the plane's loads do not.  400 graphs of 2, 12, 16, 24, 31, 48 rows 4.7, 4.8, 5.0, 5.1,
//   5.3, 11.2 against 18.7, 13.4, 12.8, 13.7, 15.1, 15.0 (head dim 16 5.0, 5.2, 5.6, 5.7, 6.0, 12.5 against 25.8, 14.1, 13.5, 15.3, 16.9, 18.6); 32 graphs of up
//   to 31 rows 2.9 (3.1) against 4.1 to 5.3 (4.2 to 6.6), of 48 3.9 (4.2) against 4.5 (4.8).
// - Forward, a plane of more than 64 KiB leaves one workgroup on a CU: S = 180 30.0 against 29.9, 201 39.3 against 30.6.
// - Forward, one or two thin rows follow the walk of the first waves, which the other planes of a CU have to cover: S = 129 of 64, 128, 256
//   graphs 9.7, 14.9, 24.5 against 8.8, 15.6, 28.0.
// - Backward at head dim 8, up to 24 rows (and one behind 32) are a fraction of a tile either way, and the plane is a phase more:
//   400 graphs of 12, 20, 28 rows 8.8, 9.7, 11.0 against 8.2, 8.8, 13.7.
constexpr bool dense_plane_pays_bwd(int S, int D) {
    return plane_bwd_lds(D, S) <= kLdsLimit && (D == 8 ? S > 24 && S != 33 && S % 16 != 0 : (D == 16 ? S % 64 != 0 : true));
}
inline bool dense_plane_pays(int64_t pairs, int S, int D, bool bwd) {
    if (bwd) return dense_plane_pays_bwd(S, D);
    const int thin = S - plane_tiles(S) * 32;
    return plane_fwd_lds(D, S) <= kLdsLimit && 2 * S * S <= 64 * 1024 && (S % 16 != 0 || (S % 32 == 16 && S < (D == 32 ? 160 : 64))) && (thin < 1 || thin > 2 || pairs >= 4 * device_cus());
}

}  // namespace tgt
