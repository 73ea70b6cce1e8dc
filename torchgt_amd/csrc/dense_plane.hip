// Dense biased attention on bf16 tensors with the [S, S] bias plane of a (graph, head) pair in LDS.
//
// The arithmetic of dense_attn.hip (scores of a 32 x 32 tile by v_mfma_f32_32x32x8_bf16_1k, float32 softmax, the same roundings).  What
// differs is how the bias and its gradient travel.  A plane of S = 129 rows starts at any 2-byte address and its rows have 258 bytes: read tile by tile
// in the layout of the products, a wave asks for pieces of 2 to 36 bytes of 2 to 64 rows with every instruction, and a gradient row is written in
// pieces of 16 bytes.  Here the workgroup copies the plane as what it is, S S consecutive elements, in aligned 16-byte pieces; the walk reads its
// elements from LDS and puts dS in the place of the bias it has used, and the plane goes out as it came.  dQ is formed from it when all of it is
// there: no second image of dS, no sums of dQ to share out.
//
// Measured on 256 graphs of 129 rows, 8 heads of 8, us: backward with the bias read and dBias written in pieces 79.8 (in a copy without the
// stores 49.7, without the loads 62.4, without both 45), here 51; head dim 16 125.6 and 64.7.  Forward 28.0 and 24.5.  The copies alone take 28
// (read and write) and 14 at the rate of a large copy.  What is left is a workgroup's chain - loads 4 to 5 us, the walk 6, dQ 2 - of which a
// CU has room for two or three.  dense_plane_pays has the sizes at which dense_attn.hip's kernels stay.
//
// Tiles that add nothing are left out.  A tile of keys that are all masked (bias -inf for the wave's queries) has probabilities of exactly 0,
// a tile of queries without gradient (padded nodes: nobody read their rows) has dS = 0 and adds 0 to dV.  That holds for finite operands only:
// inf * 0 is NaN, so a workgroup first looks whether all of its q, k, v, dout are below 2^60 (products of them are finite) and its row sums
// are finite; if not, every tile is formed.
#include "dense_tile.h"
#include <algorithm>

namespace tgt {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef uint32_t vec16 __attribute__((ext_vector_type(4)));
typedef unsigned short u16x2_t __attribute__((ext_vector_type(2)));
// v_mfma_f32_16x16x32_bf16: A[r][8 gr + i] and B[8 gr + i][c] in lane r (c) + 16 gr, C[4 gr + t][c] in register t of lane c + 16 gr.  The products
// with few rows (head dim 8 or 16) and 32 or more terms go this way: half the time of 32 x 32 x 16 and a quarter of its registers.
__device__ __forceinline__ float4_t mma16(short4_t a0, short4_t a1, vec16 b, float4_t c) {
    const uint2 x = __builtin_bit_cast(uint2, a0), y = __builtin_bit_cast(uint2, a1);
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, vec16{x.x, x.y, y.x, y.y}), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}
// Columns of a 32 x 32 tile as the two 16-column operands of mma16: lane (c, half) holds in w[0 .. 3] and w[4 .. 7] the rows 8 j + 4 half + t,
// j = 0, 1 and 2, 3, of column c; afterwards lane c + 16 gr holds in w[0 .. 3] (w[4 .. 7]) the rows of half gr / 2 with j = 2 (gr % 2), 2 (gr % 2) + 1 of
// column c (16 + c).
__device__ __forceinline__ void split_columns(uint32_t (&w)[8]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const auto r = __builtin_amdgcn_permlane16_swap(w[i], w[i + 4], false, false);
        w[i] = r[0]; w[i + 4] = r[1];
    }
}

constexpr uint32_t kMasked = 0xff80u;      // -inf

// The plane between memory and LDS: the tensor's elements [0, n) at `p`, whose address is `off` above a multiple of 16 where it is
// an image of the LDS one.
struct Plane {
    unsigned char* lds;      // 16-byte aligned; element 0 at lds + off
    int off, n;
    __device__ __forceinline__ uint16_t get(int e) const { return *reinterpret_cast<const uint16_t*>(lds + off + 2 * e); }
    __device__ __forceinline__ void put(int e, uint16_t v) const { *reinterpret_cast<uint16_t*>(lds + off + 2 * e) = v; }
    __device__ __forceinline__ int pieces() const { return (off + 2 * n + 15) >> 4; }
    // dwords of elements e, e + 1, ... (any e): the aligned words that hold them, shifted into place
    template <int W> __device__ __forceinline__ void words(int e, uint32_t (&out)[W]) const {
        const int o = off + 2 * e;
        const uint32_t* q = reinterpret_cast<const uint32_t*>(lds) + (o >> 2);
        const uint32_t sh = (uint32_t)(o & 2) * 8;
        uint32_t w[W + 1];
#pragma unroll
        for (int i = 0; i <= W; ++i) w[i] = q[i];
#pragma unroll
        for (int i = 0; i < W; ++i) out[i] = __builtin_amdgcn_alignbit(w[i + 1], w[i], sh);
    }
};
// `words` from the last element on, and the copy's pieces, end inside the LDS of the plane wherever it begins
constexpr bool plane_fits(int S) {
    for (int off = 0; off < 16; off += 2)
        if ((off + 2 * (S * S - 1)) / 4 * 4 + 4 * (kPlaneAhead + 1) > plane_bytes(S) || (off + 2 * S * S + 15) / 16 * 16 > plane_bytes(S)) return false;
    return S <= 1 || plane_fits(S - 1);
}
static_assert(plane_fits(288) && 2 * 288 * 288 > kLdsLimit, "every size that fits the LDS");
// The first kAhead pieces of a thread are asked for at once (`ask`), in front of everything else; `arrive` puts them into LDS and fetches what is left.
// (A piece may begin or end outside the tensor, never outside the 16 bytes that one of its elements is in.)
// As many as the largest plane of the variant has, at most eight: eight for every one cost small planes 12 to 22 registers and a wave per SIMD
// (backward, 8 heads of 8, us with eight / as many: 256 graphs of 41 rows 16.4 / 14.9, 129 54.6 / 54.3, 101 45.2 / 44.7).
template <int THREADS, int S_MAX> struct PlaneIn {
    static constexpr int kAhead = std::min(8, (2 * S_MAX * S_MAX + 14 + 15) / 16 / THREADS + 1);
    vec16 v[kAhead];
    const vec16* src;
    int pieces;
    bool aligned;
    __device__ __forceinline__ void ask(const Plane& p, const dbf16* from) {
        aligned = (reinterpret_cast<uintptr_t>(from) & 15) == (uintptr_t)p.off;
        if (!aligned) return;
        src = reinterpret_cast<const vec16*>(reinterpret_cast<const unsigned char*>(from) - p.off);
        pieces = p.pieces();
#pragma unroll
        for (int i = 0; i < kAhead; ++i) v[i] = src[min((int)threadIdx.x + i * THREADS, pieces - 1)];
    }
    __device__ __forceinline__ void arrive(const Plane& p, const dbf16* from) const {
        if (!aligned) {      // bias and dBias begin at different places of 16 bytes
            for (int e = threadIdx.x; e < p.n; e += THREADS) p.put(e, from[e].x);
            return;
        }
        vec16* dst = reinterpret_cast<vec16*>(p.lds);
#pragma unroll
        for (int i = 0; i < kAhead; ++i)
            if ((int)threadIdx.x + i * THREADS < pieces) dst[threadIdx.x + i * THREADS] = v[i];
        for (int at = threadIdx.x + kAhead * THREADS; at < pieces; at += THREADS) dst[at] = src[at];
    }
};
template <int THREADS> __device__ __forceinline__ void plane_out(const Plane& p, dbf16* to) {
    vec16* dst = reinterpret_cast<vec16*>(reinterpret_cast<unsigned char*>(to) - p.off);
    const vec16* src = reinterpret_cast<const vec16*>(p.lds);
    const int pieces = p.pieces(), end = p.off + 2 * p.n;
    for (int at = threadIdx.x; at < pieces; at += THREADS) {
        if (at * 16 >= p.off && at * 16 + 16 <= end) dst[at] = src[at];
        else
            for (int e = max(0, at * 8 - p.off / 2); e < p.n && 2 * e + p.off < at * 16 + 16; ++e) to[e].x = p.get(e);
    }
}

// whether all values seen are below 2^60 in size (exponent field below 187)
struct Tame {
    u16x2_t top = {0, 0};
    __device__ __forceinline__ void look(short4_t x) {
        const uint2 w = __builtin_bit_cast(uint2, x);
        top = __builtin_elementwise_max(top, __builtin_bit_cast(u16x2_t, w.x & 0x7fff7fffu));
        top = __builtin_elementwise_max(top, __builtin_bit_cast(u16x2_t, w.y & 0x7fff7fffu));
    }
    __device__ __forceinline__ bool yes() const { return top.x < (187u << 7) && top.y < (187u << 7); }
};

// four elements of a head's row per item, THREADS items at a time: item c is part c % (D / 4) of row c / (D / 4)
template <int D> struct Item {
    int row, part;
    __device__ __forceinline__ explicit Item(int c) : row(c / (D / 4)), part(c % (D / 4)) {}
};
template <int D, int SP> __device__ __forceinline__ void put_rm(short* rm, const Item<D>& it, short4_t x) {
    *reinterpret_cast<short4_t*>(&rm[it.row * D + it.part * 4]) = x;
}
template <int D, int SP> __device__ __forceinline__ void put_tr(short* tr, const Item<D>& it, short4_t x) {
    tr[(it.part * 4 + 0) * (SP + 4) + it.row] = x.x;
    tr[(it.part * 4 + 1) * (SP + 4) + it.row] = x.y;
    tr[(it.part * 4 + 2) * (SP + 4) + it.row] = x.z;
    tr[(it.part * 4 + 3) * (SP + 4) + it.row] = x.w;
}

// ---- forward ----------------------------------------------------------------------------------------------------------
// Wave w owns query tile w: the walk of dense_attn.hip, its products and sums in the same order (the results are the same bits), with the bias
// from the plane.  The rows of a thin last tile are taken by the waves one after the other, lane = key.
template <int D, int NW, bool THIN, bool DROP>
__global__ __launch_bounds__(64 * NW, 4) void k_plane_fwd(const dbf16* __restrict__ Q, const dbf16* __restrict__ K, const dbf16* __restrict__ V,
                                                          const dbf16* __restrict__ bias, dbf16* __restrict__ out, float* __restrict__ lse, int S, int H, float scale,
                                                          int nb, const DropArgs da) {
    constexpr int KS = D / 8, SP = (NW + THIN) * 32, THREADS = 64 * NW, ITEMS = (SP * (D / 4) + THREADS - 1) / THREADS;
    extern __shared__ __align__(16) char smem[];
    short* k_rm = reinterpret_cast<short*>(smem);
    short* v_tr = k_rm + rm_elems<D, SP>();
    int* flags = reinterpret_cast<int*>(v_tr + tr_elems<D, SP>());
    const int pair = blockIdx.x, win = pair / (8 * H), rem = pair % (8 * H);
    const int g = win * 8 + (rem & 7), h = rem >> 3;
    if (g >= nb) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), col = lane & 31, half = lane >> 5;
    const dbf16* bias_gh = bias + ((int64_t)g * H + h) * S * S;
    Plane plane;
    plane.lds = reinterpret_cast<unsigned char*>(flags) + kFlagBytes;
    plane.off = (int)(reinterpret_cast<uintptr_t>(bias_gh) & 15);
    plane.n = S * S;
    PlaneIn<THREADS, NW * 32 + (THIN ? 4 : 0)> in;
    in.ask(plane, bias_gh);
    const int64_t base = ((int64_t)g * S * H + h) * D;
    const auto row_at = [&](int row) { return base + (int64_t)row * H * D; };
    const int qi = wave * 32 + col, tail = S - NW * 32;
    const bool qok = THIN || qi < S;
    short4_t bq[KS];
    {
        short4_t xk[ITEMS], xv[ITEMS];
#pragma unroll
        for (int j = 0; j < ITEMS; ++j) {
            const Item<D> it(tid + j * THREADS);
            xk[j] = xv[j] = zero4();
            if (it.row < S) {
                const int64_t e = row_at(it.row) + it.part * 4;
                xk[j] = ld4(K + e); xv[j] = ld4(V + e);
            }
        }
#pragma unroll
        for (int s = 0; s < KS; ++s) bq[s] = qok ? ld4(Q + row_at(qi) + s * 8 + half * 4) : zero4();
        in.arrive(plane, bias_gh);
        Tame tame_in;
#pragma unroll
        for (int j = 0; j < ITEMS; ++j) {
            const Item<D> it(tid + j * THREADS);
            tame_in.look(xk[j]); tame_in.look(xv[j]);
            if (it.row < SP) { put_rm<D, SP>(k_rm, it, xk[j]); put_tr<D, SP>(v_tr, it, xv[j]); }
        }
#pragma unroll
        for (int s = 0; s < KS; ++s) tame_in.look(bq[s]);
        const bool ok = __ballot(!tame_in.yes()) == 0;
        if (lane == 0) flags[wave] = ok;
    }
    __syncthreads();
    bool tame = true;
#pragma unroll
    for (int w = 0; w < NW; ++w) tame = tame && flags[w] != 0;
    tame = __builtin_amdgcn_readfirstlane(tame);
    const int krow = key_of_row(col);            // key (inside a tile) of this lane's A-operand row
    // the row sums ride on the second product, as in dense_attn.hip
    constexpr bool SUM_MMA = !DROP && D < 32;
    const short one_bits = 0x3f80;
    const uint32_t rh = DROP ? drop_row_hash(da, g * H + h, qi) : 0u;
    float m = -INFINITY, l = 0.f;
    float16_t o = zero16();      // O^T: a lane's query is qi
    const int qrow = (qok ? qi : S - 1) * S;
    // one key tile: from its scores to the sums.  GROUPS: of four keys per lane that it has at most
    const auto add_tile = [&](float (&sc)[16], int kt, auto groups) {
        constexpr int GROUPS = decltype(groups)::value;
        float tmax = max3(sc[0], sc[1], sc[2]);
#pragma unroll
        for (int r = 3; r < 4 * GROUPS - 1; r += 2) tmax = max3(tmax, sc[r], sc[r + 1]);
        tmax = fmaxf(tmax, sc[4 * GROUPS - 1]);
        {
            const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(tmax), __float_as_uint(tmax), false, false);
            tmax = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
        }
        const float m_new = fmaxf(m, tmax);
        const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
        const float alpha = fast_exp2((m - m_use) * kLog2e);
        const float nm2 = -m_use * kLog2e;
#pragma unroll
        for (int r = 0; r < 4 * KS + (SUM_MMA ? 4 : 0); ++r) o[r] *= alpha;
        if (!SUM_MMA) l *= alpha;
#pragma unroll
        for (int r = 0; r < 4 * GROUPS; ++r) {
            sc[r] = fast_exp2(fmaf(sc[r], kLog2e, nm2));
            if (!SUM_MMA) l += sc[r];
            if (DROP) sc[r] = drop_keep(da, rh, kt * 32 + 16 * half + r) ? sc[r] : 0.f;
        }
#pragma unroll
        for (int t = 0; t < GROUPS; ++t) {
            const short4_t pb = pack4(sc[4 * t + 0], sc[4 * t + 1], sc[4 * t + 2], sc[4 * t + 3]);
            short4_t av = zero4();
            if (col < D) av = *reinterpret_cast<const short4_t*>(&v_tr[col * (SP + 4) + kt * 32 + 16 * half + 4 * t]);
            if (SUM_MMA && col == D) av.x = av.y = av.z = av.w = one_bits;
            o = mfma(av, pb, o);
        }
        m = m_new;
    };
#pragma unroll 1
    for (int kt = 0; kt < NW; ++kt) {
        const int kb = kt * 32 + 16 * half;      // this lane's keys: kb .. kb + 15
        const bool full = THIN || kt * 32 + 32 <= S;
        uint32_t b[kPlaneAhead];
        plane.words(qrow + (full ? kb : min(kb, S - 1)), b);
        if (tame && full) {      // (a row's last tile is formed: what lies behind the row's end is another row's)
            uint32_t other = 0;
#pragma unroll
            for (int i = 0; i < 8; ++i) other |= b[i] ^ (kMasked << 16 | kMasked);
            if (__ballot(other != 0) == 0) continue;
        }
        float16_t s16 = zero16();
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            const short4_t a = *reinterpret_cast<const short4_t*>(&k_rm[(kt * 32 + krow) * D + s * 8 + half * 4]);
            s16 = mfma(a, bq[s], s16);
        }
        float sc[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) sc[r] = fmaf(s16[r], scale, __uint_as_float((r & 1) ? b[r / 2] & 0xffff0000u : b[r / 2] << 16));
        if (!full) {
#pragma unroll
            for (int r = 0; r < 16; ++r) sc[r] = kb + r < S ? sc[r] : -INFINITY;
        }
        add_tile(sc, kt, std::integral_constant<int, 4>{});
    }
    if constexpr (THIN) {
        // the last tile's one to four keys: registers 0..3 of the lower half
        float16_t s16 = zero16();
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            const short4_t a = *reinterpret_cast<const short4_t*>(&k_rm[(NW * 32 + krow) * D + s * 8 + half * 4]);
            s16 = mfma(a, bq[s], s16);
        }
        float sc[16];
#pragma unroll
        for (int r = 0; r < 4; ++r) sc[r] = half == 0 && r < tail ? fmaf(s16[r], scale, bf2f((short)plane.get(qrow + NW * 32 + r))) : -INFINITY;
        add_tile(sc, NW, std::integral_constant<int, 1>{});
    }
    if (SUM_MMA) l = __shfl(o[4 * KS], col);      // row D is the lower half's register 4 KS
    else l += __shfl_xor(l, 32);
    if (qok) {
        const float inv = (DROP ? da.inv_keep : 1.0f) / l;
#pragma unroll
        for (int i = 0; i < KS; ++i) st4(out + row_at(qi) + 8 * i + 4 * half, o[4 * i] * inv, o[4 * i + 1] * inv, o[4 * i + 2] * inv, o[4 * i + 3] * inv);
        if (half == 0) lse[((int64_t)g * H + h) * S + qi] = (m == -INFINITY ? 0.f : m) + __logf(l);
    }
    if constexpr (THIN)
        for (int t = wave; t < tail; t += NW)
            thin_rows_fwd<dbf16, dbf16, D, SP, DROP>(Q, k_rm, v_tr, reinterpret_cast<const dbf16*>(plane.lds + plane.off), S, out, lse, g, h, S, H, scale, NW * 32 + t, 1, lane, da);
}

// ---- backward ---------------------------------------------------------------------------------------------------------
// sum over the 32 lanes of a half of N values per lane: a reduce-scatter, after which lane c of the half holds the sum of value c % N
// (N a power of two of at most 32)
template <int N> __device__ __forceinline__ float half_sums(float (&x)[N], int lane) {
    const auto halve = [&](auto n, int bit) {      // the first n values or the n behind them, by the lane's bit
        const bool up = (lane & bit) != 0;
#pragma unroll
        for (int i = 0; i < decltype(n)::value; ++i) {
            const float keep = up ? x[i + decltype(n)::value] : x[i], send = up ? x[i] : x[i + decltype(n)::value];
            x[i] = keep + __shfl_xor(send, bit);
        }
    };
    if constexpr (N >= 32) halve(std::integral_constant<int, 16>{}, 16);
    if constexpr (N >= 16) halve(std::integral_constant<int, 8>{}, 8);
    if constexpr (N >= 8) halve(std::integral_constant<int, 4>{}, 4);
    halve(std::integral_constant<int, 2>{}, 2);
    halve(std::integral_constant<int, 1>{}, 1);
    float t = x[0];
#pragma unroll
    for (int bit = N; bit < 32; bit <<= 1) t += __shfl_xor(t, bit);
    return t;
}

// Wave w owns key tile w and walks the query tiles (dK, dV in registers, dS into the plane); behind a barrier it owns query tile w and forms dQ
// from the plane's rows while the plane goes out.  THIN: the rows end with a tile of one to four (a virtual node behind a multiple of 32),
// which has no wave of its own: a workgroup of four waves has one on every SIMD and three of them fit a CU - five waves put two on one SIMD,
// and fewer than two such workgroups were resident on average (from the waves' clocks: 14 us each, 374 of 2048 at a time).  Every wave takes
// the thin queries as a strip of its key tile, and the thin keys for its query tile with a lane per query.
//
// W waves share a key tile (every W-th query tile each), and in the second phase a query tile (half of its queries each): a workgroup's
// time is two chains behind its loads, and the planes leave room for two or three workgroups in a CU's LDS.  Measured with W = 1 and 2, us:
// 256 graphs of 129 rows 51.7 and 51.1, 5 of them 12.4 and 10.2, 64 of 201 45.9 and 39.6.  With three tiles a workgroup of six waves
// leaves two SIMDs half empty (400 graphs of 90 rows 43.8 and 67.5, 8 of them 10.0 and 8.3): two waves only where there are fewer than two
// workgroups per CU.
//
// Registers: four waves per SIMD, two at head dim 32 (its images leave no room for more; with four 60 to 98 spilled: 259 graphs of 129 rows 218 us,
// 158 without).
template <int D, int NW, int W, bool THIN, bool DROP>
__global__ __launch_bounds__(64 * NW * W, (D == 32 ? 2 : 4)) void k_plane_bwd(const dbf16* __restrict__ Q, const dbf16* __restrict__ K, const dbf16* __restrict__ V,
                                                                       const dbf16* __restrict__ bias, const dbf16* __restrict__ O, const float* __restrict__ lse,
                                                                       const dbf16* __restrict__ dO, dbf16* __restrict__ dQ, dbf16* __restrict__ dK, dbf16* __restrict__ dV,
                                                                       dbf16* __restrict__ dbias, int S, int H, float scale, int nb, const DropArgs da) {
    constexpr int KS = D / 8, SP = (NW + THIN) * 32, THREADS = 64 * NW * W, RM = rm_elems<D, SP>(), TR = tr_elems<D, SP>(), ITEMS = (SP * (D / 4) + THREADS - 1) / THREADS;
    extern __shared__ __align__(16) char smem[];
    short* q_rm = reinterpret_cast<short*>(smem);
    short* g_rm = q_rm + RM;          // g = dout
    short* q_tr = g_rm + RM;
    short* g_tr = q_tr + TR;
    short* k_tr = g_tr + TR;
    float* lse_l = reinterpret_cast<float*>(k_tr + TR);   // lse * log2(e)
    float* dd_l = lse_l + SP;                             // dout . out
    int* flags = reinterpret_cast<int*>(dd_l + SP);
    float* thin_part = reinterpret_cast<float*>(flags + kFlagBytes / 4);      // [NW][4][2][D]
    const int pair = blockIdx.x, win = pair / (8 * H), rem = pair % (8 * H);      // the heads of a graph on one XCD (dense_attn.hip)
    const int g = win * 8 + (rem & 7), h = rem >> 3;
    if (g >= nb) return;
    const int tid = threadIdx.x, lane = tid & 63, col = lane & 31, half = lane >> 5;
    const int which = __builtin_amdgcn_readfirstlane(tid >> 6), wave = which % NW, share = which / NW;      // tile, and which of its W waves
    const int64_t at = ((int64_t)g * H + h) * S * S;
    const dbf16* bias_gh = bias ? bias + at : nullptr;
    dbf16* dbias_gh = dbias ? dbias + at : nullptr;
    Plane plane;
    plane.lds = reinterpret_cast<unsigned char*>(thin_part + (THIN ? NW * 8 * D : 0));
    plane.off = (int)(reinterpret_cast<uintptr_t>(dbias ? dbias_gh : bias_gh) & 15);
    plane.n = S * S;
    PlaneIn<THREADS, NW * 32 + (THIN ? 4 : 0)> in;
    if (bias) in.ask(plane, bias_gh);
    // rows of this head: element (row, c) at ((g S + row) H + h) D + c
    const int64_t base = ((int64_t)g * S * H + h) * D;
    const auto row_at = [&](int row) { return base + (int64_t)row * H * D; };
    const int ki = wave * 32 + col, tail = S - NW * 32;      // tail: rows of the thin tile
    const int c16 = lane & 15, gr = lane >> 4;               // column and group of mma16
    constexpr int DB = (D + 15) / 16;                        // its blocks of rows
    const bool kok = THIN || ki < S;
    short4_t bk[KS], bv[KS];
    {
        short4_t xq[ITEMS], xg[ITEMS], xk[ITEMS], xo[ITEMS];
        float L[(SP + THREADS - 1) / THREADS];
#pragma unroll
        for (int j = 0; j < ITEMS; ++j) {
            const Item<D> it(tid + j * THREADS);
            xq[j] = xg[j] = xk[j] = xo[j] = zero4();
            if (it.row < S) {
                const int64_t e = row_at(it.row) + it.part * 4;
                xq[j] = ld4(Q + e); xg[j] = ld4(dO + e); xk[j] = ld4(K + e); xo[j] = ld4(O + e);
            }
        }
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            bk[s] = bv[s] = zero4();
            if (kok) {
                bk[s] = ld4(K + row_at(ki) + s * 8 + half * 4);
                bv[s] = ld4(V + row_at(ki) + s * 8 + half * 4);
            }
        }
#pragma unroll
        for (int j = 0; j < (SP + THREADS - 1) / THREADS; ++j) L[j] = tid + j * THREADS < S ? lse[((int64_t)g * H + h) * S + tid + j * THREADS] : 0.f;
        if (bias) in.arrive(plane, bias_gh);
        Tame tame_in;
        bool finite = true;
#pragma unroll
        for (int j = 0; j < ITEMS; ++j) {
            const Item<D> it(tid + j * THREADS);
            tame_in.look(xq[j]); tame_in.look(xg[j]); tame_in.look(xk[j]);
            float t = bf2f(xo[j].x) * bf2f(xg[j].x) + bf2f(xo[j].y) * bf2f(xg[j].y) + bf2f(xo[j].z) * bf2f(xg[j].z) + bf2f(xo[j].w) * bf2f(xg[j].w);
#pragma unroll
            for (int off = 1; off < D / 4; off <<= 1) t += __shfl_xor(t, off);
            finite = finite && fabsf(t) < 1e30f;
            if (it.row < SP) {
                put_rm<D, SP>(q_rm, it, xq[j]); put_tr<D, SP>(q_tr, it, xq[j]);
                put_rm<D, SP>(g_rm, it, xg[j]); put_tr<D, SP>(g_tr, it, xg[j]);
                put_tr<D, SP>(k_tr, it, xk[j]);
                if (it.part == 0) dd_l[it.row] = t;
            }
        }
#pragma unroll
        for (int j = 0; j < (SP + THREADS - 1) / THREADS; ++j) {
            finite = finite && fabsf(L[j]) < 1e30f;
            if (tid + j * THREADS < SP) lse_l[tid + j * THREADS] = L[j] * kLog2e;
        }
#pragma unroll
        for (int s = 0; s < KS; ++s) tame_in.look(bv[s]);
        if (THIN) {      // the values of the thin rows
            const int r = NW * 32 + (lane & 3);
            if (r < S) {
#pragma unroll
                for (int c = 0; c < D / 4; ++c) tame_in.look(ld4(V + row_at(r) + 4 * c));
            }
        }
        const bool ok = __ballot(!(finite && tame_in.yes())) == 0;
        if (lane == 0) flags[which] = ok;
    }
    __syncthreads();
    bool tame = true;
#pragma unroll
    for (int w = 0; w < NW * W; ++w) tame = tame && flags[w] != 0;
    tame = __builtin_amdgcn_readfirstlane(tame);
    const float scale2 = scale * kLog2e;
    float4_t dk[2][DB], dv[2][DB];      // [columns 0 .. 15, 16 .. 31][rows]
    {
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
            for (int i = 0; i < DB; ++i) dk[n][i] = dv[n][i] = float4_t{0.f, 0.f, 0.f, 0.f};
        const int bkey = kok ? ki : 0;
#pragma unroll 1
        for (int qt = share; qt < NW; qt += W) {
            const bool full = THIN || qt * 32 + 32 <= S;
            short4_t aq[KS], ag[KS];
            uint32_t any = 0;
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                aq[s] = *reinterpret_cast<const short4_t*>(&q_rm[(qt * 32 + col) * D + s * 8 + half * 4]);
                ag[s] = *reinterpret_cast<const short4_t*>(&g_rm[(qt * 32 + col) * D + s * 8 + half * 4]);
                const uint2 w = __builtin_bit_cast(uint2, ag[s]);
                any |= (w.x | w.y) & 0x7fff7fffu;
            }
            const int r0 = qt * 32 + 4 * half;      // register r: row r0 + 8 (r / 4) + r % 4
            // element of register r: the plane's rows are S apart in every lane, so that is one add next to the lane's first element
            // (which the compiler is kept from knowing: it would carry sixteen addresses through the tile)
            int e0 = r0 * S + bkey;
            const auto element = [&](int r) { const int e = e0 + (8 * (r / 4) + (r % 4)) * S; return full ? e : min(e, (S - 1) * S + bkey); };
            const auto hide = [&]() { asm volatile("" : "+v"(e0)); };
            hide();
            bool skip = tame && __ballot(any != 0) == 0;
            u16x2_t b[8];
            if (bias && !skip) {
                uint32_t other = 0;
#pragma unroll
                for (int r = 0; r < 16; r += 2) {
                    b[r / 2].x = plane.get(element(r));
                    b[r / 2].y = plane.get(element(r + 1));
                    other |= __builtin_bit_cast(uint32_t, b[r / 2]) ^ (kMasked << 16 | kMasked);
                }
                skip = tame && __ballot(kok && other != 0) == 0;
            }
            hide();
            if (skip) {      // dS = 0, nothing for dV
                if (kok) {
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        if (full || r0 + 8 * (r / 4) + (r % 4) < S) plane.put(element(r), 0);
                }
                continue;
            }
            float16_t sc = zero16(), dp = zero16();
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                sc = mfma(aq[s], bk[s], sc);     // S[query, key]
                dp = mfma(ag[s], bv[s], dp);     // dP[query, key] = dout V^T
            }
            float pr[16];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int qb = r0 + 8 * j;                          // four consecutive queries
                const float4_t L4 = *reinterpret_cast<const float4_t*>(&lse_l[qb]);
                const float4_t D4 = *reinterpret_cast<const float4_t*>(&dd_l[qb]);
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const int r = 4 * j + t;
                    const float bb = bias ? bf2f((short)((r & 1) ? b[r / 2].y : b[r / 2].x)) : 0.f;
                    pr[r] = fast_exp2(fmaf(sc[r], scale2, fmaf(bb, kLog2e, -L4[t])));
                    float ks = 1.0f;
                    if (DROP) ks = drop_keep(da, drop_row_hash(da, g * H + h, qb + t), ki) ? da.inv_keep : 0.f;
                    sc[r] = pr[r] * (dp[r] * ks - D4[t]);
                    if (DROP) pr[r] *= ks;
                }
            }
            if (!THIN && (!full || !kok)) {                  // queries past the end of the batch entry (wave-uniform) or a key past it
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const bool inside = kok && r0 + 8 * (r / 4) + (r % 4) < S;
                    pr[r] = inside ? pr[r] : 0.f;
                    sc[r] = inside ? sc[r] : 0.f;
                }
            }
            // dS of the tile, rounded to bf16 once: into the plane, and as it is the B operand of dK^T += Q^T dS (P likewise for dV^T)
            uint32_t dsp[8], prp[8];
#pragma unroll
            for (int r = 0; r < 16; r += 2) {
                dsp[r / 2] = cvt_pk(sc[r], sc[r + 1]);
                prp[r / 2] = cvt_pk(pr[r], pr[r + 1]);
            }
            if (kok) {
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    if (full || r0 + 8 * (r / 4) + (r % 4) < S) plane.put(element(r), (uint16_t)((r & 1) ? dsp[r / 2] >> 16 : dsp[r / 2] & 0xffffu));
            }
            split_columns(dsp);
            split_columns(prp);
#pragma unroll
            for (int i = 0; i < DB; ++i) {      // dK^T[dd, key] += Q^T dS, dV^T += dout^T P
                short4_t aq0 = zero4(), aq1 = zero4(), ag0 = zero4(), ag1 = zero4();
                if (D >= 16 || c16 < D) {
                    const int e = (16 * i + c16) * (SP + 4) + qt * 32 + 16 * (gr & 1) + 4 * (gr >> 1);
                    aq0 = *reinterpret_cast<const short4_t*>(&q_tr[e]); aq1 = *reinterpret_cast<const short4_t*>(&q_tr[e + 8]);
                    ag0 = *reinterpret_cast<const short4_t*>(&g_tr[e]); ag1 = *reinterpret_cast<const short4_t*>(&g_tr[e + 8]);
                }
#pragma unroll
                for (int n = 0; n < 2; ++n) {
                    dk[n][i] = mma16(aq0, aq1, vec16{dsp[4 * n], dsp[4 * n + 1], dsp[4 * n + 2], dsp[4 * n + 3]}, dk[n][i]);
                    dv[n][i] = mma16(ag0, ag1, vec16{prp[4 * n], prp[4 * n + 1], prp[4 * n + 2], prp[4 * n + 3]}, dv[n][i]);
                }
            }
        }
        if (THIN && share == 0) {
            // the thin queries: registers 0..3 of the lower half
            constexpr int qt = NW;
            float16_t sc = zero16(), dp = zero16();
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                const short4_t aq = *reinterpret_cast<const short4_t*>(&q_rm[(qt * 32 + col) * D + s * 8 + half * 4]);
                const short4_t ag = *reinterpret_cast<const short4_t*>(&g_rm[(qt * 32 + col) * D + s * 8 + half * 4]);
                sc = mfma(aq, bk[s], sc);
                dp = mfma(ag, bv[s], dp);
            }
            const int qb = qt * 32 + 4 * half;
            const float4_t L4 = *reinterpret_cast<const float4_t*>(&lse_l[qb]);
            const float4_t D4 = *reinterpret_cast<const float4_t*>(&dd_l[qb]);
            float p4[4], s4[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const bool inside = half == 0 && t < tail;
                const float bb = bias && inside ? bf2f((short)plane.get((qt * 32 + t) * S + ki)) : 0.f;
                const float pv = fast_exp2(fmaf(sc[t], scale2, fmaf(bb, kLog2e, -L4[t])));
                float ks = 1.0f;
                if (DROP) ks = drop_keep(da, drop_row_hash(da, g * H + h, qb + t), ki) ? da.inv_keep : 0.f;
                p4[t] = inside ? pv * ks : 0.f;
                s4[t] = inside ? pv * (dp[t] * ks - D4[t]) : 0.f;
            }
            const uint2 db = __builtin_bit_cast(uint2, pack4(s4[0], s4[1], s4[2], s4[3])), pb = __builtin_bit_cast(uint2, pack4(p4[0], p4[1], p4[2], p4[3]));
#pragma unroll
            for (int t = 0; t < 4; ++t)
                if (half == 0 && t < tail) plane.put((qt * 32 + t) * S + ki, (uint16_t)((t & 1 ? (t & 2 ? db.y : db.x) >> 16 : (t & 2 ? db.y : db.x)) & 0xffffu));
            uint32_t dsp[8] = {db.x, db.y, 0, 0, 0, 0, 0, 0}, prp[8] = {pb.x, pb.y, 0, 0, 0, 0, 0, 0};
            split_columns(dsp);
            split_columns(prp);
#pragma unroll
            for (int i = 0; i < DB; ++i) {
                short4_t aq = zero4(), ag = zero4();
                if (gr == 0 && (D >= 16 || c16 < D)) {
                    const int e = (16 * i + c16) * (SP + 4) + qt * 32;
                    aq = *reinterpret_cast<const short4_t*>(&q_tr[e]);
                    ag = *reinterpret_cast<const short4_t*>(&g_tr[e]);
                }
#pragma unroll
                for (int n = 0; n < 2; ++n) {
                    dk[n][i] = mma16(aq, zero4(), vec16{dsp[4 * n], dsp[4 * n + 1], dsp[4 * n + 2], dsp[4 * n + 3]}, dk[n][i]);
                    dv[n][i] = mma16(ag, zero4(), vec16{prp[4 * n], prp[4 * n + 1], prp[4 * n + 2], prp[4 * n + 3]}, dv[n][i]);
                }
            }
        }
    }
    if (THIN && share == W - 1) {
        // the thin keys with the queries of tile `wave`, lane = query (both halves; the lower one sums dK, the upper one dV), and in wave 0
        // with the thin queries
        for (int tk = 0; tk < tail; ++tk) {
            const int key = NW * 32 + tk;
            float sums[D];
#pragma unroll
            for (int d = 0; d < D; ++d) sums[d] = 0.f;
            const auto add = [&](int qq, bool in) {
                float qv[D], gv[D], kv[D], vv[D];
                lds_row<D>(q_rm, qq, qv);
                lds_row<D>(g_rm, qq, gv);
#pragma unroll
                for (int c = 0; c < D / 4; ++c) {
                    const short4_t x = ld4(K + row_at(key) + 4 * c), y = ld4(V + row_at(key) + 4 * c);
                    kv[4 * c] = bf2f(x.x); kv[4 * c + 1] = bf2f(x.y); kv[4 * c + 2] = bf2f(x.z); kv[4 * c + 3] = bf2f(x.w);
                    vv[4 * c] = bf2f(y.x); vv[4 * c + 1] = bf2f(y.y); vv[4 * c + 2] = bf2f(y.z); vv[4 * c + 3] = bf2f(y.w);
                }
                const float bb = bias ? bf2f((short)plane.get(qq * S + key)) : 0.f;
                const float pv = fast_exp2(fmaf(dot_d<D>(qv, kv), scale2, fmaf(bb, kLog2e, -lse_l[qq])));
                const float ks = !DROP ? 1.0f : (drop_keep(da, drop_row_hash(da, g * H + h, qq), key) ? da.inv_keep : 0.f);
                const float dS = pv * (dot_d<D>(gv, vv) * ks - dd_l[qq]);
                const short bits = f2bf(dS);
                const float pb = round_bf(pv * ks), dsb = bf2f(bits);
                if (in) {
                    if (half == 0) plane.put(qq * S + key, (uint16_t)bits);
#pragma unroll
                    for (int d = 0; d < D; ++d) sums[d] = half == 0 ? fmaf(dsb, qv[d], sums[d]) : fmaf(pb, gv[d], sums[d]);
                }
            };
            add(wave * 32 + col, true);
            if (wave == 0) add(NW * 32 + min(col, tail - 1), col < tail);
            const float t = half_sums<D>(sums, lane);
            if (col < D) thin_part[((wave * 4 + tk) * 2 + half) * D + col] = t;
        }
    }
    __syncthreads();      // all of dS is in the plane
    if (dbias) plane_out<THREADS>(plane, dbias_gh);
    // dK and dV of a tile: its waves' shares in order, through what the q and dout images were
    constexpr int kLanes = D >= 16 ? 64 : 16 * (D / 4);      // lanes that hold rows
    float4_t* const shares = reinterpret_cast<float4_t*>(smem) + wave * 4 * DB * kLanes;
    static_assert(W == 1 || NW * 4 * DB * kLanes * 16 <= 2 * (2 * RM + 2 * TR), "the shares fit the images");
    if (W > 1 && share > 0 && lane < kLanes) {
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
            for (int i = 0; i < DB; ++i) {
                shares[((n * DB + i) * 2 + 0) * kLanes + lane] = dk[n][i];
                shares[((n * DB + i) * 2 + 1) * kLanes + lane] = dv[n][i];
            }
    }
    if constexpr (THIN) {
        for (int i = tid; i < tail * 2 * D; i += THREADS) {      // dK, dV of the thin keys: the waves' shares in order
            const int tk = i / (2 * D), of_v = (i / D) & 1, d = i % D;
            float t = 0.f;
#pragma unroll
            for (int w = 0; w < NW; ++w) t += thin_part[((w * 4 + tk) * 2 + of_v) * D + d];
            st1((of_v ? dV : dK) + row_at(NW * 32 + tk) + d, of_v ? t : t * scale);
        }
        for (int t = NW * W - 1 - which; t < tail; t += NW * W) {      // dQ of the thin queries, lane = key
            const int q = NW * 32 + t;
            float dq[D];
#pragma unroll
            for (int d = 0; d < D; ++d) dq[d] = 0.f;
            for (int key = lane; key < S; key += 64) {
                const float ds = bf2f((short)plane.get(q * S + key));
#pragma unroll
                for (int d = 0; d < D; ++d) dq[d] = fmaf(ds, bf2f(k_tr[d * (SP + 4) + key]), dq[d]);
            }
            float t2 = half_sums<D>(dq, lane);
            t2 += __shfl_xor(t2, 32);
            if (lane < D) st1(dQ + row_at(q) + lane, t2 * scale);
        }
    }
    constexpr int NQ = 2 / W;      // sixteens of queries of this wave
    float4_t dq[NQ][DB];
    int qrow[NQ];
    const int q0 = wave * 32 + 16 * NQ * share + c16;
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
        qrow[n] = min(q0 + 16 * n, S - 1) * S;
#pragma unroll
        for (int i = 0; i < DB; ++i) dq[n][i] = float4_t{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll 1
    for (int kt = 0; kt < NW; ++kt) {
        const int key = kt * 32 + 8 * gr;      // eight keys: key ... key + 7
        uint32_t w[NQ][4];
#pragma unroll
        for (int n = 0; n < NQ; ++n) {
            if (THIN || kt * 32 + 32 <= S) plane.words(qrow[n] + key, w[n]);
            else {
                plane.words(qrow[n] + min(key, S - 1), w[n]);
#pragma unroll
                for (int i = 0; i < 4; ++i) w[n][i] = key + 2 * i + 1 < S ? w[n][i] : (key + 2 * i < S ? w[n][i] & 0xffffu : 0u);
            }
        }
#pragma unroll
        for (int i = 0; i < DB; ++i) {
            short4_t a0 = zero4(), a1 = zero4();
            if (D >= 16 || c16 < D) {
                a0 = *reinterpret_cast<const short4_t*>(&k_tr[(16 * i + c16) * (SP + 4) + key]);
                a1 = *reinterpret_cast<const short4_t*>(&k_tr[(16 * i + c16) * (SP + 4) + key + 4]);
            }
#pragma unroll
            for (int n = 0; n < NQ; ++n) dq[n][i] = mma16(a0, a1, vec16{w[n][0], w[n][1], w[n][2], w[n][3]}, dq[n][i]);      // dQ^T[dd, query] += K^T dS^T
        }
    }
    if constexpr (THIN) {
        for (int t = 0; t < tail; ++t) {
            const int key = NW * 32 + t;
#pragma unroll
            for (int n = 0; n < NQ; ++n) {
                const float ds = bf2f((short)plane.get(qrow[n] + key));
#pragma unroll
                for (int i = 0; i < DB; ++i)
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        if (D >= 16 || 4 * gr < D) dq[n][i][k] = fmaf(ds, bf2f(k_tr[(16 * i + 4 * gr + k) * (SP + 4) + key]), dq[n][i][k]);
            }
        }
    }
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
        const int q = q0 + 16 * n;
        if (q < S) {
#pragma unroll
            for (int i = 0; i < DB; ++i)
                if (D >= 16 || 4 * gr < D) st4(dQ + row_at(q) + 16 * i + 4 * gr, dq[n][i][0] * scale, dq[n][i][1] * scale, dq[n][i][2] * scale, dq[n][i][3] * scale);
        }
    }
    if (W > 1) {
        __syncthreads();
        if (share > 0) return;
    }
#pragma unroll
    for (int n = 0; n < 2; ++n) {
        const int key = wave * 32 + 16 * n + c16;
#pragma unroll
        for (int i = 0; i < DB; ++i) {
            if (W > 1 && lane < kLanes) {
                dk[n][i] += shares[((n * DB + i) * 2 + 0) * kLanes + lane];
                dv[n][i] += shares[((n * DB + i) * 2 + 1) * kLanes + lane];
            }
            if (key < S && (D >= 16 || 4 * gr < D)) {
                st4(dK + row_at(key) + 16 * i + 4 * gr, dk[n][i][0] * scale, dk[n][i][1] * scale, dk[n][i][2] * scale, dk[n][i][3] * scale);
                st4(dV + row_at(key) + 16 * i + 4 * gr, dv[n][i][0], dv[n][i][1], dv[n][i][2], dv[n][i][3]);
            }
        }
    }
}

template <int D, int NW, int W, bool THIN> int launch_bwd(const DensePlaneCall& c) {
    const float scale = sqrtf((float)c.d);     // the reference MULTIPLIES q by sqrt(d)
    const dim3 grid((unsigned)((c.b + 7) / 8 * 8 * c.H)), block(64 * NW * W);
    const DropArgs da = drop_args(c.p_drop, c.seed);
    const bool drop = c.p_drop > 0.f;
    static std::atomic<uint64_t> done[2];
    constexpr int most = plane_bwd_lds(D, NW * 32 + (THIN ? 4 : 0));
    const int lds = plane_bwd_lds(D, c.S);
    KernelTimer t(KS_DENSE_BWD, c.st);
    const void* kernel = drop ? reinterpret_cast<const void*>(&k_plane_bwd<D, NW, W, THIN, true>) : reinterpret_cast<const void*>(&k_plane_bwd<D, NW, W, THIN, false>);
    if (int rc = allow_lds(kernel, std::min(most, kLdsLimit), done[drop])) return rc;
    const auto run = [&](auto k) {
        hipLaunchKernelGGL(k, grid, block, lds, c.st, (const dbf16*)c.q, (const dbf16*)c.k, (const dbf16*)c.v, (const dbf16*)c.bias, (const dbf16*)c.out, c.lse,
                           (const dbf16*)c.dout, (dbf16*)c.dq, (dbf16*)c.dk, (dbf16*)c.dv, (dbf16*)c.dbias, c.S, c.H, scale, c.b, da);
    };
    if (drop) run(&k_plane_bwd<D, NW, W, THIN, true>);
    else run(&k_plane_bwd<D, NW, W, THIN, false>);
    TGT_HIP_CHECK(hipGetLastError());
    return TGT_OK;
}
template <int D, int NW, bool THIN> int launch_fwd(const DensePlaneCall& c) {
    const float scale = sqrtf((float)c.d);
    const dim3 grid((unsigned)((c.b + 7) / 8 * 8 * c.H)), block(64 * NW);
    const DropArgs da = drop_args(c.p_drop, c.seed);
    const bool drop = c.p_drop > 0.f;
    static std::atomic<uint64_t> done[2];
    constexpr int most = plane_fwd_lds(D, NW * 32 + (THIN ? 4 : 0));
    const int lds = plane_fwd_lds(D, c.S);
    KernelTimer t(KS_DENSE_FWD, c.st);
    const void* kernel = drop ? reinterpret_cast<const void*>(&k_plane_fwd<D, NW, THIN, true>) : reinterpret_cast<const void*>(&k_plane_fwd<D, NW, THIN, false>);
    if (int rc = allow_lds(kernel, std::min(most, kLdsLimit), done[drop])) return rc;
    const auto run = [&](auto k) {
        hipLaunchKernelGGL(k, grid, block, lds, c.st, (const dbf16*)c.q, (const dbf16*)c.k, (const dbf16*)c.v, (const dbf16*)c.bias, (dbf16*)c.o_out, c.o_lse, c.S, c.H,
                           scale, c.b, da);
    };
    if (drop) run(&k_plane_fwd<D, NW, THIN, true>);
    else run(&k_plane_fwd<D, NW, THIN, false>);
    TGT_HIP_CHECK(hipGetLastError());
    return TGT_OK;
}
template <int D, int NW, bool THIN> int launch(const DensePlaneCall& c, bool bwd) {
    if (!bwd) return launch_fwd<D, NW, THIN>(c);
    // waves per tile: k_plane_bwd
    if constexpr (NW == 3)
        if ((int64_t)c.b * c.H < 2 * device_cus()) return launch_bwd<D, NW, 2, THIN>(c);
    return launch_bwd<D, NW, NW == 1 || NW == 3 ? 1 : 2, THIN>(c);
}
template <int D, int NW> int launch_tiles(const DensePlaneCall& c, bool bwd) {
    if constexpr (NW < 8)
        if (c.S > NW * 32) return launch<D, NW, true>(c, bwd);
    return launch<D, NW, false>(c, bwd);
}

}  // namespace

template <int D> int dense_plane(const DensePlaneCall& c, bool bwd) {
    switch (plane_tiles(c.S)) {
        case 1: return launch_tiles<D, 1>(c, bwd);
        case 2: return launch_tiles<D, 2>(c, bwd);
        case 3: return launch_tiles<D, 3>(c, bwd);
        case 4: return launch_tiles<D, 4>(c, bwd);
        case 5: return launch_tiles<D, 5>(c, bwd);
        case 6: return launch_tiles<D, 6>(c, bwd);
        case 7: return launch_tiles<D, 7>(c, bwd);
        case 8: return launch_tiles<D, 8>(c, bwd);
    }
    set_error("dense attention: no plane kernel for %d rows", c.S);
    return TGT_ERR_UNSUPPORTED;
}
#ifndef TGT_PLANE_PART
#error "compile with -DTGT_PLANE_PART=0, 1 or 2 (head dim 8, 16 or 32)"
#endif
template int dense_plane<8 << TGT_PLANE_PART>(const DensePlaneCall&, bool);
}  // namespace tgt
