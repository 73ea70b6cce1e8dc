// Building blocks of the fused per-node kernels (node_layer.hip): everything between two attention launches of an
// encoder layer works on node rows of 64 features, so a wave takes R = 32 or 16 rows and keeps them in registers from the
// first load to the last store.
//
// Register layout.  v_mfma_f32_32x32x16_bf16 leaves D[8 j + 4 h + t][c] in lane c + 32 h (register 4 j + t) and takes
// operand B[k][c] in lane c + 32 h (eight k per lane); v_mfma_f32_16x16x32_bf16 leaves D[4 g + t][c] in lane c + 16 g and
// takes B[k][c] there (eight k per lane, four groups of lanes).  With node rows as columns (c = node) and the rows of the
// weights handed over in a permuted order, lane (node n, group g = lane / R) of a product holds the output features
// R g .. R g + R - 1 of its node in register order, and these registers are the B operand of the next product as they stand: a
// chain of linears, residual adds, LayerNorms and activations never leaves the registers.  LayerNorm sums are R adds in a
// lane and one or two exchanges between the groups.
//
// R = 32 reads every weight once per 32 rows and takes 256 registers in float32; R = 16 halves what a wave holds and the length
// of its chain, and reads the weights twice as often from LDS (in float32 about as long as the products take).
//
// Number formats.  bf16 kernels round where a chain of separate kernels would have stored a tensor (`stored`).  The numbers are those
// of the separate kernels up to the order of float32 sums and, in the node-level Graphormer, to another evaluation of GELU
// (normal_cdf): in float32 both are a few 2^-24 of a row; in bf16 a sum that rounds the other way moves a value by 2^-8 of it, and a
// model's outputs and gradients differ by 0.2 to 1 % of their norm between the two ways of running it, each as far from float32 as
// the other.  Where bits of the separate kernels are wanted (`SAME`), sums and GELU follow them.
// float32 rows go through the matrix unit as three bf16 planes (see linear.hip: hi + mid + lo is exact, six products per pair of planes
// give the float32 product to a few 2^-23); bf16 rows as one.  P = number of planes.
#pragma once
#include "common.h"

namespace tgt {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float float16_t __attribute__((ext_vector_type(16)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef short short4_t __attribute__((ext_vector_type(4)));
typedef uint32_t vec16 __attribute__((ext_vector_type(4)));      // 16 bytes in registers
struct nbf16 { uint16_t x; };
__device__ __forceinline__ float as_float(float v) { return v; }
__device__ __forceinline__ float as_float(nbf16 v) { return __uint_as_float((uint32_t)v.x << 16); }
constexpr int kVec = 64;      // floats per parameter vector

template <typename T> struct Num;
template <> struct Num<float> { static constexpr int P = 3; };
template <> struct Num<nbf16> { static constexpr int P = 1; };

// Lane (n = lane % R, g = lane / R) holds features R g .. R g + R - 1 of node n: get(i) is feature R g + i.
template <int R> struct TileOf {
    float v[R];
    __device__ __forceinline__ float get(int i) const { return v[i]; }
    __device__ __forceinline__ void set(int i, float x) { v[i] = x; }
};
using Tile = TileOf<32>;
#define TGT_EACH(i) _Pragma("unroll") for (int i = 0; i < R; ++i)      // R: rows per wave and features per lane

template <int R> __device__ __forceinline__ void zero(TileOf<R>& t) { TGT_EACH(i) t.set(i, 0.f); }

// The three parts of a float as float words whose lower half is zero (hi, mid) or unused (lo).  The subtractions are of x itself: joined
// with a product that made x (a fused multiply-add), they would be of the unrounded one, whose parts do not end where lo does - the cut
// would then truncate instead of x being rounded (rms error of an activation behind it 7.8e-9 instead of 6.1e-9).
__device__ __forceinline__ void cut3(float x, uint32_t& hi, uint32_t& mid, uint32_t& lo) {
#pragma clang fp contract(off)
    hi = __float_as_uint(x) & 0xffff0000u;
    const float r1 = x - __uint_as_float(hi);
    mid = __float_as_uint(r1) & 0xffff0000u;
    lo = __float_as_uint(r1 - __uint_as_float(mid));
}
__device__ __forceinline__ bf16x8_t upper8(const uint32_t (&w)[8]) {
    vec16 u;
    u.x = __builtin_amdgcn_perm(w[1], w[0], 0x07060302u);
    u.y = __builtin_amdgcn_perm(w[3], w[2], 0x07060302u);
    u.z = __builtin_amdgcn_perm(w[5], w[4], 0x07060302u);
    u.w = __builtin_amdgcn_perm(w[7], w[6], 0x07060302u);
    return __builtin_bit_cast(bf16x8_t, u);
}
__device__ __forceinline__ void to_planes(const float (&v)[8], bf16x8_t (&p)[3]) {
    uint32_t a[8], b[8], c[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) cut3(v[i], a[i], b[i], c[i]);
    p[0] = upper8(a); p[1] = upper8(b); p[2] = upper8(c);
}
__device__ __forceinline__ void to_planes(const float (&v)[8], bf16x8_t (&p)[1]) {
#pragma unroll
    for (int i = 0; i < 8; ++i) p[0][i] = static_cast<__bf16>(v[i]);
}
// the eight contraction indices of step s as matrix operands
template <int P, int R> __device__ __forceinline__ void step_planes(const TileOf<R>& t, int s, bf16x8_t (&p)[P]) {
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = t.get(8 * s + i);
    to_planes(v, p);
}

__device__ __forceinline__ float16_t mma(bf16x8_t a, bf16x8_t b, float16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ float4_t mma(bf16x8_t a, bf16x8_t b, float4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
// c += a b for one contraction step in P planes each, small terms first
template <typename C> __device__ __forceinline__ C mma_planes(const bf16x8_t (&a)[3], const bf16x8_t (&b)[3], C c) {
    c = mma(a[2], b[0], c);
    c = mma(a[0], b[2], c);
    c = mma(a[1], b[1], c);
    c = mma(a[1], b[0], c);
    c = mma(a[0], b[1], c);
    return mma(a[0], b[0], c);
}
template <typename C> __device__ __forceinline__ C mma_planes(const bf16x8_t (&a)[1], const bf16x8_t (&b)[1], C c) { return mma(a[0], b[0], c); }
// The same with the five small terms in a sum of their own, 2^-8 of c: c is rounded once per step instead of six times, the small sum's
// roundings hardly count
__device__ __forceinline__ void mma_planes(const bf16x8_t (&a)[3], const bf16x8_t (&b)[3], float16_t& c, float16_t& small) {
    small = mma(a[2], b[0], small);
    small = mma(a[0], b[2], small);
    small = mma(a[1], b[1], small);
    small = mma(a[1], b[0], small);
    small = mma(a[0], b[1], small);
    c = mma(a[0], b[0], c);
}
__device__ __forceinline__ void mma_planes(const bf16x8_t (&a)[1], const bf16x8_t (&b)[1], float16_t& c, float16_t&) { c = mma(a[0], b[0], c); }
// one plane as two products of half the depth, in the order linear.hip adds them
__device__ __forceinline__ float16_t mma_halves(bf16x8_t a, bf16x8_t b, float16_t c) {
    typedef short short8_t __attribute__((ext_vector_type(8)));
    const short8_t x = __builtin_bit_cast(short8_t, a), y = __builtin_bit_cast(short8_t, b);
    c = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(short4_t{x[0], x[1], x[2], x[3]}, short4_t{y[0], y[1], y[2], y[3]}, c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(short4_t{x[4], x[5], x[6], x[7]}, short4_t{y[4], y[5], y[6], y[7]}, c, 0, 0, 0);
}

// A packed 64 x 64 weight is one layout for both R, 16-byte vectors of eight contraction indices.  R = 16: operand A of step s and block
// m of 16 rows, plane p, is in the 64 vectors from ((4 s + m) P + p) * 64 on; row r of the block is output feature 16 (r / 4) + 4 m +
// r % 4, the indices are the input features 16 (lane / 16) + 8 s ... + 7, and the vector is number 16 (lane / 16) + 4 gray(r / 4) + r % 4
// of the 64.  R = 32 (step s of 16, block m of 32 rows) takes for its row r the output feature 32 ((r / 4) % 2) + 16 m + 4 (r / 8) +
// r % 4 and the input features 32 (lane / 32) + 8 s ... + 7.  The Gray code 0 1 3 2 makes both reads free of bank conflicts: eight
// neighbouring lanes differ in bit 4 of the output feature (R = 16) or in bit 5 (R = 32), and the slot has their exclusive or as its third bit
// (without it the reads of R = 32 meet two by two: 200 K nodes forward in bf16 41.0 us instead of 38.8).
__host__ __device__ constexpr int gray2(int a) { return a ^ (a >> 1); }      // its own inverse for two bits
template <int P> constexpr int kFragVecs = 8 * P * 64;

// Nothing is moved across: left alone, the scheduler asks for every operand of a product before its first instruction, and
// the registers for that are not there
__device__ __forceinline__ void fence_schedule() { __builtin_amdgcn_sched_barrier(0); }

// B operands of a whole tile
template <int P, int R = 32> struct Frags { bf16x8_t p[R / 8][P]; };
template <int P, int R> __device__ __forceinline__ void make_frags(Frags<P, R>& f, const TileOf<R>& t) {
#pragma unroll
    for (int s = 0; s < R / 8; ++s) step_planes<P>(t, s, f.p[s]);
}

// acc += W b: w = packed weight in LDS, b = node rows (a tile, cut into planes one contraction step at a time, or planes);
// the weight operands of the next step are asked for before the products of this one
template <int P> struct StepWeights { bf16x8_t a[2][P]; };
template <int P> __device__ __forceinline__ void step_weights(StepWeights<P>& f, const vec16* const (&w)[2], int s) {
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int p = 0; p < P; ++p) f.a[m][p] = __builtin_bit_cast(bf16x8_t, w[m][((s & 1) * 4 * P + p) * 64 + 16 * (s >> 1)]);
}
template <int P, int R> __device__ __forceinline__ void step_operand(bf16x8_t (&x)[P], const TileOf<R>& b, int s) { step_planes<P>(b, s, x); }
template <int P, int R> __device__ __forceinline__ void step_operand(bf16x8_t (&x)[P], const Frags<P, R>& b, int s) {
#pragma unroll
    for (int p = 0; p < P; ++p) x[p] = b.p[s][p];
}
// HALVES: bits of the separate linears (linear.hip), for one plane
template <int P, bool HALVES = false, typename B> __device__ __forceinline__ void gemm(TileOf<32>& acc, const B& b, const vec16* w0, int lane) {
    const int r = lane & 31, upper = (r >> 2) & 1;
    const vec16* const mine = w0 + (r >> 3) * P * 64 + (r & 3) + (lane & 32);
    const vec16* const w[2] = {mine + 12 * upper, mine + 4 + 4 * upper};      // 4 gray(2 upper + m)
    StepWeights<P> f[2];
    step_weights<P>(f[0], w, 0);
    float16_t c[2];
#pragma unroll
    for (int i = 0; i < 32; ++i) c[i >> 4][i & 15] = acc.get(i);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        if (s < 3) step_weights<P>(f[(s + 1) & 1], w, s + 1);
        bf16x8_t x[P];
        step_operand<P>(x, b, s);
#pragma unroll
        for (int m = 0; m < 2; ++m) {
            if constexpr (HALVES && P == 1) c[m] = mma_halves(f[s & 1].a[m][0], x[0], c[m]);
            else c[m] = mma_planes(f[s & 1].a[m], x, c[m]);
        }
        fence_schedule();
    }
#pragma unroll
    for (int i = 0; i < 32; ++i) acc.set(i, c[i >> 4][i & 15]);
}
template <int P, bool HALVES = false, typename B> __device__ __forceinline__ void gemm(TileOf<16>& acc, const B& b, const vec16* w, int lane) {
    static_assert(!HALVES, "products of half the depth are made by R = 32");
    w += (lane & 0x33) | (gray2((lane >> 2) & 3) << 2);
    bf16x8_t a[2][P], x[P];
    const auto ask = [&](int q) {
#pragma unroll
        for (int p = 0; p < P; ++p) a[q & 1][p] = __builtin_bit_cast(bf16x8_t, w[(q * P + p) * 64]);
    };
    float4_t c[4];
#pragma unroll
    for (int i = 0; i < 16; ++i) c[i >> 2][i & 3] = acc.get(i);
    ask(0);
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        if (q < 7) ask(q + 1);
        if (q % 4 == 0) step_operand<P>(x, b, q / 4);
        c[q & 3] = mma_planes(a[q & 1], x, c[q & 3]);
        fence_schedule();
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) acc.set(i, c[i >> 2][i & 3]);
}
// acc += W b with the small terms of three planes in a sum of their own, one row block after the other and the weights of a step asked
// for when it begins: beside 96 registers of operands there is room for one block's two sums and one step's weights - with the next
// step's too, 22 registers go to scratch and 128 -> 64 of 64 K rows takes 19.6 us instead of 14.9.
// (linear_tiles.hip packs its pieces of a weight for this: operand A of step s and block m of 32 rows, plane p, at ((2 s + m) P + p) * 64 + lane.)
template <int P> __device__ __forceinline__ void gemm_apart(Tile& acc, const Frags<P>& b, const vec16* w, int lane) {
#pragma unroll
    for (int m = 0; m < 2; ++m) {
        float16_t c, small;
#pragma unroll
        for (int i = 0; i < 16; ++i) { c[i] = acc.get(16 * m + i); small[i] = 0.f; }
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            bf16x8_t a[P];
#pragma unroll
            for (int p = 0; p < P; ++p) a[p] = __builtin_bit_cast(bf16x8_t, w[((2 * s + m) * P + p) * 64 + lane]);
            mma_planes(a, b.p[s], c, small);
            fence_schedule();
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) acc.set(16 * m + i, P == 3 ? c[i] + small[i] : c[i]);
    }
}

// acc += W b for sixteen rows, weights in the layout above, one block of rows after the other: its small terms in a sum of their own, the main product of each step
// by itself, and these added up by float adds - a matrix instruction does not round its sum to nearest, and what it leaves adds up over nodes (with both main
// products on top of the small sum, the gradients of four GT layers behind it are off by 5.7e-7 rms, 5.1e-7 this way).  A block's planes
// are asked for as soon as those of the block before have been used.
__device__ __forceinline__ void gemm_apart(TileOf<16>& acc, const Frags<3, 16>& b, const vec16* w, int lane) {
    w += (lane & 0x33) | (gray2((lane >> 2) & 3) << 2);
    bf16x8_t a[2][3];      // [step][plane]
    const auto ask = [&](int m, int p) {
#pragma unroll
        for (int s = 0; s < 2; ++s) a[s][p] = __builtin_bit_cast(bf16x8_t, w[((4 * s + m) * 3 + p) * 64]);
    };
    ask(0, 2); ask(0, 1); ask(0, 0);
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        float4_t c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            c = mma(a[s][2], b.p[s][0], c);
            c = mma(a[s][1], b.p[s][1], c);
            c = mma(a[s][1], b.p[s][0], c);
        }
        if (m < 3) { ask(m + 1, 2); ask(m + 1, 1); }
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            c = mma(a[s][0], b.p[s][2], c);
            c = mma(a[s][0], b.p[s][1], c);
        }
        float4_t main[2];
#pragma unroll
        for (int s = 0; s < 2; ++s) main[s] = mma(a[s][0], b.p[s][0], float4_t{0.f, 0.f, 0.f, 0.f});
        if (m < 3) ask(m + 1, 0);
#pragma unroll
        for (int t = 0; t < 4; ++t) acc.set(4 * m + t, (main[0][t] + main[1][t]) + (c[t] + acc.get(4 * m + t)));
        fence_schedule();
    }
}

// Whether a lane of the wave holds a NaN.  An infinity has no planes (what is left of it behind hi is NaN, and an infinite hi times the
// mid plane of the other operand has any sign): every output that it touches comes out as NaN and is formed again by plain float32
// multiply-adds, which give the +-inf or NaN that it has.  That second computation runs for waves with a NaN only.
template <typename V> __device__ __forceinline__ bool holds_nan(const V& value, int n) {
    float t = 0.f;
#pragma unroll
    for (int i = 0; i < n; ++i) t = fmaf(value(i), 0.f, t);      // (infinities too: they may have become what they are on the way)
    return __ballot(t != 0.f) != 0;
}

// LDS exchanges between lanes of one wave: the hardware runs a wave's LDS accesses in order, this keeps the compiler to it
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The `per` rows of a wave: first row and how many of them exist (wave-uniform, so the addresses have scalar bases)
struct Rows {
    int64_t first;
    int left;       // <= 0: none
    __device__ __forceinline__ Rows(int64_t tile, int64_t N, int per = 32) {
        const int64_t r = N - tile * per;
        left = r > per ? per : (int)r;
        first = left > 0 ? tile * per : 0;
    }
};

// A wave's node rows on their way between global memory (coalesced: consecutive lanes, consecutive 16-byte pieces) and the
// register layout, through a wave-private LDS image of the rows.  Piece q of row r sits in slot q ^ (r mod pieces): both
// the row-wise and the node-wise accesses spread over all banks, and the slots of a lane differ from its first one by an
// exclusive or, which is formed at each access (kept in registers, the addresses of all accesses would crowd out the tiles).
template <typename T, int R = 32> struct RowShape {
    static constexpr int kPieces = 64 * (int)sizeof(T) / 16;      // 16-byte pieces of a row: 16 or 8
    static constexpr int kPer = 64 / kPieces;                     // rows per access of the wave
    static constexpr int kAcc = R / kPer;                         // accesses per tile
    static constexpr int kVecs = R * kPieces;                     // 16-byte vectors of the image
    static constexpr int kMine = kPieces * R / 64;                // pieces of its node's row that a lane holds
};
template <typename T, int R = 32> struct Raw { vec16 v[RowShape<T, R>::kAcc]; };

__device__ __forceinline__ int forgotten(int v) { asm volatile("" : "+v"(v)); return v; }
// slot of access i of the row-wise walk: rows i * kPer ..., consecutive lanes along a row
template <typename T> __device__ __forceinline__ int row_slot(int base, int i) {
    constexpr int PP = RowShape<T>::kPieces, PER = RowShape<T>::kPer;
    return (base ^ ((i * PER) & (PP - 1))) + i * PER * PP;
}
template <typename T> __device__ __forceinline__ int row_base(int lane) {
    constexpr int PP = RowShape<T>::kPieces;
    const int r = lane / PP;
    return forgotten(r * PP + ((lane % PP) ^ r));
}
// slot of the first piece of the lane's share of its node's row (piece i: exclusive or with i)
template <typename T, int R = 32> __device__ __forceinline__ int node_base(int lane) {
    constexpr int PP = RowShape<T, R>::kPieces;
    const int n = lane % R, g = lane / R;
    return forgotten(n * PP + ((g * RowShape<T, R>::kMine) ^ (n & (PP - 1))));
}

template <typename T, int R> __device__ __forceinline__ void fetch(Raw<T, R>& raw, const T* __restrict__ src, const Rows& rows, int lane) {
    constexpr int PP = RowShape<T, R>::kPieces, PER = RowShape<T, R>::kPer;
    const vec16* p = reinterpret_cast<const vec16*>(src) + rows.first * PP;
    const int last = rows.left > 0 ? rows.left - 1 : 0, r0 = forgotten(lane / PP), q = lane % PP;
#pragma unroll
    for (int i = 0; i < RowShape<T, R>::kAcc; ++i) {
        const int r = r0 + i * PER;
        raw.v[i] = p[(uint32_t)((r < last ? r : last) * PP + q)];
    }
}
__device__ __forceinline__ void unpack16(const vec16& u, float (&f)[4], const float*) {
    f[0] = __uint_as_float(u.x); f[1] = __uint_as_float(u.y); f[2] = __uint_as_float(u.z); f[3] = __uint_as_float(u.w);
}
__device__ __forceinline__ void unpack16(const vec16& u, float (&f)[8], const nbf16*) {
    const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        f[2 * i] = __uint_as_float(w[i] << 16);
        f[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
    }
}
__device__ __forceinline__ vec16 pack16(const float (&f)[4], const float*) {
    return vec16{__float_as_uint(f[0]), __float_as_uint(f[1]), __float_as_uint(f[2]), __float_as_uint(f[3])};
}
__device__ __forceinline__ vec16 pack16(const float (&f)[8], const nbf16*) {
    bf16x8_t b;
#pragma unroll
    for (int i = 0; i < 8; ++i) b[i] = static_cast<__bf16>(f[i]);
    return __builtin_bit_cast(vec16, b);
}
// ZERO: rows past the end read as zero (they enter sums over nodes); otherwise they repeat the last row
template <typename T, bool ZERO, int R> __device__ __forceinline__ void settle(TileOf<R>& t, Raw<T, R>& raw, vec16* stage, const Rows& rows, int lane) {
    using Shape = RowShape<T, R>;
    constexpr int PP = Shape::kPieces, PER = Shape::kPer, VE = 16 / (int)sizeof(T);
    if (ZERO && rows.left < R) {
#pragma unroll
        for (int i = 0; i < Shape::kAcc; ++i)
            if (i * PER + lane / PP >= rows.left) raw.v[i] = vec16{0u, 0u, 0u, 0u};
    }
    wave_sync();
    const int rb = row_base<T>(lane);
#pragma unroll
    for (int i = 0; i < Shape::kAcc; ++i) stage[row_slot<T>(rb, i)] = raw.v[i];
    wave_sync();
    const int nb = node_base<T, R>(lane);
#pragma unroll
    for (int i = 0; i < Shape::kMine; ++i) {
        float f[VE];
        unpack16(stage[nb ^ i], f, (const T*)nullptr);
#pragma unroll
        for (int e = 0; e < VE; ++e) t.set(i * VE + e, f[e]);
    }
}
template <typename T, int R> __device__ __forceinline__ void put_rows(T* __restrict__ dst, const TileOf<R>& t, vec16* stage, const Rows& rows, int lane) {
    using Shape = RowShape<T, R>;
    constexpr int PP = Shape::kPieces, PER = Shape::kPer, VE = 16 / (int)sizeof(T);
    wave_sync();
    const int nb = node_base<T, R>(lane);
#pragma unroll
    for (int i = 0; i < Shape::kMine; ++i) {
        float f[VE];
#pragma unroll
        for (int e = 0; e < VE; ++e) f[e] = t.get(i * VE + e);
        stage[nb ^ i] = pack16(f, (const T*)nullptr);
    }
    wave_sync();
    vec16* p = reinterpret_cast<vec16*>(dst) + rows.first * PP;
    const int rb = row_base<T>(lane), r0 = forgotten(lane / PP), q = lane % PP;
    vec16 v[Shape::kAcc];
#pragma unroll
    for (int i = 0; i < Shape::kAcc; ++i) v[i] = stage[row_slot<T>(rb, i)];
    if (rows.left >= R) {
#pragma unroll
        for (int i = 0; i < Shape::kAcc; ++i) p[(uint32_t)((r0 + i * PER) * PP + q)] = v[i];
    } else {
#pragma unroll
        for (int i = 0; i < Shape::kAcc; ++i)
            if (r0 + i * PER < rows.left) p[(uint32_t)((r0 + i * PER) * PP + q)] = v[i];
    }
}
// the value as it will be read back from a T row
__device__ __forceinline__ float stored(float v, const float*) { return v; }
__device__ __forceinline__ float stored(float v, const nbf16*) { return static_cast<float>(static_cast<__bf16>(v)); }

// relu(u), and (bit i) where its slope is 1: as F.relu and its backward, a NaN stays one
template <typename T, int R> __device__ __forceinline__ uint32_t relu(TileOf<R>& u) {
    uint32_t on = 0;
    TGT_EACH(i) {
        const float v = stored(u.get(i), (const T*)nullptr);
        on |= v <= 0.f ? 0u : 1u << i;
        u.set(i, v <= 0.f ? 0.f : v);
    }
    return on;
}

// v of this lane plus v of the lane that is 32 further on or back
__device__ __forceinline__ float both_halves(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// sum over the lanes that share a node
template <int R> __device__ __forceinline__ float node_sum(float v) {
    if constexpr (R == 16) {
        const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
        v = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
    return both_halves(v);
}

// vec: 64 floats in LDS.  (float4_t: an access of float4 may be taken apart, as it was in k_node_bwd_post of 32 rows - 42 reads of two words, 14 registers in
// scratch, 33 K rows 26.1 us instead of 25.1.)
template <int R> __device__ __forceinline__ void load_vec(TileOf<R>& t, const float* vec, int g) {
#pragma unroll
    for (int i = 0; i < R / 4; ++i) {
        const float4_t f = *reinterpret_cast<const float4_t*>(vec + R * g + 4 * i);
        t.set(4 * i, f.x); t.set(4 * i + 1, f.y); t.set(4 * i + 2, f.z); t.set(4 * i + 3, f.w);
    }
}
// y = W x + bias (vec: 64 floats in LDS).  SAME: the bits of linear.hip, which adds the bias behind the products.
template <int P, bool SAME, int R, typename B> __device__ __forceinline__ void linear(TileOf<R>& y, const B& x, const vec16* w, const float* vec, int lane) {
    if constexpr (SAME) {
        zero(y);
        gemm<P, true>(y, x, w, lane);
#pragma unroll
        for (int i = 0; i < R / 4; ++i) {
            const float4_t f = *reinterpret_cast<const float4_t*>(vec + R * (lane / R) + 4 * i);
            y.set(4 * i, y.get(4 * i) + f.x); y.set(4 * i + 1, y.get(4 * i + 1) + f.y);
            y.set(4 * i + 2, y.get(4 * i + 2) + f.z); y.set(4 * i + 3, y.get(4 * i + 3) + f.w);
        }
    } else {
        load_vec(y, vec, lane / R);
        gemm<P>(y, x, w, lane);
    }
}

struct MeanRstd { float mean, rstd; };
// sum of f(i) over the 64 features; SAME: eights in order, then the eights as elementwise.hip's lanes exchange them
template <bool SAME, int R, typename F> __device__ __forceinline__ float sum_features(const F& f) {
    if constexpr (SAME) {
        static_assert(R == 32, "the separate kernels' bits are made by R = 32");
        float t[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float s = 0.f;
#pragma unroll
            for (int k = 0; k < 8; ++k) s += f(8 * i + k);
            t[i] = both_halves(s);
        }
        return (t[0] + t[2]) + (t[1] + t[3]);
    } else {
        float s = 0.f;
        TGT_EACH(i) s += f(i);
        return node_sum<R>(s);
    }
}
template <bool SAME, int R> __device__ __forceinline__ MeanRstd row_stats(const TileOf<R>& x, float eps) {
    const float mean = sum_features<SAME, R>([&](int i) { return x.get(i); }) * (1.f / 64);
    const float var = sum_features<SAME, R>([&](int i) { const float d = x.get(i) - mean; return d * d; }) * (1.f / 64);
    return {mean, rsqrtf(var + eps)};
}
// x -> (x - mean) * rstd; returns rstd
template <bool SAME, int R> __device__ __forceinline__ float normalise(TileOf<R>& x, float eps) {
    const MeanRstd m = row_stats<SAME>(x, eps);
    TGT_EACH(i) x.set(i, (x.get(i) - m.mean) * m.rstd);
    return m.rstd;
}
// xhat * gamma + beta, vectors in LDS
template <int R> __device__ __forceinline__ void affine(TileOf<R>& y, const TileOf<R>& xhat, const float* gamma, const float* beta, int g) {
#pragma unroll
    for (int i = 0; i < R / 4; ++i) {
        const float4_t c = *reinterpret_cast<const float4_t*>(gamma + R * g + 4 * i);
        const float4_t b = *reinterpret_cast<const float4_t*>(beta + R * g + 4 * i);
        y.set(4 * i, xhat.get(4 * i) * c.x + b.x);
        y.set(4 * i + 1, xhat.get(4 * i + 1) * c.y + b.y);
        y.set(4 * i + 2, xhat.get(4 * i + 2) * c.z + b.z);
        y.set(4 * i + 3, xhat.get(4 * i + 3) * c.w + b.w);
    }
}
// g += LayerNorm backward of dy (gamma in LDS)
template <int R> __device__ __forceinline__ void ln_back(TileOf<R>& g, const TileOf<R>& dy, const TileOf<R>& xhat, float rstd, const float* gamma, int group) {
    TileOf<R> d;
    load_vec(d, gamma, group);
    float c1 = 0.f, c2 = 0.f;
    TGT_EACH(i) {
        const float v = d.get(i) * dy.get(i);
        d.set(i, v);
        c1 += v;
        c2 += v * xhat.get(i);
    }
    c1 = node_sum<R>(c1) * (1.f / 64);
    c2 = node_sum<R>(c2) * (1.f / 64);
    TGT_EACH(i) g.set(i, g.get(i) + rstd * (d.get(i) - c1 - xhat.get(i) * c2));
}

// Standard normal distribution function and exp(-u^2 / 2), what GELU and its derivative are made of.  For |u| < 1 the distribution
// function is 1/2 + u P(u^2) with a polynomial P of degree 6 (least squares fit, made for this kernel: 2e-12 from the exact function);
// outside, the upper tail of z = |u| is exp(-z^2 / 2) R(1 / (1 + 0.36 z)) with a polynomial R of degree 5 without constant term (minimax
// fit of the scaled complementary error function for z >= 1: the product with z is within 3.5e-9).  About 26 instructions without a
// branch, the exponential shared by value and derivative, instead of fifty for 0.5 (1 + erff(u / sqrt 2)).
// Measured against 64 bits on this card, rms error of u cdf, here / with erff: u ~ N(0, 0.3) 6.1e-9 / 6.6e-9, N(0, 1) 2.2e-8 / 2.5e-8,
// N(0, 2) 4.3e-8 / 4.9e-8, smaller on each of thirteen intervals of [-8, 8]; of the derivative 2.1e-8 / 2.1e-8, 2.7e-8 / 2.7e-8,
// 2.8e-8 / 2.9e-8, larger on [-1, -0.5] only (1.9e-8 / 1.6e-8).  The tail for all u would take 20 instructions (a training step of 64 K
// nodes in float32 980 us instead of 989, of 870 K nodes in bf16 16.73 ms instead of 16.87), but with the larger error of the two near 0
// (N(0, 0.3) 1.1e-8, derivative 4.7e-8).
__device__ __forceinline__ void normal_cdf(float u, float& cdf, float& bell) {
    const float z = u * u, t = __builtin_amdgcn_rcpf(fmaf(fabsf(u), 0.36f, 1.f));
    bell = __builtin_amdgcn_exp2f(z * -0.72134752044448170f);
    float r = -0.10379677265882492f;
    r = fmaf(r, t, 0.2656746208667755f);
    r = fmaf(r, t, 0.027572302147746086f);
    r = fmaf(r, t, 0.1695895493030548f);
    r = fmaf(r, t, 0.14086511731147766f);
    const float tail = r * t * bell;
    float p = 5.291234970172809e-07f;
    p = fmaf(p, z, -9.247920388588682e-06f);
    p = fmaf(p, z, 0.00011528761388035491f);
    p = fmaf(p, z, -0.001187268877401948f);
    p = fmaf(p, z, 0.009973544627428055f);
    p = fmaf(p, z, -0.06649038195610046f);
    p = fmaf(p, z, 0.3989422917366028f);
    const float outside = u > 0.f ? 1.f - tail : tail;
    cdf = z < 1.f ? fmaf(u, p, 0.5f) : outside;
}

// Sum over the R nodes of every feature: lane l returns the sum of feature l.  A reduce-scatter over the lanes of a
// group: at each of the four or five steps a lane hands half of its values to a partner and keeps the other half.  All exchanges are
// operands of vector instructions (row swap, mirrors within 16 and 8 lanes, quad permutes), none goes through the LDS.
template <int CTRL> __device__ __forceinline__ float lane_permuted(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xf, 0xf, true));
}
template <int BIT, int CTRL, int NV> __device__ __forceinline__ void scatter_step(float (&v)[NV], int lane) {
    const bool up = (lane & BIT) != 0;
#pragma unroll
    for (int i = 0; i < BIT; ++i) {
        const float keep = up ? v[i + BIT] : v[i], send = up ? v[i] : v[i + BIT];
        v[i] = keep + lane_permuted<CTRL>(send);
    }
}
template <int R> __device__ __forceinline__ float column_sums(const TileOf<R>& t, int lane) {
    float v[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        if constexpr (R == 32) {      // rows of 16 lanes: the first keeps value i, the second value i + 16
            const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(t.get(i)), __float_as_uint(t.get(i + 16)), false, false);
            v[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
        } else v[i] = t.get(i);
    }
    scatter_step<8, 0x140>(v, lane);      // row_mirror
    scatter_step<4, 0x141>(v, lane);      // row_half_mirror
    scatter_step<2, 0x4e>(v, lane);       // quad_perm 2 3 0 1
    scatter_step<1, 0xb1>(v, lane);       // quad_perm 1 0 3 2
    return v[0];
}

// Makes the compiler forget what it knows about the values: without it, the planes of a tile that two products use (some
// forty instructions' worth each) are computed once and kept in registers that are not there
template <int R> __device__ __forceinline__ void forget(TileOf<R>& t) {
    TGT_EACH(i) asm volatile("" : "+v"(t.v[i]));
}

// ---- weight gradients: contraction over nodes ---------------------------------------------------------------------------
// The node rows of a workgroup's operand in LDS, P bf16 planes of 64 or 128 rows x 128 bytes (BYTES); a wave writes its rows as they
// sit in its registers and the products read them back transposed (ds_read_b64_tr_b16: within 16 lanes, lane i hands over the address
// of four consecutive elements of row i / 4 and receives column i of the four rows).  16-byte chunk c of row r sits in slot
// c ^ (r mod 8): eight lanes of a write and sixteen of a transposed read touch different banks.
template <int BYTES, int P, int R> __device__ __forceinline__ void put_planes(unsigned char* planes, int row, int g, const Frags<P, R>& f) {
    const int base = forgotten(row * 128 + (((R / 8 * g) ^ (row & 7)) << 4));
#pragma unroll
    for (int s = 0; s < R / 8; ++s)
#pragma unroll
        for (int p = 0; p < P; ++p) *reinterpret_cast<bf16x8_t*>(planes + p * BYTES + (base ^ (s << 4))) = f.p[s][p];
}
// the same of a tile, cut one contraction step at a time (its planes are not kept)
template <int BYTES, int P, int R> __device__ __forceinline__ void put_tile_planes(unsigned char* planes, int row, int g, const TileOf<R>& t) {
    const int base = forgotten(row * 128 + (((R / 8 * g) ^ (row & 7)) << 4));
#pragma unroll
    for (int s = 0; s < R / 8; ++s) {
        bf16x8_t f[P];
        step_planes<P>(t, s, f);
#pragma unroll
        for (int p = 0; p < P; ++p) *reinterpret_cast<bf16x8_t*>(planes + p * BYTES + (base ^ (s << 4))) = f[p];
    }
}
// The float whose three planes these are (an infinity and a NaN are their first)
__device__ __forceinline__ float from_planes(float hi, float mid, float lo) { return fabsf(hi) < INFINITY ? hi + (mid + lo) : hi; }
// feature c of row r of the planes in LDS
template <int BYTES> __device__ __forceinline__ float plane_elem(const unsigned char* planes, int r, int c) {
    const nbf16* e = reinterpret_cast<const nbf16*>(planes + r * 128 + (((c >> 3) ^ (r & 7)) << 4)) + (c & 7);
    return from_planes(as_float(e[0]), as_float(e[BYTES / 2]), as_float(e[BYTES]));
}
// Address of a lane's first piece of the operand that has features 32 block .. + 31 as rows: nodes 8 (lane / 32) ... + 3
__device__ __forceinline__ int operand_base(int block, int lane) {
    const int i = lane & 15, chunk = 4 * block + 2 * ((lane >> 4) & 1) + ((i & 3) >> 1);
    return (8 * (lane >> 5) + (i >> 2)) * 128 + ((chunk ^ (i >> 2)) << 4) + 8 * (i & 1);
}
template <int P, int BYTES> __device__ __forceinline__ void node_operand(bf16x8_t (&out)[P], const unsigned char* planes, int base, int node0) {
    typedef __attribute__((address_space(3))) short4_t lds_short4;
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const unsigned char* q = planes + p * BYTES + node0 * 128;
        const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(q + base));
        const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(q + (base ^ 64) + 512));     // rows + 4
        const uint2 a = __builtin_bit_cast(uint2, lo), b = __builtin_bit_cast(uint2, hi);
        out[p] = __builtin_bit_cast(bf16x8_t, vec16{a.x, a.y, b.x, b.y});
    }
}
// acc += dy^T x over the nodes of the planes, one 32 x 32 block (bases of its rows and columns from operand_base); the operands of
// the next sixteen nodes are asked for before the products of these
// (APART: the small terms in a sum of their own)
template <int P, int BYTES, bool APART = false>
__device__ __forceinline__ void node_product(float16_t& acc, const unsigned char* dy, const unsigned char* x, int base_dy, int base_x, float16_t* small = nullptr) {
    bf16x8_t a[2][P], b[2][P];
    node_operand<P, BYTES>(a[0], dy, base_dy, 0);
    node_operand<P, BYTES>(b[0], x, base_x, 0);
#pragma unroll
    for (int k = 0; k < BYTES / 128; k += 16) {
        const int now = (k >> 4) & 1;
        if (k + 16 < BYTES / 128) {
            node_operand<P, BYTES>(a[now ^ 1], dy, base_dy, k + 16);
            node_operand<P, BYTES>(b[now ^ 1], x, base_x, k + 16);
        }
        if constexpr (APART) mma_planes(a[now], b[now], acc, *small);
        else acc = mma_planes(a[now], b[now], acc);
        fence_schedule();
    }
}

}  // namespace
}  // namespace tgt
