// The readout of the node-level GT (MLPReadout and log_softmax, models/gt_dist_node_level.py:270-286, 337-341) behind layers of 64 features:
//
//     forward   logp = log_softmax(Wc relu(Wb relu(Wa x + ba) + bb) + bc)
//     backward  d logp -> dx and the gradients of the three weights and biases, the activations formed again from x
//
// Widths up to 64, 32 and 16 in the model: as a kernel per linear, activation and softmax these are fourteen launches of 3 to 12 us for 64 K nodes
// that read and write rows of 32 to 128 bytes (33 us forward and 58 backward, and their host time).  Here a wave carries its nodes
// through all of it (node_tile.h), the narrow weights packed as 64 x 64 with zeros.  Backward: the roles of node_roles.h; bound by the chain of a
// group's products.  64 K rows (kernel trace): bf16 10.8 us forward, 24.9 + 4 (the sums) backward; float32 16.6 and 54 + 4.  Of these 0.4 and 0.8, 0.9 and
// 3.5 keep infinities what they are (`mend`, `add_product`) and the float32 sums as exact as the linears' (`product`).
#include "node_roles.h"
#include "class_rows.h"

namespace tgt {
namespace {

constexpr int kMats = 3, kRows = 16, kWaves = 16;      // weights; forward: rows of a wave, waves of a workgroup at most
template <typename T> constexpr int readout_lds(int waves) { return kMats * kFragVecs<Num<T>::P> * 16 + kMats * kVec * 4 + waves * RowShape<T, kRows>::kVecs * 16; }

// float32 weight element (o, k) of a packed 64 x 64 weight: o = 16 g + i, i = 0 .. 15, lies `i` further on (node_tile.h)
struct WeightColumn {
    const nbf16* e;
    __device__ __forceinline__ WeightColumn(const vec16* w, int g, int k)
        : e(reinterpret_cast<const nbf16*>(w + (k >> 3 & 1) * 4 * 3 * 64 + 16 * (k >> 4) + 4 * gray2(g)) + (k & 7)) {}
    __device__ __forceinline__ float at(int i) const {
        const nbf16* p = e + ((i >> 2) * 3 * 64 + (i & 3)) * 8;
        return from_planes(as_float(p[0]), as_float(p[64 * 8]), as_float(p[2 * 64 * 8]));
    }
};
// y = W x + bias (null: without) by plain float32 multiply-adds, x and the weight of `ins` x `outs` that count, zero behind them
__device__ __forceinline__ void linear_again(TileOf<kRows>& y, const TileOf<kRows>& x, const vec16* w, const float* bias, int outs, int ins, vec16* stage, int lane) {
    constexpr int R = kRows;
    const int n = lane % R, g = lane / R;
    float* row = reinterpret_cast<float*>(stage) + 64 * n;
    wave_sync();
    TGT_EACH(i) row[R * g + i] = x.get(i);
    wave_sync();
    TGT_EACH(i) y.set(i, bias ? bias[R * g + i] : 0.f);
#pragma unroll 1
    for (int k = 0; k < ins; ++k) {
        const WeightColumn c(w, g, k);
        const float v = row[k];
        TGT_EACH(i) {
            y.set(i, fmaf(c.at(i), v, y.get(i)));
            if (i % 4 == 3) fence_schedule();
        }
    }
    TGT_EACH(i) if (R * g + i >= outs) y.set(i, 0.f);
    wave_sync();
}
__device__ __forceinline__ void whole(TileOf<kRows>& t, const Frags<3, kRows>& f) {
#pragma unroll
    for (int s = 0; s < kRows / 8; ++s) {
        float v[3][8];
#pragma unroll
        for (int p = 0; p < 3; ++p) unpack16(__builtin_bit_cast(vec16, f.p[s][p]), v[p], (const nbf16*)nullptr);
#pragma unroll
        for (int e = 0; e < 8; ++e) t.set(8 * s + e, from_planes(v[0][e], v[1][e], v[2][e]));
    }
}
// Behind a product y = W x: what operands that are not finite leave of it where it does not belong.  float32: the product again, without planes
// (`holds_nan`).  bf16: zeros in the features behind `outs`, where the packing's zeros met an infinity and the next product would read the NaN (the last
// feature has one if any has).  TAIL: zeros in the rows past the end, whose ReLUs are off then: they must not add to
// sums over nodes (0 times an infinite weight).
// The rare part stands apart from the rest: in its place it is a few KB that every wave fetches its way around (bf16, 64 K rows, backward: 25.8 us
// without `mend`, 28.1 in its place, 26.4 apart; a look of half the instructions, v_maximum3 of two values each, takes as long).
template <int P, bool TAIL> __device__ __forceinline__ void mend(TileOf<kRows>& y, const Frags<P, kRows>& x, const vec16* w, const float* bias, int outs, int ins, vec16* stage, const Rows& rows, int lane) {
    constexpr int R = kRows;
    const int g = lane / R;
    bool off;
    if constexpr (P == 3) off = holds_nan([&](int i) { return y.get(i); }, R);
    else off = __ballot(g == 3 && outs < 64 && !(y.get(R - 1) == 0.f)) != 0;
    if (__builtin_expect(off || (TAIL && rows.left < R), 0)) {
        if constexpr (P == 3) {
            if (off) {
                TileOf<R> t;
                whole(t, x);
                linear_again(y, t, w, bias, outs, ins, stage, lane);
            }
        }
        TGT_EACH(i) if ((P == 1 && R * g + i >= outs) || (TAIL && lane % R >= rows.left)) y.set(i, 0.f);
    }
}

// y = W x + bias (null: without).  float32: the small terms of the planes in a sum of their own, as the linears of any width have them.  rms
// error of the log-probabilities and of dx against 64 bits, widths 32, 16, 40 (64, 64, 64), here / with all six terms in one sum / as separate kernels: 4.5e-8 /
// 6.9e-8 / 6.2e-8 (4.3e-8 / 7.5e-8 / 6.7e-8) and 1.70e-7 / 1.97e-7 / 1.67e-7 (1.70e-7 / 2.22e-7 / 2.09e-7).  (put_classes has its share in the first.)
template <int P> __device__ __forceinline__ void product(TileOf<kRows>& y, const Frags<P, kRows>& x, const vec16* w, const float* bias, int lane) {
    if (bias) load_vec(y, bias, lane / kRows);
    else zero(y);
    if constexpr (P == 3) gemm_apart(y, x, w, lane);
    else gemm<P>(y, x, w, lane);
}

template <typename T> __global__ __launch_bounds__(kWaves * 64) void k_readout_fwd(const tgt_readout_fwd_args a) {
    constexpr int P = Num<T>::P, FV = kFragVecs<P>, R = kRows;
    extern __shared__ __align__(16) unsigned char smem[];
    vec16* w = reinterpret_cast<vec16*>(smem);
    float* vec = reinterpret_cast<float*>(w + kMats * FV);
    const int threads = blockDim.x, NW = threads >> 6;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    vec16* stage = reinterpret_cast<vec16*>(vec + kMats * kVec) + wave * RowShape<T, R>::kVecs;
    const int64_t N = a.rows, tiles = (N + R - 1) / R;
    Raw<T, R> raw;
    const int64_t first = (int64_t)blockIdx.x * NW + wave;
    fetch(raw, reinterpret_cast<const T*>(a.x), Rows(first, N, R), lane);
    copy_direct<kMats * FV>(threads, w, reinterpret_cast<const vec16*>(a.w));
    copy_direct<kMats * kVec>(threads, vec, a.v);
    landed();
    __syncthreads();
    for (int64_t t0 = first; t0 < tiles;) {
        const Rows rows(t0, N, R);
        TileOf<R> y;
        Frags<P, R> x;
        settle<T, false>(y, raw, stage, rows, lane);
        make_frags(x, y);
        product<P>(y, x, w, vec, lane);
        mend<P, false>(y, x, w, vec, a.m1, 64, stage, rows, lane);
        relu<T>(y);
        make_frags(x, y);
        product<P>(y, x, w + FV, vec + kVec, lane);
        mend<P, false>(y, x, w + FV, vec + kVec, a.m2, a.m1, stage, rows, lane);
        relu<T>(y);
        make_frags(x, y);
        product<P>(y, x, w + 2 * FV, vec + 2 * kVec, lane);
        if constexpr (P == 3) mend<P, false>(y, x, w + 2 * FV, vec + 2 * kVec, a.out, a.m2, stage, rows, lane);
        put_classes<T, P == 3>(reinterpret_cast<T*>(a.logp), y, false, a.classes, 0, t0 * R, N, stage, lane);
        t0 += (int64_t)gridDim.x * NW;
        if (t0 < tiles) fetch(raw, reinterpret_cast<const T*>(a.x), Rows(t0, N, R), lane);
    }
}

// Where the sums of a worker lie: the three weights as they are, then the biases
struct Sizes {
    int m1, m2, out;
    __host__ __device__ constexpr int rows(int j) const { return j == 0 ? m1 : (j == 1 ? m2 : out); }
    __host__ __device__ constexpr int cols(int j) const { return j == 0 ? 64 : (j == 1 ? m1 : m2); }
    __host__ __device__ constexpr int at(int j) const {      // weight j, bias j - 3, behind them all (6)
        const int w1 = m1 * 64, w2 = w1 + m2 * m1, b0 = w2 + out * m2;
        return j == 0 ? 0 : (j == 1 ? w1 : (j == 2 ? w2 : (j == 3 ? b0 : (j == 4 ? b0 + m1 : (j == 5 ? b0 + m1 + m2 : b0 + m1 + m2 + out)))));
    }
};

// t where the activation's slope is 1, as a T row would hold it
template <typename T, int R> __device__ __forceinline__ void relu_back(TileOf<R>& t, uint32_t on) {
    TGT_EACH(i) t.set(i, on >> i & 1u ? stored(t.get(i), (const T*)nullptr) : 0.f);
}

// acc += dy^T x over a group's nodes, one 32 x 32 block q of it (node_product).  float32: a group's product in sums of its own, the small terms
// apart, so that acc is rounded once per 64 nodes; and again without planes where it `holds_nan`.  rms error of the sums over all nodes
// against 64 bits, exact operands ~ normal, here / with all six terms in acc: 4 K nodes 1.2e-7 / 1.7e-7, 64 K 1.4e-7 / 3.4e-7, 300 K 1.6e-7 / 1.05e-6 (float32
// matrix instructions would leave 1.5e-7, 2.8e-7 and 6.2e-7); the time is the same.
template <int P, int PB> __device__ __forceinline__ void add_product(float16_t& acc, const unsigned char* dy, const unsigned char* x, int base_dy, int base_x, int q, int lane) {
    if constexpr (P == 1) node_product<P, PB>(acc, dy, x, base_dy, base_x);
    else {
        float16_t c, small;
#pragma unroll
        for (int r = 0; r < 16; ++r) c[r] = small[r] = 0.f;
        node_product<P, PB, true>(c, dy, x, base_dy, base_x, &small);
        c += small;
        if (__builtin_expect(holds_nan([&](int r) { return c[r]; }, 16), 0)) {
#pragma unroll
            for (int r = 0; r < 16; ++r) c[r] = 0.f;
#pragma unroll 1
            for (int n = 0; n < PB / 128; ++n) {
                const float v = plane_elem<PB>(x, n, 32 * (q & 1) + (lane & 31));
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    c[r] = fmaf(plane_elem<PB>(dy, n, 32 * (q >> 1) + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3)), v, c[r]);
                    if (r % 4 == 3) fence_schedule();
                }
            }
        }
        acc += c;
    }
}

template <typename T, int R, int CN> __global__ __launch_bounds__((Bwd<T, R, CN, kMats>::kThreads)) void k_readout_bwd(const tgt_readout_bwd_args a) {
    using L = Bwd<T, R, CN, kMats>;
    constexpr int P = Num<T>::P, FV = kFragVecs<P>, PB = L::kPlane, NC = L::kChain;
    extern __shared__ __align__(16) unsigned char smem[];
    unsigned char *p_dy = smem, *p_x = smem + P * PB;
    vec16* w = reinterpret_cast<vec16*>(smem + L::kW);
    float* vec = reinterpret_cast<float*>(smem + L::kVecs);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), n = lane % R, h = lane / R;
    const int64_t N = a.rows, groups = (N + CN - 1) / CN;
    copy_vecs<kMats * kVec / 4, L::kThreads>(reinterpret_cast<vec16*>(vec), reinterpret_cast<const vec16*>(a.v));
    __syncthreads();
    float16_t acc[kMats];
    float col[kMats];
#pragma unroll
    for (int j = 0; j < kMats; ++j) {
        col[j] = 0.f;
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[j][r] = 0.f;
    }
    if (wave < NC) {
        vec16* stage = reinterpret_cast<vec16*>(smem + L::kStage) + wave * RowShape<T, R>::kVecs;
        const int row = R * wave + n;
        Raw<T, R> raw;
        fetch(raw, reinterpret_cast<const T*>(a.x), Rows(NC * (int64_t)blockIdx.x + wave, N, R), lane);
        for (int64_t g0 = blockIdx.x; g0 < groups; g0 += gridDim.x) {
            const int64_t tile = NC * g0 + wave;
            const Rows rows(tile, N, R);
            TileOf<R> t, d;
            Frags<P, R> f, fx, fy;      // x and the first activation, for the weight gradients
            settle<T, true>(t, raw, stage, rows, lane);
            make_frags(fx, t);
            ClassGrads<T, R> classes(reinterpret_cast<const T*>(a.dlogp), reinterpret_cast<const T*>(a.logp), false, a.classes, 0, tile * R, N, stage, lane);
            if (g0 + gridDim.x < groups) fetch(raw, reinterpret_cast<const T*>(a.x), Rows(tile + NC * (int64_t)gridDim.x, N, R), lane);
            __syncthreads();                                        // Wa is there; product Wa of the round before is done
            product<P>(t, fx, w, vec, lane);
            mend<P, true>(t, fx, w, vec, a.m1, 64, stage, rows, lane);
            __syncthreads();                                        // Wa has been used
            const uint32_t on1 = relu<T>(t);
            make_frags(fy, t);
            classes.settle(d);
            TGT_EACH(i) d.set(i, stored(d.get(i), (const T*)nullptr));
            col[2] += column_sums(d, lane);
            make_frags(f, d);
            __syncthreads();                                        // Wb
            product<P>(t, fy, w, vec + kVec, lane);
            mend<P, true>(t, fy, w, vec + kVec, a.m2, a.m1, stage, rows, lane);
            __syncthreads();                                        // Wb has been used
            const uint32_t on2 = relu<T>(t);
            put_tile_planes<PB, P>(p_x, row, h, t);
            put_planes<PB>(p_dy, row, h, f);
            __syncthreads();                                        // planes of Wc; Wc^T
            product<P>(t, f, w, nullptr, lane);                     // beside product Wc
            if constexpr (P == 3) mend<P, false>(t, f, w, nullptr, a.m2, a.out, stage, rows, lane);
            relu_back<T>(t, on2);
            col[1] += column_sums(t, lane);
            make_frags(f, t);
            __syncthreads();                                        // product Wc is done, Wc^T has been used
            put_planes<PB>(p_dy, row, h, f);
            put_planes<PB>(p_x, row, h, fy);
            __syncthreads();                                        // planes of Wb; Wb^T
            product<P>(t, f, w, nullptr, lane);                     // beside product Wb
            if constexpr (P == 3) mend<P, false>(t, f, w, nullptr, a.m1, a.m2, stage, rows, lane);
            relu_back<T>(t, on1);
            col[0] += column_sums(t, lane);
            make_frags(f, t);
            __syncthreads();                                        // product Wb is done, Wb^T has been used
            put_planes<PB>(p_dy, row, h, f);
            put_planes<PB>(p_x, row, h, fx);
            __syncthreads();                                        // planes of Wa; Wa^T
            product<P>(t, f, w, nullptr, lane);                     // dx, beside product Wa
            if constexpr (P == 3) mend<P, false>(t, f, w, nullptr, 64, a.m1, stage, rows, lane);
            __syncthreads();                                        // Wa^T has been used
            put_rows(reinterpret_cast<T*>(a.dx), t, stage, rows, lane);
        }
    } else {
        const int q = wave - NC, base_dy = operand_base(q >> 1, lane), base_x = operand_base(q & 1, lane);
        const vec16 *fw = reinterpret_cast<const vec16*>(a.w), *bw = reinterpret_cast<const vec16*>(a.w_back);
        WeightsAhead<FV> next;
        next.fetch(fw);
        for (int64_t g0 = blockIdx.x; g0 < groups; g0 += gridDim.x) {
            next.hand_over(w, fw + FV);             // Wa, then on to Wb
            __syncthreads();
            next.hand_over(w, bw + 2 * FV);         // Wb
            __syncthreads();
            next.hand_over(w, bw + FV);             // Wc^T and the planes of Wc
            add_product<P, PB>(acc[2], p_dy, p_x, base_dy, base_x, q, lane);
            __syncthreads();
            next.hand_over(w, bw);                  // Wb^T and the planes of Wb
            add_product<P, PB>(acc[1], p_dy, p_x, base_dy, base_x, q, lane);
            __syncthreads();
            next.hand_over(w, fw);                  // Wa^T and the planes of Wa
            add_product<P, PB>(acc[0], p_dy, p_x, base_dy, base_x, q, lane);
            __syncthreads();
        }
    }
    // the worker's sums, in the weights' own sizes
    __syncthreads();
    const Sizes z{a.m1, a.m2, a.out};
    float* mine = a.partial + (int64_t)blockIdx.x * z.at(2 * kMats);
    float* buf = reinterpret_cast<float*>(smem);
    if (wave < NC) {
#pragma unroll
        for (int c = 0; c < kMats; ++c) buf[(wave * kMats + c) * 64 + lane] = col[c];
    } else {
        const int q = wave - NC, c = 32 * (q & 1) + (lane & 31);
#pragma unroll
        for (int j = 0; j < kMats; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int i = 32 * (q >> 1) + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                if (i < z.rows(j) && c < z.cols(j)) mine[z.at(j) + i * z.cols(j) + c] = acc[j][r];
            }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < kMats * 64; i += L::kThreads) {
        float t = 0.f;
#pragma unroll
        for (int c = 0; c < NC; ++c) t += buf[c * kMats * 64 + i];
        if ((i & 63) < z.rows(i >> 6)) mine[z.at(kMats + (i >> 6)) + (i & 63)] = t;
    }
}

// Sums over the workers, 64 elements x 16 slices of them per workgroup: a slice in worker order, then the slices
struct Outs { void* p[2 * kMats]; };
template <typename T> __global__ __launch_bounds__(1024) void k_readout_sums(const float* __restrict__ partial, int workers, Sizes z, Outs out) {
    __shared__ float part[16][64];
    const int total = z.at(2 * kMats), e = blockIdx.x * 64 + (threadIdx.x & 63), sl = threadIdx.x >> 6;
    const int w0 = workers * sl / 16, w1 = workers * (sl + 1) / 16;
    const float* __restrict__ src = partial + (e < total ? e : total - 1);
    float s = 0.f;
    for (int w = w0; w < w1; w += 16) {
        float t[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) t[i] = src[(int64_t)(w + i < w1 ? w + i : w0) * total];
#pragma unroll
        for (int i = 0; i < 16; ++i) s += w + i < w1 ? t[i] : 0.f;
    }
    part[sl][threadIdx.x & 63] = s;
    __syncthreads();
    if (sl != 0 || e >= total) return;
    s = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) s += part[i][threadIdx.x];
    int j = 0;
    while (j + 1 < 2 * kMats && e >= z.at(j + 1)) ++j;
    if (out.p[j]) reinterpret_cast<T*>(out.p[j])[e - z.at(j)] = to_elem<T>(s);
}

template <typename T> int run_fwd(const tgt_readout_fwd_args& a, hipStream_t st) {
    static std::atomic<uint64_t> done{0};
    const int waves = fwd_waves_for(a.rows, kRows, kWaves);
    if (int rc = allow_lds(reinterpret_cast<const void*>(&k_readout_fwd<T>), readout_lds<T>(kWaves), done)) return rc;
    hipLaunchKernelGGL((k_readout_fwd<T>), dim3(fwd_grid(a.rows, kRows, waves)), dim3(waves * 64), readout_lds<T>(waves), st, a);
    TGT_HIP_CHECK(hipGetLastError());
    return TGT_OK;
}
template <typename T, int R, int CN> int run_bwd(const tgt_readout_bwd_args& a, hipStream_t st) {
    using L = Bwd<T, R, CN, kMats>;
    static std::atomic<uint64_t> done{0};
    const int workers = bwd_workers(a.rows);
    if (int rc = launch(&k_readout_bwd<T, R, CN>, done, workers, L::kThreads, L::kBytes, st, a)) return rc;
    const Sizes z{a.m1, a.m2, a.out};
    Outs out;
    for (int j = 0; j < 2 * kMats; ++j) out.p[j] = a.grads[j];
    hipLaunchKernelGGL((k_readout_sums<T>), dim3((z.at(2 * kMats) + 63) / 64), dim3(1024), 0, st, (const float*)a.partial, workers, z, out);
    TGT_HIP_CHECK(hipGetLastError());
    return TGT_OK;
}
bool widths_ok(int dtype, int m1, int m2, int out, int classes) {
    return (dtype == TGT_DTYPE_F32 || dtype == TGT_DTYPE_BF16) && m1 >= 1 && m1 <= 64 && m2 >= 1 && m2 <= 64 && out >= 1 && out <= 64 && classes >= 1 && classes <= out;
}

}  // namespace
}  // namespace tgt

extern "C" {

int tgt_readout_fwd(const tgt_readout_fwd_args* a, void* stream) {
    using namespace tgt;
    if (!a || a->rows < 0 || !widths_ok(a->dtype, a->m1, a->m2, a->out, a->classes)) return bad("tgt_readout_fwd", "null or bad argument");
    if (a->rows == 0) return TGT_OK;
    if (!a->x || !a->w || !a->v || !a->logp) return bad("tgt_readout_fwd", "null pointer");
    const hipStream_t st = (hipStream_t)stream;
    KernelTimer t(KS_GT_FWD, st);
    // sixteen rows per wave, also with many: us with 16 / 32, float32 4 K rows 6.4 / 8.8, 64 K 13.6 / 14.9, 500 K 75.6 / 83.5; bf16 4.6 / 6.8,
    // 8.4 / 9.5, 47.6 / 46.6
    return a->dtype == TGT_DTYPE_F32 ? run_fwd<float>(*a, st) : run_fwd<nbf16>(*a, st);
}
int64_t tgt_readout_partial_floats(int64_t rows, int m1, int m2, int out) {
    if (rows < 0 || !tgt::widths_ok(TGT_DTYPE_F32, m1, m2, out, 1)) return -1;
    return (int64_t)tgt::bwd_workers(rows) * tgt::Sizes{m1, m2, out}.at(2 * tgt::kMats);
}
int tgt_readout_bwd(const tgt_readout_bwd_args* a, void* stream) {
    using namespace tgt;
    if (!a || a->rows < 1 || !widths_ok(a->dtype, a->m1, a->m2, a->out, a->classes) || !a->x || !a->dlogp || !a->logp || !a->w || !a->w_back || !a->v || !a->dx || !a->partial)
        return bad("tgt_readout_bwd", "null or bad argument");
    const hipStream_t st = (hipStream_t)stream;
    KernelTimer t(KS_GT_BWD, st);
    // Nodes of a workgroup's group: float32 has registers for the chain with eight waves only (128 nodes put 75 to scratch: 16385 rows 29.9 us with 64
    // and 33.0, 64000 53 and 66, 500000 356 and 496); bfloat16 as elsewhere (16384 rows 15.9 and 16.2, 16385 21.7 and 16.4, 64000 36 and 26).
    if (a->dtype == TGT_DTYPE_F32) return run_bwd<float, 16, 64>(*a, st);
    if (groups_of_192(a->rows)) return run_bwd<nbf16, 16, 192>(*a, st);
    return groups_of_64(a->rows, false) ? run_bwd<nbf16, 16, 64>(*a, st) : run_bwd<nbf16, 16, 128>(*a, st);
}

}  // extern "C"
