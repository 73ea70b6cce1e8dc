// The node-local part of a GT encoder layer (models/gt_dist_node_level.py:218-267), hidden 64, feed-forward 128, as one forward and
// one backward kernel:
//     y = a O^T + bo;  x1 = LN1(x + y);  s2 = x1 + W2 relu(W1 y + b1) + b2;  x' = LN2(s2);  q, k, v = x' W^T + b
// (the gradient of q, k, v goes through k_node_bwd_pre of node_layer.hip, without its LayerNorm).
//
// What bounds them and why this shape: as in node_layer.hip, whose roles and register tiles these kernels use.  As separate
// kernels the part moves 33 rows of 64 features per node forward and 61 backward through memory, here 7 and 7 (forward: x, a in;
// s2, x', q, k, v out; backward: g, x, a (float32: twice), s2 in, two rows out); y, u and relu(u) are recomputed in the backward (three
// products), s2 is kept, which saves the two products behind them.  The 128 features between the feed-forward linears are two
// tiles; the backward takes them one after the other, so that no more than one is alive, and keeps of u only its signs.
// Measured at 65536 nodes (forward with q, k, v / backward, us): float32 38 / 79, bf16 15 / 29.5; a bf16 training step of four layers
// 1030 us with the separate kernels behind one operator, 557 with these.
// bf16 forward moves 68 MB in 15 us (4.5 TB/s); float32 is bound by its products (six MFMAs for one and the splitting into planes).
#include "node_roles.h"

namespace tgt {
namespace {

enum { V_BO = 0, V_GAMMA1, V_BETA1, V_B1A, V_B1B, V_B2, V_GAMMA2, V_BETA2, kVecs8 };
enum { W_O = 0, W_1A, W_1B, W_2A, W_2B };

template <typename T, int R> __device__ __forceinline__ void round_to(TileOf<R>& t) { TGT_EACH(i) t.set(i, stored(t.get(i), (const T*)nullptr)); }
// Rows per wave and waves of a workgroup at most.  Four launches of a model, us with sixteen rows / with thirty-two and eight waves: float32 4 K nodes 63 / 82,
// 64 K 143 / 153, 300 K 606 / 650; bf16 4 K 38 / 46, 64 K 77 / 81, 300 K 216 / 225.
constexpr int kFwdRows = 16, kFwdWaves = 16;
// float32 takes its packed weights in turns (O and W1, W2, then q, k, v: 72 KB at most next to the row images), bf16 keeps all of them
template <typename T> constexpr int gt_fwd_mats() { return sizeof(T) == 4 ? 3 : 8; }
template <typename T> constexpr int gt_fwd_lds(int waves) { return gt_fwd_mats<T>() * kFragVecs<Num<T>::P> * 16 + (kVecs8 + 3) * kVec * 4 + waves * RowShape<T, kFwdRows>::kVecs * 16; }

template <typename T, bool NEXT> __global__ __launch_bounds__(kFwdWaves * 64) void k_gt_fwd(const tgt_gt_fwd_args a) {
    constexpr int P = Num<T>::P, FV = kFragVecs<P>, R = kFwdRows;
    const int threads = blockDim.x, NW = threads >> 6;
    constexpr bool RESIDENT = sizeof(T) == 2;
    extern __shared__ __align__(16) unsigned char smem[];
    vec16* w = reinterpret_cast<vec16*>(smem);
    float* vec = reinterpret_cast<float*>(w + gt_fwd_mats<T>() * FV);
    float* vn = vec + kVecs8 * kVec;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    vec16* stage = reinterpret_cast<vec16*>(vn + 3 * kVec) + wave * RowShape<T, R>::kVecs;
    const vec16 *gw = reinterpret_cast<const vec16*>(a.w), *gn = reinterpret_cast<const vec16*>(a.w_next);
    const int64_t N = a.rows, tiles = (N + R - 1) / R;
    const vec16 *w2 = RESIDENT ? w + 3 * FV : w, *wn = RESIDENT ? w + 5 * FV : w;
    Raw<T, R> raw_x, raw_a;
    const auto ask = [&](int64_t t0) {
        const Rows rows(t0 + wave, N, R);      // (a wave without rows reads the first one)
        fetch(raw_a, reinterpret_cast<const T*>(a.attn), rows, lane);
        fetch(raw_x, reinterpret_cast<const T*>(a.x), rows, lane);
    };
    const int64_t first = (int64_t)blockIdx.x * NW;
    ask(first);
    copy_direct<(RESIDENT ? 5 : 3) * FV>(threads, w, gw);
    if constexpr (RESIDENT && NEXT) copy_direct<3 * FV>(threads, w + 5 * FV, gn);
    copy_direct<kVecs8 * kVec>(threads, vec, a.vec);
    if constexpr (NEXT) copy_direct<3 * kVec>(threads, vn, a.v_next);
    landed();
    __syncthreads();
    for (int64_t t0 = first;;) {
        const Rows rows(t0 + wave, N, R);
        const bool active = rows.left > 0;
        TileOf<R> s, r[2];
        if (active) {
            TileOf<R> x, y;
            settle<T, false>(x, raw_a, stage, rows, lane);
            linear<P, false>(y, x, w, vec + V_BO * kVec, lane);
            round_to<T>(y);
            settle<T, false>(s, raw_x, stage, rows, lane);
            TGT_EACH(i) s.set(i, s.get(i) + y.get(i));
            normalise<false>(s, a.eps1);
            affine(s, s, vec + V_GAMMA1 * kVec, vec + V_BETA1 * kVec, lane / R);
            round_to<T>(s);      // x1
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                linear<P, false>(r[j], y, w + (W_1A + j) * FV, vec + (V_B1A + j) * kVec, lane);
                relu<T>(r[j]);
            }
        }
        if (!RESIDENT) replace_weights<2 * FV>(threads, w, gw + W_2A * FV);
        if (active) {
            TileOf<R> y;
            load_vec(y, vec + V_B2 * kVec, lane / R);
            gemm<P>(y, r[0], w2, lane);
            gemm<P>(y, r[1], w2 + FV, lane);
            TGT_EACH(i) s.set(i, s.get(i) + stored(y.get(i), (const T*)nullptr));
            if (a.s2) put_rows(reinterpret_cast<T*>(a.s2), s, stage, rows, lane);
            normalise<false>(s, a.eps2);
            affine(s, s, vec + V_GAMMA2 * kVec, vec + V_BETA2 * kVec, lane / R);
            round_to<T>(s);
            put_rows(reinterpret_cast<T*>(a.x_out), s, stage, rows, lane);
        }
        if constexpr (NEXT) {
            if (!RESIDENT) replace_weights<3 * FV>(threads, w, gn);
            if (active) {
#pragma unroll
                for (int j = 0; j < 3; ++j) {
                    TileOf<R> y;
                    linear<P, false>(y, s, wn + j * FV, vn + j * kVec, lane);
                    put_rows(reinterpret_cast<T*>(j == 0 ? a.q : (j == 1 ? a.k : a.v)), y, stage, rows, lane);
                }
            }
        }
        t0 += (int64_t)gridDim.x * NW;
        if (t0 >= tiles) break;
        ask(t0);
        if (!RESIDENT) replace_weights<3 * FV>(threads, w, gw);
    }
}

// ---- backward -------------------------------------------------------------------------------------------------------------
// Weights in the order the chain uses them: O, W1a, W2a^T, W1a^T, W1b, W2b^T, W1b^T, O^T.  Every step has two barriers: its weight
// (and the planes of its weight gradient) are there; they have been used.
template <typename T, int R, int CN> __global__ __launch_bounds__((Bwd<T, R, CN, kVecs8>::kThreads)) void k_gt_bwd(const tgt_gt_bwd_args a) {
    using L = Bwd<T, R, CN, kVecs8>;
    constexpr int P = Num<T>::P, FV = kFragVecs<P>, PB = L::kPlane, NC = L::kChain;
    constexpr bool CUT_AGAIN = P != 1;
    extern __shared__ __align__(16) unsigned char smem[];
    unsigned char *p_dy = smem, *p_x = smem + P * PB;
    vec16* w = reinterpret_cast<vec16*>(smem + L::kW);
    float* vec = reinterpret_cast<float*>(smem + L::kVecs);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), n = lane % R, h = lane / R;
    const int64_t N = a.rows, groups = (N + CN - 1) / CN;
    float16_t acc_a[3], acc_b[2];      // O, W1a, W1b; W2a, W2b
    float col_a[5], col_b[4];          // bo, b1a, b1b, gamma1, beta1; b2, -, gamma2, beta2
#pragma unroll
    for (int r = 0; r < 16; ++r) {
#pragma unroll
        for (int j = 0; j < 3; ++j) acc_a[j][r] = 0.f;
        acc_b[0][r] = acc_b[1][r] = 0.f;
    }
#pragma unroll
    for (int j = 0; j < 5; ++j) col_a[j] = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) col_b[j] = 0.f;
    if (wave < NC) {
        vec16* stage = reinterpret_cast<vec16*>(smem + L::kStage) + wave * RowShape<T, R>::kVecs;
        const int row = R * wave + n;
        // bf16 has the registers to ask for a group's rows in the group before it; float32 asks for the attention rows there, for the
        // others one after the other (64 K nodes in bf16: 32.0 us with every row asked for where it is needed, 29.5)
        constexpr bool AHEAD = P == 1;
        Raw<T, R> raw, raw_s2, raw_g, raw_x;
        const auto ask = [&](Raw<T, R>& r, const void* from, int64_t g) { fetch(r, reinterpret_cast<const T*>(from), Rows(NC * g + wave, N, R), lane); };
        ask(raw, a.attn, blockIdx.x);
        if (AHEAD) {
            ask(raw_s2, a.s2, blockIdx.x);
            ask(raw_g, a.g_in, blockIdx.x);
            ask(raw_x, a.x, blockIdx.x);
        }
        for (int64_t g0 = blockIdx.x; g0 < groups; g0 += gridDim.x) {
            const Rows rows(NC * g0 + wave, N, R);
            const int64_t after = g0 + gridDim.x < groups ? g0 + gridDim.x : g0;
            TileOf<R> y, ds2, dy, t;
            settle<T, false>(t, raw, stage, rows, lane);
            if (!AHEAD) ask(raw, a.s2, g0);
            __syncthreads();                                        // O
            linear<P, false>(y, t, w, vec + V_BO * kVec, lane);
            round_to<T>(y);
            __syncthreads();
            {
                TileOf<R> g;
                settle<T, false>(t, AHEAD ? raw_s2 : raw, stage, rows, lane);
                if (AHEAD) ask(raw_s2, a.s2, after);
                else ask(raw, a.g_in, g0);
                const float rstd = normalise<false>(t, a.eps2);
                settle<T, true>(g, AHEAD ? raw_g : raw, stage, rows, lane);
                if (AHEAD) ask(raw_g, a.g_in, after);
                col_b[3] += column_sums(g, lane);
                zero(ds2);
                ln_back(ds2, g, t, rstd, vec + V_GAMMA2 * kVec, h);
                TGT_EACH(i) t.set(i, t.get(i) * g.get(i));
                col_b[2] += column_sums(t, lane);
                round_to<T>(ds2);
                col_b[0] += column_sums(ds2, lane);
            }
            zero(dy);
#pragma unroll
            for (int j = 0; j < 2; ++j) {      // the two halves of the feed-forward features
                Frags<P, R> f;
                if (CUT_AGAIN) forget(y);      // (planes are formed again where they are used: there are no registers to keep them)
                __syncthreads();                                    // W1
                linear<P, false>(t, y, w, vec + (V_B1A + j) * kVec, lane);
                __syncthreads();
                const uint32_t on = relu<T>(t);
                put_tile_planes<PB, P>(p_x, row, h, t);
                if (CUT_AGAIN) forget(ds2);
                make_frags(f, ds2);
                put_planes<PB>(p_dy, row, h, f);
                __syncthreads();                                    // W2^T; planes of W2
                zero(t);
                gemm<P>(t, f, w, lane);
                TGT_EACH(i) t.set(i, on & (1u << i) ? stored(t.get(i), (const T*)nullptr) : 0.f);      // du
                col_a[1 + j] += column_sums(t, lane);
                if (CUT_AGAIN) forget(y);
                __syncthreads();
                put_tile_planes<PB, P>(p_x, row, h, y);
                make_frags(f, t);
                put_planes<PB>(p_dy, row, h, f);
                __syncthreads();                                    // W1^T; planes of W1
                gemm<P>(dy, f, w, lane);
                __syncthreads();
            }
            if (!AHEAD) ask(raw, a.x, g0);
            settle<T, false>(t, AHEAD ? raw_x : raw, stage, rows, lane);
            if (AHEAD) ask(raw_x, a.x, after);
            else ask(raw, a.attn, g0);
            TGT_EACH(i) t.set(i, t.get(i) + y.get(i));              // s1
            const MeanRstd stat = row_stats<false>(t, a.eps1);
            TGT_EACH(i) t.set(i, (stored(t.get(i), (const T*)nullptr) - stat.mean) * stat.rstd);
            col_a[4] += column_sums(ds2, lane);
            zero(y);
            ln_back(y, ds2, t, stat.rstd, vec + V_GAMMA1 * kVec, h);      // of x and of y alike
            TGT_EACH(i) t.set(i, t.get(i) * ds2.get(i));
            col_a[3] += column_sums(t, lane);
            round_to<T>(y);
            put_rows(reinterpret_cast<T*>(a.g_out), y, stage, rows, lane);
            TGT_EACH(i) dy.set(i, stored(stored(dy.get(i), (const T*)nullptr) + y.get(i), (const T*)nullptr));
            col_a[0] += column_sums(dy, lane);
            settle<T, false>(t, raw, stage, rows, lane);
            ask(raw, a.attn, after);
            Frags<P, R> f;
            put_tile_planes<PB, P>(p_x, row, h, t);
            make_frags(f, dy);
            put_planes<PB>(p_dy, row, h, f);
            __syncthreads();                                        // O^T; planes of O
            zero(dy);
            gemm<P>(dy, f, w, lane);
            __syncthreads();
            put_rows(reinterpret_cast<T*>(a.d_attn), dy, stage, rows, lane);
            put_node_side<T>(dy, t, a.Z, a.nd, a.heads, rows.first + n, h, n < rows.left);
        }
    } else {
        const int q = wave - NC, base_dy = operand_base(q >> 1, lane), base_x = operand_base(q & 1, lane);
        const vec16 *fw = reinterpret_cast<const vec16*>(a.w), *bw = reinterpret_cast<const vec16*>(a.w_back);
        WeightsAhead<FV> next;
        next.fetch(fw + W_O * FV);
        copy_direct<kVecs8 * kVec>(kBlockWaves * 64, vec, a.vec, NC * 64);
        landed();
        for (int64_t g0 = blockIdx.x; g0 < groups; g0 += gridDim.x) {
            next.hand_over(w, fw + W_1A * FV);          // O
            __syncthreads();
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                next.hand_over(w, bw + (W_2A + j) * FV);      // W1
                __syncthreads();
                next.hand_over(w, bw + (W_1A + j) * FV);      // W2^T
                node_product<P, PB>(acc_b[j], p_dy, p_x, base_dy, base_x);
                __syncthreads();
                next.hand_over(w, j == 0 ? fw + W_1B * FV : bw + W_O * FV);      // W1^T
                node_product<P, PB>(acc_a[1 + j], p_dy, p_x, base_dy, base_x);
                __syncthreads();
            }
            next.hand_over(w, fw + W_O * FV);           // O^T
            node_product<P, PB>(acc_a[0], p_dy, p_x, base_dy, base_x);
            __syncthreads();
        }
    }
    float* buf = reinterpret_cast<float*>(smem);
    write_partial<L, 3, 5>(a.partial_a + (int64_t)blockIdx.x * (3 * 4096 + 5 * 64), acc_a, col_a, buf, wave, lane);
    write_partial<L, 2, 4>(a.partial_b + (int64_t)blockIdx.x * (2 * 4096 + 4 * 64), acc_b, col_b, buf, wave, lane);
}

template <typename T, bool NEXT> int run_fwd(const tgt_gt_fwd_args& a, hipStream_t st) {
    static std::atomic<uint64_t> done{0};
    const int waves = fwd_waves_for(a.rows, kFwdRows, kFwdWaves);
    if (int rc = allow_lds(reinterpret_cast<const void*>(&k_gt_fwd<T, NEXT>), gt_fwd_lds<T>(kFwdWaves), done)) return rc;
    hipLaunchKernelGGL((k_gt_fwd<T, NEXT>), dim3(fwd_grid(a.rows, kFwdRows, waves)), dim3(waves * 64), (gt_fwd_lds<T>(waves)), st, a);
    TGT_HIP_CHECK(hipGetLastError());
    return TGT_OK;
}
template <typename T, int R, int CN> int run_bwd(const tgt_gt_bwd_args& a, hipStream_t st) {
    using L = Bwd<T, R, CN, kVecs8>;
    static std::atomic<uint64_t> done{0};
    return launch(&k_gt_bwd<T, R, CN>, done, bwd_workers(a.rows), L::kThreads, L::kBytes, st, a);
}
bool dtype_ok(int dtype) { return dtype == TGT_DTYPE_F32 || dtype == TGT_DTYPE_BF16; }

}  // namespace
}  // namespace tgt

extern "C" {

int tgt_gt_fwd(const tgt_gt_fwd_args* a, void* stream) {
    using namespace tgt;
    if (!a || a->rows < 0 || !dtype_ok(a->dtype) || !a->attn || !a->x || !a->x_out || !a->w || !a->vec) return bad("tgt_gt_fwd", "null or bad argument");
    if (a->q && (!a->k || !a->v || !a->w_next || !a->v_next)) return bad("tgt_gt_fwd", "q needs k, v, w_next and v_next");
    if (a->rows == 0) return TGT_OK;
    const hipStream_t st = (hipStream_t)stream;
    KernelTimer t(KS_GT_FWD, st);
    if (a->dtype == TGT_DTYPE_F32) return a->q ? run_fwd<float, true>(*a, st) : run_fwd<float, false>(*a, st);
    return a->q ? run_fwd<nbf16, true>(*a, st) : run_fwd<nbf16, false>(*a, st);
}

int tgt_gt_bwd(const tgt_gt_bwd_args* a, void* stream) {
    using namespace tgt;
    if (!a || a->rows < 1 || !dtype_ok(a->dtype) || !a->g_in || !a->x || !a->attn || !a->s2 || !a->w || !a->w_back || !a->vec || !a->g_out || !a->d_attn || !a->partial_a ||
        !a->partial_b)
        return bad("tgt_gt_bwd", "null or bad argument");
    if (!a->nd || !a->Z || (a->heads != 8 && a->heads != 4 && a->heads != 2)) return bad("tgt_gt_bwd", "nd, Z and 8, 4 or 2 heads");
    const hipStream_t st = (hipStream_t)stream;
    KernelTimer t(KS_GT_BWD, st);
    // (node_roles.h; eight chain waves of sixteen rows and the blocks' accumulators of five weights do not fit the registers in float32: 64 nodes
    // per group as soon as that leaves the number of workgroups alone - 64 K nodes 77 us, 200 K 222, with 128 nodes and 32 rows per
    // wave 80 and 232 -, those in between)
    if (a->dtype == TGT_DTYPE_F32) return groups_of_64(a->rows, true) || a->rows >= (int64_t)128 * num_cus() ? run_bwd<float, 16, 64>(*a, st) : run_bwd<float, 32, 128>(*a, st);
    return groups_of_64(a->rows, false) ? run_bwd<nbf16, 16, 64>(*a, st) : run_bwd<nbf16, 16, 128>(*a, st);
}

}  // extern "C"
