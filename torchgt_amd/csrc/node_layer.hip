// The node-local part of a Graphormer encoder layer (models/graphormer_dist_node_level.py:246-314 and
// models/graphormer_graph_level.py:267-306), hidden and feed-forward width 64, as one forward and one or two backward kernels.
//
//   forward   [attention rows a, residual stream s] -> s1 = s + a Wo^T + bo;  s' = s1 + W2 gelu(W1 LN2(s1) + b1) + b2
//             and, in the same pass, what the next layer's attention reads: q, k, v = LN1(s') W^T + b - or the class
//             log-probabilities log_softmax(LN(s') Wh^T + bh) behind the last layer
//   backward  k_node_bwd_pre:  dq, dk, dv, ds' (residual) -> ds', gradients of Wq / Wk / Wv and LN1 (and the same for the
//             classes: one weight, d log_softmax in front)
//             k_node_bwd_post: ds' -> ds (residual), da, gradients of Wo, W1, W2 and LN2, and (1 / (Z + eps), da . a) per
//             node and head, which the sparse attention's backward starts from
//             k_node_bwd_both: the first for a layer and the second for the layer in front of it, as one launch (node level)
//
// What bounds them and why this shape.  As one kernel per linear, LayerNorm and activation the part moves 29 rows of 64
// features per node forward and 47 backward through memory; here it moves 6 and 12 (q, k, v, the residual stream and the
// attention rows; the intermediate activations are recomputed in the backward from s and a: two products, against two rows
// written and read).  A wave takes 32 or 16 nodes and keeps them in registers through the whole chain (node_tile.h); the waves of
// a workgroup share the packed weights in LDS.  Weight gradients contract over nodes: in the backward kernels two to eight waves carry
// 32 or 16 nodes each through the chain and put the bf16 planes of both operands into LDS, four others keep one 32 x 32 block of every
// weight gradient each and add the products over these 64 or 128 nodes beside it (node_roles.h).  Which of the sizes a call takes is said with
// both sides' times at the entry points below and at `groups_of_64`.
#include "node_roles.h"
#include "class_rows.h"
#include "node_pack.h"

namespace tgt {
namespace {

// workgroup = one (weight, direction); the workgroups behind the weights copy vectors
constexpr int kPackThreads = 512;
template <typename T> __global__ __launch_bounds__(kPackThreads) void k_node_pack(const PackArgs a) { pack_block<T, kPackThreads>(a, blockIdx.x); }

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
template <typename T, bool SAME, int R> __device__ __forceinline__ void gelu(TileOf<R>& u) {
    TGT_EACH(i) {
        const float v = stored(u.get(i), (const T*)nullptr);
        float bell;
        if constexpr (SAME) u.set(i, act_value<false>(v));
        else u.set(i, v * cdf_and_bell<T, SAME>(v, bell));
        if (i % 8 == 7) fence_schedule();
    }
}
template <typename T, bool SAME, int R> __device__ __forceinline__ void gelu(TileOf<R>& u, TileOf<R>& slope) {
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

// waves of a workgroup at most (float32 of 32 rows: as many as their row images leave room for)
template <typename T, int R, bool SAME> constexpr int fwd_waves() { return R == 32 && SAME ? 8 : (R == 32 && sizeof(T) == 4 ? 10 : 16); }
// bf16 keeps all weights of a launch in LDS for the life of the workgroup; float32 planes of six weights (144 KB) do not
// leave room for the row images, so its two halves take turns (the L2 has them)
template <typename T, bool POST, int NEXT> constexpr int fwd_resident_mats() {
    const int post = POST ? 3 : 0, next = NEXT == NEXT_QKV ? 3 : (NEXT == NEXT_CLASSES ? 1 : 0);
    return sizeof(T) == 4 ? (post > next ? post : next) : post + next;
}
template <typename T, int R, bool POST, int NEXT> constexpr int fwd_lds(int waves) {
    return fwd_resident_mats<T, POST, NEXT>() * kFragVecs<Num<T>::P> * 16 + 10 * kVec * 4 + waves * RowShape<T, R>::kVecs * 16;
}

template <typename T, int R, bool SAME, bool POST, int NEXT>
__global__ __launch_bounds__((fwd_waves<T, R, SAME>() * 64)) void k_node_fwd(const tgt_node_fwd_args a) {
    constexpr int P = Num<T>::P, FV = kFragVecs<P>;
    constexpr bool RESIDENT = sizeof(T) == 2;
    constexpr int NMP = NEXT == NEXT_QKV ? 3 : (NEXT == NEXT_CLASSES ? 1 : 0);
    using Shape = RowShape<T, R>;
    extern __shared__ __align__(16) unsigned char smem[];
    vec16* w = reinterpret_cast<vec16*>(smem);
    vec16* w_next = w + (RESIDENT && POST ? 3 * FV : 0);
    float* vec = reinterpret_cast<float*>(w + fwd_resident_mats<T, POST, NEXT>() * FV);
    float* vn = vec + 5 * kVec;
    const int threads = blockDim.x, NW = threads >> 6;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane / R;
    vec16* stage = reinterpret_cast<vec16*>(vec + 10 * kVec) + wave * Shape::kVecs;
    const int64_t N = a.rows, tiles = (N + R - 1) / R;
    Raw<T, R> raw_a, raw_s;
    const auto ask = [&](int64_t t0) {
        const Rows rows(t0 + wave, N, R);      // (a wave without rows reads the first one)
        fetch(raw_s, reinterpret_cast<const T*>(a.s_in), rows, lane);
        if (POST) fetch(raw_a, reinterpret_cast<const T*>(a.attn), rows, lane);
    };
    const vec16 *w_post = reinterpret_cast<const vec16*>(a.w_post), *w_after = reinterpret_cast<const vec16*>(a.w_next);
    const int64_t first = (int64_t)blockIdx.x * NW;
    ask(first);
    if constexpr (POST) copy_direct<3 * FV>(threads, w, w_post);
    if constexpr (NEXT != NEXT_NONE && (RESIDENT || !POST)) copy_direct<NMP * FV>(threads, w_next, w_after);
    if constexpr (POST) copy_direct<5 * kVec>(threads, vec, a.v_post);
    if constexpr (NEXT != NEXT_NONE) copy_direct<(2 + NMP) * kVec>(threads, vn, a.v_next);
    landed();
    __syncthreads();
    for (int64_t t0 = first;;) {
        const Rows rows(t0 + wave, N, R);
        const int64_t row0 = (t0 + wave) * R;
        const bool active = rows.left > 0;
        TileOf<R> s;
        if (active) {
            if (!POST && row0 < a.tokens) {      // the global tokens in front of the nodes: from their table, and into the stream
                constexpr int PP = Shape::kPieces, PER = Shape::kPer;
#pragma unroll
                for (int i = 0; i < Shape::kAcc; ++i) {
                    const int64_t r = row0 + i * PER + lane / PP;
                    if (r < a.tokens) {
                        raw_s.v[i] = reinterpret_cast<const vec16*>(a.token)[r * PP + lane % PP];
                        reinterpret_cast<vec16*>(a.s_out)[r * PP + lane % PP] = raw_s.v[i];
                    }
                }
            }
            settle<T, false>(s, raw_s, stage, rows, lane);
            if (POST) {
                TileOf<R> x, y;
                settle<T, false>(x, raw_a, stage, rows, lane);
                linear<P, SAME>(y, x, w, vec, lane);
                TGT_EACH(i) s.set(i, s.get(i) + stored(y.get(i), (const T*)nullptr));      // s1 = s + (a Wo^T + bo)
                x = s;
                normalise<SAME>(x, a.eps_post);
                affine(x, x, vec + kVec, vec + 2 * kVec, g);      // y2
                linear<P, SAME>(y, x, w + FV, vec + 3 * kVec, lane);    // u
                gelu<T, SAME>(y);
                linear<P, SAME>(x, y, w + 2 * FV, vec + 4 * kVec, lane);
                TGT_EACH(i) s.set(i, stored(s.get(i), (const T*)nullptr) + stored(x.get(i), (const T*)nullptr));      // s'
                put_rows(reinterpret_cast<T*>(a.s_out), s, stage, rows, lane);
            }
        }
        constexpr bool SWAP = !RESIDENT && POST && NEXT != NEXT_NONE;
        if constexpr (SWAP) replace_weights<NMP * FV>(threads, w, w_after);
        if (NEXT && active) {
            normalise<SAME>(s, a.eps_next);
            affine(s, s, vn, vn + kVec, g);
            if constexpr (NEXT == NEXT_QKV) {
                // float32: sixteen rows' planes fit beside a product, thirty-two rows' are cut again for each of the three
                using Operand = std::conditional_t<R == 16, Frags<P, R>, TileOf<R>>;
                Operand f;
                if constexpr (R == 16) make_frags(f, s);
                else f = s;
#pragma unroll
                for (int j = 0; j < 3; ++j) {
                    TileOf<R> y;
                    linear<P, SAME>(y, f, w_next + j * FV, vn + (2 + j) * kVec, lane);
                    put_rows(reinterpret_cast<T*>(j == 0 ? a.q : (j == 1 ? a.k : a.v)), y, stage, rows, lane);
                }
            } else {
                TileOf<R> y;
                linear<P, SAME>(y, s, w_next, vn + 2 * kVec, lane);
                put_classes<T, false>(reinterpret_cast<T*>(a.logp), y, a.linear, a.classes, a.tokens, row0, N, stage, lane);
            }
        }
        t0 += (int64_t)gridDim.x * NW;
        if (t0 >= tiles) break;
        ask(t0);
        if constexpr (SWAP) replace_weights<3 * FV>(threads, w, w_post);
    }
}

// ---- backward of the part in front of an attention (or of the classes) ------------------------------------------------------
// NORM false (GT): q, k, v are made of the rows s themselves.
// What a chain wave has at hand
template <typename T, int R, int CN> struct Chain {
    using L = Bwd<T, R, CN>;
    vec16* stage;
    const vec16* w;
    const float* vec;
    unsigned char *p_dy, *p_x;
    int lane, wave;
    // its rows of a group
    __device__ __forceinline__ int64_t tile(int64_t group) const { return (int64_t)L::kChain * group + wave; }
    __device__ __forceinline__ Rows rows(int64_t group, int64_t N) const { return Rows(tile(group), N, R); }
};
// and a block wave
// (of BW; with two of them a wave has the two blocks of its columns)
template <int P, int PB, int BW = kBlockWaves> struct Blocks {
    static constexpr int FV = kFragVecs<P>, EACH = 4 / BW;
    vec16* w;
    unsigned char *p_dy, *p_x;
    int base_dy[EACH], base_x;
    WeightsAhead<FV, BW * 64> next;
    __device__ __forceinline__ Blocks(vec16* w_, unsigned char* planes, int q, int lane) : w(w_), p_dy(planes), p_x(planes + P * PB), base_x(operand_base(q & 1, lane)) {
#pragma unroll
        for (int i = 0; i < EACH; ++i) base_dy[i] = operand_base((q + i * BW) >> 1, lane);
    }
    __device__ __forceinline__ void add(float16_t* acc) const {
#pragma unroll
        for (int i = 0; i < EACH; ++i) node_product<P, PB>(acc[i], p_dy, p_x, base_dy[i], base_x);
    }
};

// One group: d = g_in + what the products and LayerNorm make of dq, dk, dv (or of the classes' gradients).  raw_s and raw_d come with s and
// the first of the gradients; then_s and then_d say what is asked for when they are free again.
template <typename T, int R, int CN, bool CLASSES, bool NORM, typename F, typename G>
__device__ __forceinline__ void pre_chain(const tgt_node_bwd_pre_args& a, const Chain<T, R, CN>& me, int64_t group, Raw<T, R>& raw_s, Raw<T, R>& raw_d, float (&col)[(CLASSES ? 1 : 3) + 2],
                                          TileOf<R>& d, const F& then_s, const G& then_d) {
    using L = Bwd<T, R, CN>;
    constexpr int P = Num<T>::P, NM = CLASSES ? 1 : 3, PB = L::kPlane;
    const T* src[3] = {reinterpret_cast<const T*>(a.dq), reinterpret_cast<const T*>(a.dk), reinterpret_cast<const T*>(a.dv)};
    const int64_t N = a.rows;
    const int lane = me.lane, row = R * me.wave + lane % R, h = lane / R;
    const Rows rows = me.rows(group, N);
    TileOf<R> xhat, dy;
    Frags<P, R> f;
    settle<T, false>(xhat, raw_s, me.stage, rows, lane);
    float rstd = 1.f;
    if constexpr (NORM) rstd = normalise<false>(xhat, a.eps);
    zero(dy);
#pragma unroll
    for (int j = 0; j < NM; ++j) {
        if (CLASSES) ClassGrads<T, R>(reinterpret_cast<const T*>(a.dlogp), reinterpret_cast<const T*>(a.logp), a.linear, a.classes, a.tokens, me.tile(group) * R, N, me.stage, lane).settle(d);
        else {
            settle<T, true>(d, raw_d, me.stage, rows, lane);
            fetch(raw_d, j + 1 < NM ? src[j + 1] : reinterpret_cast<const T*>(a.g_in), rows, lane);
        }
        make_frags(f, d);
        col[j] += column_sums(d, lane);
        __syncthreads();                       // weight j is there; j = 0: the planes are free
        gemm<P>(dy, f, me.w, lane);            // beside product j - 1 of the block waves
        if (j > 0) __syncthreads();            // product j - 1 is done
        else {
            TileOf<R> y;
            if constexpr (NORM) affine(y, xhat, me.vec, me.vec + kVec, h);
            else y = xhat;
            put_tile_planes<PB, P>(me.p_x, row, h, y);
        }
        put_planes<PB>(me.p_dy, row, h, f);
        __syncthreads();                       // planes j are there, weight j has been used
    }
    then_s();
    TGT_EACH(i) dy.set(i, stored(dy.get(i), (const T*)nullptr));
    if constexpr (NORM) {
        col[NM + 1] += column_sums(dy, lane);
        TGT_EACH(i) d.set(i, dy.get(i) * xhat.get(i));
        col[NM] += column_sums(d, lane);
    }
    if (CLASSES) zero(d);
    else settle<T, true>(d, raw_d, me.stage, rows, lane);
    then_d();
    if constexpr (NORM) ln_back(d, dy, xhat, rstd, me.vec, h);
    else TGT_EACH(i) d.set(i, d.get(i) + dy.get(i));
}
// The products beside it.  `after`: the weight that the group's next step begins with.
template <int NM, int P, int PB> __device__ __forceinline__ void pre_blocks(Blocks<P, PB>& me, const vec16* weights, const vec16* after, float16_t (&acc)[NM]) {
    constexpr int FV = kFragVecs<P>;
    me.next.put(me.w);
    me.next.fetch(NM > 1 ? weights + FV : after);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < NM; ++j) {
        __syncthreads();                       // planes j
        if (j + 1 < NM) {
            me.next.put(me.w);
            me.next.fetch(j + 2 < NM ? weights + (j + 2) * FV : after);
            __syncthreads();                   // weight j + 1
        }
        me.add(acc + j);
        if (j + 1 < NM) __syncthreads();       // product j is done
    }
}

template <int N> __device__ __forceinline__ void clear(float16_t (&acc)[N]) {
#pragma unroll
    for (int j = 0; j < N; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[j][r] = 0.f;
}
template <int N> __device__ __forceinline__ void clear(float (&col)[N]) {
#pragma unroll
    for (int j = 0; j < N; ++j) col[j] = 0.f;
}

// What the kernels begin with, and the block waves' part of it
#define TGT_BWD_ROLES(...)                                                                                                       \
    using L = Bwd<T, R, CN, NV, ##__VA_ARGS__>;                                                                                                 \
    constexpr int P = Num<T>::P, PB = L::kPlane, NC = L::kChain;                                                                 \
    extern __shared__ __align__(16) unsigned char smem[];                                                                        \
    vec16* w = reinterpret_cast<vec16*>(smem + L::kW);                                                                           \
    float* vec = reinterpret_cast<float*>(smem + L::kVecs);                                                                      \
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);                                 \
    const Chain<T, R, CN> chain{reinterpret_cast<vec16*>(smem + L::kStage) + wave * RowShape<T, R>::kVecs, w, vec, smem, smem + P * PB, lane, wave}
#define TGT_BWD_BLOCKS() Blocks<P, PB, L::kBlocks> blocks(w, smem, wave - NC, lane)

template <typename T, int R, int CN, bool CLASSES, bool NORM>
__global__ __launch_bounds__((Bwd<T, R, CN>::kThreads)) void k_node_bwd_pre(const tgt_node_bwd_pre_args a) {
    constexpr int NV = 5, NM = CLASSES ? 1 : 3;
    TGT_BWD_ROLES();
    const int64_t N = a.rows, groups = (N + CN - 1) / CN;
    if constexpr (NORM) copy_vecs<2 * kVec / 4, L::kThreads>(reinterpret_cast<vec16*>(vec), reinterpret_cast<const vec16*>(a.v_next));
    __syncthreads();
    float16_t acc[NM];
    float col[NM + 2];
    clear(acc); clear(col);
    if (wave < NC) {
        Raw<T, R> raw_s, raw_d;
        const auto ask_s = [&](int64_t g) { fetch(raw_s, reinterpret_cast<const T*>(a.s), chain.rows(g, N), lane); };
        const auto ask_d = [&](int64_t g) { if (!CLASSES) fetch(raw_d, reinterpret_cast<const T*>(a.dq), chain.rows(g, N), lane); };
        ask_s(blockIdx.x);
        ask_d(blockIdx.x);
        for (int64_t g0 = blockIdx.x; g0 < groups; g0 += gridDim.x) {
            TileOf<R> d;
            const int64_t ahead = g0 + gridDim.x;
            pre_chain<T, R, CN, CLASSES, NORM>(a, chain, g0, raw_s, raw_d, col, d, [&]() { if (ahead < groups) ask_s(ahead); }, [&]() { if (ahead < groups) ask_d(ahead); });
            put_rows(reinterpret_cast<T*>(a.g_out), d, chain.stage, chain.rows(g0, N), lane);
            if (a.d_token && chain.tile(g0) < (a.tokens + R - 1) / R) put_rows(reinterpret_cast<T*>(a.d_token), d, chain.stage, Rows(chain.tile(g0), a.tokens, R), lane);
        }
    } else {
        TGT_BWD_BLOCKS();
        const vec16* weights = reinterpret_cast<const vec16*>(a.w_back);
        blocks.next.fetch(weights);
        for (int64_t g0 = blockIdx.x; g0 < groups; g0 += gridDim.x) pre_blocks<NM>(blocks, weights, weights, acc);
    }
    write_partial<L, NM, NM + 2>(a.partial + (int64_t)blockIdx.x * (NM * 4096 + (NM + 2) * 64), acc, col, reinterpret_cast<float*>(smem), wave, lane);
}

// ---- backward of the part behind an attention -------------------------------------------------------------------------------
// One group: g = ds' in, ds out, and da (d_attn) and the sparse attention's nd to memory.  take_g: hands the group's g over; then: asks for the
// next group's rows when the registers of these are free.
template <typename T, int R, int CN, bool SAME, typename F, typename G>
__device__ __forceinline__ void post_chain(const tgt_node_bwd_post_args& a, const Chain<T, R, CN>& me, const Rows& rows, Raw<T, R>& raw_a, Raw<T, R>& raw_s, float (&col)[5],
                                           const F& take_g, const G& then) {
    using L = Bwd<T, R, CN>;
    constexpr int P = Num<T>::P, PB = L::kPlane;
    constexpr bool KEEP = P == 1 || CN == 64;      // whether there are registers for the planes of LayerNorm's output
    const int lane = me.lane, row = R * me.wave + lane % R, h = lane / R;
    const vec16* w = me.w;
    const float* vec = me.vec;
    vec16* stage = me.stage;
    unsigned char *p_dy = me.p_dy, *p_x = me.p_x;
    TileOf<R> g, xhat, slope, t;
    Frags<P, R> f, fy;      // fy: LayerNorm's output, formed again from xhat where it is not kept
    settle<T, false>(t, raw_a, stage, rows, lane);
    make_frags(f, t);
    settle<T, false>(xhat, raw_s, stage, rows, lane);
    take_g(g);
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
    put_tile_planes<PB, P>(p_x, row, h, t);
    make_frags(f, g);
    put_planes<PB>(p_dy, row, h, f);
    __syncthreads();                                        // planes of W2; W2^T
    zero(t);
    gemm<P>(t, f, w, lane);                                 // d gelu, beside product W2
    TGT_EACH(i) t.set(i, stored(t.get(i) * slope.get(i), (const T*)nullptr));      // du
    col[1] += column_sums(t, lane);
    make_frags(f, t);
    if (!KEEP) {
        forget(xhat);
        affine(t, xhat, vec + kVec, vec + 2 * kVec, h);
    }
    __syncthreads();                                        // product W2 is done, W2^T has been used
    put_planes<PB>(p_dy, row, h, f);
    if constexpr (KEEP) put_planes<PB>(p_x, row, h, fy);
    else put_tile_planes<PB, P>(p_x, row, h, t);
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
    put_planes<PB>(p_dy, row, h, f);
    put_tile_planes<PB, P>(p_x, row, h, t);
    __syncthreads();                                        // planes of Wo; Wo^T
    if (P == 1) then();      // float32 has the registers only after the products
    zero(g);
    gemm<P>(g, f, w, lane);                                 // da, beside product Wo
    __syncthreads();                                        // Wo^T has been used
    put_rows(reinterpret_cast<T*>(a.d_attn), g, stage, rows, lane);
    if (a.nd) put_node_side<T>(g, t, a.Z, a.nd, a.heads, rows.first + lane % R, h, lane % R < rows.left);
    if (P != 1) then();
}
template <int P, int PB, int BW> __device__ __forceinline__ void post_blocks(Blocks<P, PB, BW>& me, const vec16* fw, const vec16* bw, const vec16* after, float16_t (&acc)[3 * (4 / BW)]) {
    constexpr int FV = kFragVecs<P>, EACH = 4 / BW;
    me.next.hand_over(me.w, fw + FV);             // Wo, then on to W1
    __syncthreads();
    me.next.hand_over(me.w, bw + 2 * FV);         // W1
    __syncthreads();
    me.next.hand_over(me.w, bw + FV);             // W2^T and the planes of W2
    me.add(acc + 2 * EACH);
    __syncthreads();
    me.next.hand_over(me.w, bw);                  // W1^T and the planes of W1
    me.add(acc + 1 * EACH);
    __syncthreads();
    me.next.hand_over(me.w, after);               // Wo^T and the planes of Wo
    me.add(acc);
    __syncthreads();
}

template <typename T, int R, int CN> constexpr int post_block_waves() { return CN / R + kBlockWaves <= 8 || R == 16 ? kBlockWaves : 2; }
template <typename T, int R, int CN, bool SAME>
__global__ __launch_bounds__((Bwd<T, R, CN, 5, post_block_waves<T, R, CN>()>::kThreads)) void k_node_bwd_post(const tgt_node_bwd_post_args a) {
    constexpr int NV = 5, BW = post_block_waves<T, R, CN>();
    TGT_BWD_ROLES(BW);
    const int64_t N = a.rows, groups = (N + CN - 1) / CN;
    copy_vecs<5 * kVec / 4, L::kThreads>(reinterpret_cast<vec16*>(vec), reinterpret_cast<const vec16*>(a.v_post));
    __syncthreads();
    float16_t acc[3 * (4 / BW)];       // Wo, W1, W2
    float col[5];           // bo, b1, b2, gamma, beta
    clear(acc); clear(col);
    if (wave < NC) {
        Raw<T, R> raw_a, raw_s, raw_g;
        const auto ask = [&](int64_t g) {
            const Rows rows = chain.rows(g, N);
            fetch(raw_a, reinterpret_cast<const T*>(a.attn), rows, lane);
            fetch(raw_s, reinterpret_cast<const T*>(a.s), rows, lane);
            fetch(raw_g, reinterpret_cast<const T*>(a.g_in), rows, lane);
        };
        ask(blockIdx.x);
        for (int64_t g0 = blockIdx.x; g0 < groups; g0 += gridDim.x) {
            const Rows rows = chain.rows(g0, N);
            post_chain<T, R, CN, SAME>(a, chain, rows, raw_a, raw_s, col, [&](TileOf<R>& g) { settle<T, true>(g, raw_g, chain.stage, rows, lane); },
                                       [&]() { if (g0 + gridDim.x < groups) ask(g0 + gridDim.x); });
        }
    } else {
        TGT_BWD_BLOCKS();
        const vec16 *fw = reinterpret_cast<const vec16*>(a.w_post), *bw = reinterpret_cast<const vec16*>(a.w_back);
        blocks.next.fetch(fw);
        for (int64_t g0 = blockIdx.x; g0 < groups; g0 += gridDim.x) post_blocks(blocks, fw, bw, fw, acc);
    }
    write_partial<L, 3, 5>(a.partial + (int64_t)blockIdx.x * (3 * 4096 + 5 * 64), acc, col, reinterpret_cast<float*>(smem), wave, lane);
}

// The part in front of an attention (or the classes) and the part behind the attention before it, one after the other for a group: what
// passes between them (g_out of the one, g_in of the other) stays in registers, and a launch's first and last microseconds
// are there once.  A training step of four layers as a replayed graph, us, two launches / one: float32 4 K nodes 330 / 323, 16 K 398 / 389, 64 K
// 1010 / 1001; bf16 220 / 214, 295 / 283, 567 / 541 (and four launches less of host time).
constexpr int kBothVecs = 7;
template <typename T, int R, int CN, bool CLASSES>
__global__ __launch_bounds__((Bwd<T, R, CN, kBothVecs>::kThreads)) void k_node_bwd_both(const tgt_node_bwd_pre_args a, const tgt_node_bwd_post_args b) {
    constexpr int NV = kBothVecs, NM = CLASSES ? 1 : 3;
    TGT_BWD_ROLES();
    const int64_t N = a.rows, groups = (N + CN - 1) / CN;
    copy_vecs<2 * kVec / 4, L::kThreads>(reinterpret_cast<vec16*>(vec), reinterpret_cast<const vec16*>(a.v_next));
    copy_vecs<5 * kVec / 4, L::kThreads>(reinterpret_cast<vec16*>(vec + 2 * kVec), reinterpret_cast<const vec16*>(b.v_post));
    __syncthreads();
    float16_t acc[NM], acc_b[3];
    float col[NM + 2], col_b[5];
    clear(acc); clear(col); clear(acc_b); clear(col_b);
    if (wave < NC) {
        Chain<T, R, CN> behind = chain;
        behind.vec = vec + 2 * kVec;
        Raw<T, R> raw_s, raw_d, raw_a;
        const auto ask = [&](int64_t g) {
            const Rows rows = chain.rows(g, N);
            fetch(raw_s, reinterpret_cast<const T*>(a.s), rows, lane);
            if (!CLASSES) fetch(raw_d, reinterpret_cast<const T*>(a.dq), rows, lane);
        };
        ask(blockIdx.x);
        for (int64_t g0 = blockIdx.x; g0 < groups; g0 += gridDim.x) {
            TileOf<R> d;
            const Rows rows = chain.rows(g0, N);
            pre_chain<T, R, CN, CLASSES, true>(a, chain, g0, raw_s, raw_d, col, d, [&]() { fetch(raw_a, reinterpret_cast<const T*>(b.attn), rows, lane); },
                                               [&]() { fetch(raw_s, reinterpret_cast<const T*>(b.s), rows, lane); });
            post_chain<T, R, CN, false>(b, behind, rows, raw_a, raw_s, col_b,
                                        [&](TileOf<R>& g) { TGT_EACH(i) g.set(i, lane % R < rows.left ? stored(d.get(i), (const T*)nullptr) : 0.f); },
                                        [&]() { if (g0 + gridDim.x < groups) ask(g0 + gridDim.x); });
        }
    } else {
        TGT_BWD_BLOCKS();
        const vec16 *weights = reinterpret_cast<const vec16*>(a.w_back), *fw = reinterpret_cast<const vec16*>(b.w_post), *bw = reinterpret_cast<const vec16*>(b.w_back);
        blocks.next.fetch(weights);
        for (int64_t g0 = blockIdx.x; g0 < groups; g0 += gridDim.x) {
            pre_blocks<NM>(blocks, weights, fw, acc);
            post_blocks(blocks, fw, bw, weights, acc_b);
        }
    }
    write_partial<L, NM, NM + 2>(a.partial + (int64_t)blockIdx.x * (NM * 4096 + (NM + 2) * 64), acc, col, reinterpret_cast<float*>(smem), wave, lane);
    __syncthreads();
    write_partial<L, 3, 5>(b.partial + (int64_t)blockIdx.x * (3 * 4096 + 5 * 64), acc_b, col_b, reinterpret_cast<float*>(smem), wave, lane);
}

// ---- sums of the partials -----------------------------------------------------------------------------------------------
constexpr int kMaxSums = 26, kMaxOut = 8;
struct SumArgs {
    const float* partial[kMaxSums];
    int workers[kMaxSums], n[kMaxSums];
    void* out[kMaxSums][kMaxOut];      // mats x 4096 elements, then vectors of 64 (a null entry is not wanted)
    int16_t mats[kMaxSums], rows[kMaxSums], ld[kMaxSums];   // rows: of the 64 in each matrix and the vectors that follow them (classes)
    int count;                         // blockIdx.y behind them: the sum of another kernel's partials
    tgt_reduce_desc other;
};

// 64 consecutive elements x 16 slices of the workers per workgroup: slices in worker order, then the slice sums in order.  Bound by
// its reads, 50 KB of partials from every worker of every launch of a backward (108 MB for four Graphormer layers): sixteen lanes of a
// wave take 16 bytes each of a slice's 64 elements, eight workers in flight.  A lane per element and a wave per slice / this / 256 elements
// and a wave per slice, us with 64, 250 and 256 workers of four layers: 14.2 / 8.9 / 8.9, 24.3 / 19.8 / 20.0, 27.2 / 26.3 / 25.9 (GT: 34 / 34 / 39).
// `other` (of the first linear's weight gradient: slices and order are those of k_reduce_partials, so are the bits) as a launch of its own / beside the layers:
// 4 K nodes 6.5 + 4.0 / 6.7, 64 K 24.4 + 4.8 / 27.1, GT in bf16 32.3 + 4.1 / 32.8.
constexpr int kSumElems = 64;
template <int W> __device__ __forceinline__ void add_workers(float4& s, const float* __restrict__ src, int64_t n) {
    float4 t[W];
#pragma unroll
    for (int i = 0; i < W; ++i) t[i] = *reinterpret_cast<const float4*>(src + i * n);
#pragma unroll
    for (int i = 0; i < W; ++i) { s.x += t[i].x; s.y += t[i].y; s.z += t[i].z; s.w += t[i].w; }
}
template <typename T> __global__ __launch_bounds__(256) void k_node_sums(const SumArgs a) {
    __shared__ float part[16][kSumElems];
    const int d = blockIdx.y, e0 = blockIdx.x * kSumElems;
    const bool other = d == a.count;
    const int n = other ? a.other.n : a.n[d], workers = other ? a.other.workers : a.workers[d];      // (n is a multiple of 64)
    if (e0 >= n) return;
    {
        const int sl = threadIdx.x >> 4, el = 4 * (threadIdx.x & 15);
        const int w0 = (int)((int64_t)workers * sl / 16), w1 = (int)((int64_t)workers * (sl + 1) / 16);
        const float* __restrict__ src = (other ? a.other.partial : a.partial[d]) + e0 + el;
        float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
        int w = w0;
        for (; w + 8 <= w1; w += 8) add_workers<8>(s, src + (int64_t)w * n, n);
        for (; w + 2 <= w1; w += 2) add_workers<2>(s, src + (int64_t)w * n, n);
        if (w < w1) add_workers<1>(s, src + (int64_t)w * n, n);
        *reinterpret_cast<float4*>(&part[sl][el]) = s;
    }
    __syncthreads();
    if (threadIdx.x < kSumElems) {
        const int e = e0 + threadIdx.x;
        float t = 0.f;
#pragma unroll
        for (int i = 0; i < 16; ++i) t += part[i][threadIdx.x];
        if (other) {
            int seg = 0;
            for (int i = 1; i < a.other.n_out; ++i)
                if (e >= a.other.begin[i]) seg = i;
            if (a.other.out[seg]) reinterpret_cast<T*>(a.other.out[seg])[e - a.other.begin[seg]] = to_elem<T>(t);
            return;
        }
        const int mats = a.mats[d], rows = a.rows[d];
        const int seg = e < mats * 4096 ? e >> 12 : mats + ((e - mats * 4096) >> 6), at = e < mats * 4096 ? e & 4095 : (e - mats * 4096) & 63;
        const int limit = seg < mats ? rows * 64 : (seg < 2 * mats ? rows : 64);
        if (a.out[d][seg] && at < limit) reinterpret_cast<T*>(a.out[d][seg])[seg < mats ? (at >> 6) * a.ld[d] + (at & 63) : at] = to_elem<T>(t);
    }
}

template <typename T, int R, bool SAME, bool POST, int NEXT> int launch_fwd(const tgt_node_fwd_args& a, hipStream_t st) {
    static std::atomic<uint64_t> done{0};
    constexpr int most = fwd_waves<T, R, SAME>();
    const int waves = fwd_waves_for(a.rows, R, most);
    if (int rc = allow_lds(reinterpret_cast<const void*>(&k_node_fwd<T, R, SAME, POST, NEXT>), fwd_lds<T, R, POST, NEXT>(most), done)) return rc;
    hipLaunchKernelGGL((k_node_fwd<T, R, SAME, POST, NEXT>), dim3(fwd_grid(a.rows, R, waves)), dim3(waves * 64), (fwd_lds<T, R, POST, NEXT>(waves)), st, a);
    TGT_HIP_CHECK(hipGetLastError());
    return TGT_OK;
}
template <typename T, int R, bool SAME> int dispatch_fwd(const tgt_node_fwd_args& a, hipStream_t st) {
    if (a.attn) return a.logp ? launch_fwd<T, R, SAME, true, NEXT_CLASSES>(a, st) : (a.q ? launch_fwd<T, R, SAME, true, NEXT_QKV>(a, st) : launch_fwd<T, R, SAME, true, NEXT_NONE>(a, st));
    return launch_fwd<T, R, SAME, false, NEXT_QKV>(a, st);
}
template <typename T, int R, int CN, bool CLASSES, bool NORM> int launch_bwd_pre(const tgt_node_bwd_pre_args& a, hipStream_t st) {
    using L = Bwd<T, R, CN>;
    static std::atomic<uint64_t> done{0};
    return launch(&k_node_bwd_pre<T, R, CN, CLASSES, NORM>, done, bwd_workers(a.rows), L::kThreads, L::kBytes, st, a);
}
template <typename T, int R, int CN> int dispatch_bwd_pre(const tgt_node_bwd_pre_args& a, hipStream_t st) {
    if (a.dlogp) return launch_bwd_pre<T, R, CN, true, true>(a, st);
    return a.v_next ? launch_bwd_pre<T, R, CN, false, true>(a, st) : launch_bwd_pre<T, R, CN, false, false>(a, st);
}
template <typename T, int R, int CN, bool SAME> int launch_bwd_post(const tgt_node_bwd_post_args& a, hipStream_t st) {
    using L = Bwd<T, R, CN, 5, post_block_waves<T, R, CN>()>;
    static std::atomic<uint64_t> done{0};
    return launch(&k_node_bwd_post<T, R, CN, SAME>, done, bwd_workers(a.rows), L::kThreads, L::kBytes, st, a);
}
template <typename T, int R, int CN> int launch_bwd_both(const tgt_node_bwd_pre_args& a, const tgt_node_bwd_post_args& b, hipStream_t st) {
    using L = Bwd<T, R, CN, kBothVecs>;
    static std::atomic<uint64_t> done[2];
    if (a.dlogp) return launch(&k_node_bwd_both<T, R, CN, true>, done[0], bwd_workers(a.rows), L::kThreads, L::kBytes, st, a, b);
    return launch(&k_node_bwd_both<T, R, CN, false>, done[1], bwd_workers(a.rows), L::kThreads, L::kBytes, st, a, b);
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
    return tgt_node_pack_parts(mats, ld, rows, nullptr, n_mats, vecs, lens, n_vecs, dtype, d_frags, d_vecs, stream);
}
int tgt_node_pack_parts(const void* const* mats, const int* ld, const int* rows, const int* cols, int n_mats, const void* const* vecs, const int* lens, int n_vecs,
                        int dtype, void* d_frags, float* d_vecs, void* stream) {
    using namespace tgt;
    const tgt_node_pack_args p{mats, ld, rows, cols, n_mats, vecs, lens, n_vecs, d_frags, d_vecs};
    if (int rc = check_pack(&p, dtype)) return rc;
    KernelTimer t(KS_NODE_PACK, (hipStream_t)stream);
    for (int m = 0, v = 0; m < n_mats || v < n_vecs;) {
        const PackArgs a = pack_args(p, m, v);
        const int grid = pack_blocks(a, kPackThreads);
        if (dtype == TGT_DTYPE_F32) hipLaunchKernelGGL((k_node_pack<float>), dim3(grid), dim3(kPackThreads), 0, (hipStream_t)stream, a);
        else hipLaunchKernelGGL((k_node_pack<nbf16>), dim3(grid), dim3(kPackThreads), 0, (hipStream_t)stream, a);
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
    // Sixteen rows per wave unless thirty-two save rounds: with a round's time next to its number of rows, sixteen rows a wave take float32
    // 26 + 107 us a round of 64 K rows, thirty-two 25 + 149 us a round of 80 K; bf16 46 + 38 us and, of 128 K, 26 + 78 us.  Five launches of a
    // model, us with 16 / 32: float32 4 K nodes 62 / 83, 37605 107 / 124, 64 K 133 / 143, 80 K 207 / 174, 100 K 212 / 275, 150 K 328 / 317, 200 K 440 / 461,
    // 300 K 567 / 621; bf16 4 K 42 / 54, 37605 77 / 89, 64 K 84 / 90, 80 K 118 / 99, 100 K 119 / 114, 150 K 158 / 184, 200 K 194 / 188, 300 K 239 / 262.
    const auto rounds = [&](int per_cu) { return groups_of(a->rows, per_cu * num_cus()); };
    if (a->dtype == TGT_DTYPE_F32)
        return 7 * rounds(32 * fwd_waves<float, 32, false>()) < 5 * rounds(256) ? dispatch_fwd<float, 32, false>(*a, st) : dispatch_fwd<float, 16, false>(*a, st);
    if (a->same_bits) return dispatch_fwd<nbf16, 32, true>(*a, st);
    return 2 * rounds(512) <= rounds(256) ? dispatch_fwd<nbf16, 32, false>(*a, st) : dispatch_fwd<nbf16, 16, false>(*a, st);
}

int tgt_node_bwd_workers(int64_t rows) { return rows < 0 ? -1 : tgt::bwd_workers(rows); }

static int check_pre(const tgt_node_bwd_pre_args* a) {
    using namespace tgt;
    if (!a || a->rows < 1 || !dtype_ok(a->dtype) || !a->s || !a->w_back || (a->dlogp && !a->v_next) || !a->partial) return bad("tgt_node_bwd_pre", "null or bad argument");
    if (a->dlogp ? ((!a->logp && !a->linear) || a->classes < 1 || a->classes > 64 || a->tokens < 0) : (!a->dq || !a->dk || !a->dv || !a->g_in))
        return bad("tgt_node_bwd_pre", "dq, dk, dv, g_in or dlogp, logp and 1 to 64 classes are needed");
    return TGT_OK;
}
static int check_post(const tgt_node_bwd_post_args* a) {
    using namespace tgt;
    if (!a || a->rows < 1 || !dtype_ok(a->dtype) || !a->s || !a->attn || !a->g_out || !a->d_attn || !a->w_post || !a->w_back || !a->v_post || !a->partial)
        return bad("tgt_node_bwd_post", "null or bad argument");
    if (a->nd && (!a->Z || (a->heads != 8 && a->heads != 4 && a->heads != 2))) return bad("tgt_node_bwd_post", "nd needs Z and 8, 4 or 2 heads");
    return TGT_OK;
}

int tgt_node_bwd_pre(const tgt_node_bwd_pre_args* a, void* stream) {
    using namespace tgt;
    if (int rc = check_pre(a)) return rc;
    if (!a->g_out) return bad("tgt_node_bwd_pre", "null or bad argument");
    KernelTimer t(KS_NODE_BWD_PRE, (hipStream_t)stream);
    const hipStream_t st = (hipStream_t)stream;
    if (a->dtype == TGT_DTYPE_F32) return groups_of_64(a->rows, true) ? dispatch_bwd_pre<float, 16, 64>(*a, st) : dispatch_bwd_pre<float, 16, 128>(*a, st);
    if (groups_of_192(a->rows)) return dispatch_bwd_pre<nbf16, 16, 192>(*a, st);
    return groups_of_64(a->rows, false) ? dispatch_bwd_pre<nbf16, 16, 64>(*a, st) : dispatch_bwd_pre<nbf16, 16, 128>(*a, st);
}

int tgt_node_bwd_post(const tgt_node_bwd_post_args* a, void* stream) {
    using namespace tgt;
    if (int rc = check_post(a)) return rc;
    if (!a->g_in) return bad("tgt_node_bwd_post", "null or bad argument");
    KernelTimer t(KS_NODE_BWD_POST, (hipStream_t)stream);
    const hipStream_t st = (hipStream_t)stream;
    if (a->dtype == TGT_DTYPE_F32) return groups_of_64(a->rows, true) ? launch_bwd_post<float, 16, 64, false>(*a, st) : launch_bwd_post<float, 16, 128, false>(*a, st);
    const bool small = groups_of_64(a->rows, false);
    if (a->same_bits && groups_of_192(a->rows)) return launch_bwd_post<nbf16, 32, 192, true>(*a, st);
    if (a->same_bits) return small ? launch_bwd_post<nbf16, 32, 64, true>(*a, st) : launch_bwd_post<nbf16, 32, 128, true>(*a, st);
    return small ? launch_bwd_post<nbf16, 16, 64, false>(*a, st) : launch_bwd_post<nbf16, 16, 128, false>(*a, st);
}

int tgt_node_bwd_both(const tgt_node_bwd_pre_args* a, const tgt_node_bwd_post_args* b, void* stream) {
    using namespace tgt;
    if (int rc = check_pre(a)) return rc;
    if (int rc = check_post(b)) return rc;
    if (a->rows != b->rows || a->dtype != b->dtype || !a->v_next || a->d_token || b->same_bits) return bad("tgt_node_bwd_both", "the same rows, LayerNorm in front, no tokens' gradient, no same_bits");
    KernelTimer t(KS_NODE_BWD_POST, (hipStream_t)stream);
    const hipStream_t st = (hipStream_t)stream;
    // float32: groups of 64 whatever the rows (eight waves have 256 registers each; with twelve 209 of a lane's go to scratch: 64 K rows 122 us, 90 with 64)
    if (a->dtype == TGT_DTYPE_F32) return launch_bwd_both<float, 16, 64>(*a, *b, st);
    return groups_of_64(a->rows, false) ? launch_bwd_both<nbf16, 16, 64>(*a, *b, st) : launch_bwd_both<nbf16, 16, 128>(*a, *b, st);
}

int tgt_node_sums(const tgt_node_sum* sums, int count, int dtype, void* stream) { return tgt_node_sums_and_reduce(sums, count, nullptr, dtype, stream); }
int tgt_node_sums_and_reduce(const tgt_node_sum* sums, int count, const tgt_reduce_desc* desc, int dtype, void* stream) {
    using namespace tgt;
    if (!sums || count < 1 || !dtype_ok(dtype)) return bad("tgt_node_sums", "null or bad argument");
    if (desc && (!desc->partial || desc->workers < 1 || desc->n < 1 || desc->n_out < 1 || desc->n_out > 6 || desc->begin[0] != 0))
        return bad("tgt_node_sums_and_reduce", "not a descriptor that a *_deferred call filled in");
    if (desc && (desc->n % kSumElems != 0 || reinterpret_cast<uintptr_t>(desc->partial) % 16 != 0)) {      // (M K + M elements of a weight: 64 outputs or a multiple)
        if (int rc = reduce_partials(desc, 1, dtype, (hipStream_t)stream)) return rc;
        desc = nullptr;
    }
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
        const bool with_other = desc && c + m == count;
        a.count = m;
        if (with_other) { a.other = *desc; longest = std::max(longest, desc->n); }
        const dim3 grid((unsigned)(longest / kSumElems), (unsigned)(m + with_other));
        if (dtype == TGT_DTYPE_F32) hipLaunchKernelGGL((k_node_sums<float>), grid, dim3(256), 0, (hipStream_t)stream, a);
        else hipLaunchKernelGGL((k_node_sums<nbf16>), grid, dim3(256), 0, (hipStream_t)stream, a);
        TGT_HIP_CHECK(hipGetLastError());
    }
    return TGT_OK;
}

}  // extern "C"
