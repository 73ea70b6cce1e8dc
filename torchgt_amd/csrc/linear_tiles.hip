// Linears of any width (a multiple of 16 bytes per row): y_j = x W_j^T + b_j for up to three weights of one shape, and
// dx = sum_j dy_j W_j.  The node-level models' encoder and classes, and every linear of hidden sizes other than 64.
//
// Bound by the traffic of x and y at 64 K nodes and more, by latency below.  A wave takes 32 node rows; 64 features of
// them at a time become matrix operands in its registers (node_tile.h: float32 as three exact bf16 planes, six products), the
// workgroup's four waves share 64 x 64 pieces of the weight, packed into operand order on their way to LDS, and 64 output columns
// accumulate in registers.  A contraction of up to 128 keeps its operands in registers for all output columns, so x is read
// once; a longer one reads it again for every 64 columns.  The next piece of the weight is asked for before the products of
// this one.  With few rows the output columns are spread over blockIdx.y until there are two workgroups per CU.
//
// float32: six of the nine products of planes (mid lo, lo mid, lo lo are below 2^-24 of the product), the five small ones in a sum of
// their own.  rms error against 64 bits of the result's rms, here / v_mfma_f32_32x32x2_f32 (exact products, one rounding per two of
// them) / all six in one sum, x, W, dy ~ normal:
//   128 -> 64, 64 K rows     y 9.2e-8 / 1.5e-7 / 2.1e-7   dx 7.7e-8 / 1.5e-7 / 1.3e-7   dW 1.5e-7 / 3.1e-7 / 3.5e-7
//   128 -> 64, 300 K rows    y 9.2e-8 / 1.5e-7 / 2.1e-7   dx 7.7e-8 / 1.4e-7 / 1.2e-7   dW 2.0e-7 / 6.1e-7 / 7.7e-7
//   500 -> 64, 20 K rows     y 1.8e-7 / 2.7e-7 / 4.3e-7   dx 7.7e-8 / 1.4e-7 / 1.2e-7   dW 1.5e-7 / 3.3e-7 / 3.1e-7
//   16 -> 40, 64 K rows      y 5.8e-8 / 5.9e-8 / 8.1e-8   dx 7.2e-8 / 1.1e-7 / 1.0e-7   dW 1.7e-7 / 2.4e-7 / 2.9e-7
// and smaller than with the float32 instruction at every other shape of eleven (16 to 500 features, 16 to 128 columns, 1 K to 500 K rows).
// us for 128 -> 64, 64 K rows: y 14.9 / 18.3 / 14.4, dx 15.6 / 19.1 / 18.4, dW with its sum 17.4 / 20.2 / 17.0.
#include "linear_tiles.h"
#include "node_pack.h"
#include <algorithm>

namespace tgt {
namespace {

constexpr int kThreads = 256, kWaves = 4;

// 16 bytes of row r's columns k0 + ... of an array with ld columns (16-byte pieces; K of them count)
template <typename T> __device__ __forceinline__ void fetch_cols(Raw<T>& raw, const T* __restrict__ src, int ld, int k0, const Rows& rows, int lane) {
    constexpr int PP = RowShape<T>::kPieces, PER = RowShape<T>::kPer, VE = 16 / (int)sizeof(T);
    const int last = rows.left > 0 ? rows.left - 1 : 0, r0 = lane / PP, col = k0 + (lane % PP) * VE;
    const T* p = src + rows.first * ld + (col < ld ? col : 0);
#pragma unroll
    for (int i = 0; i < RowShape<T>::kAcc; ++i) {
        const int r = r0 + i * PER;
        raw.v[i] = *reinterpret_cast<const vec16*>(p + (int64_t)(r < last ? r : last) * ld);
    }
    if (k0 + 64 > ld && col >= ld) {      // (the weights are zero there, the row's neighbour may be anything)
#pragma unroll
        for (int i = 0; i < RowShape<T>::kAcc; ++i) raw.v[i] = vec16{0u, 0u, 0u, 0u};
    }
}
template <typename T> __device__ __forceinline__ void put_cols(T* __restrict__ dst, int ld, int c0, const Tile& t, vec16* stage, const Rows& rows, int lane) {
    constexpr int PP = RowShape<T>::kPieces, PER = RowShape<T>::kPer, VE = 16 / (int)sizeof(T);
    wave_sync();
    const int nb = node_base<T>(lane);
#pragma unroll
    for (int i = 0; i < PP / 2; ++i) {
        float f[VE];
#pragma unroll
        for (int e = 0; e < VE; ++e) f[e] = t.get(i * VE + e);
        stage[nb ^ i] = pack16(f, (const T*)nullptr);
    }
    wave_sync();
    const int rb = row_base<T>(lane), r0 = lane / PP, col = c0 + (lane % PP) * VE;
    vec16 v[RowShape<T>::kAcc];
#pragma unroll
    for (int i = 0; i < RowShape<T>::kAcc; ++i) v[i] = stage[row_slot<T>(rb, i)];
    if (col >= ld) return;
    T* p = dst + rows.first * ld + col;
#pragma unroll
    for (int i = 0; i < RowShape<T>::kAcc; ++i)
        if (r0 + i * PER < rows.left) *reinterpret_cast<vec16*>(p + (int64_t)(r0 + i * PER) * ld) = v[i];
}

// A thread's share of a 64 x 64 piece of the weight on its way to LDS: two operand vectors (outputs o0 .., contraction k0 ..)
template <typename T> struct Piece { T v[2][8]; };
template <typename T, bool DX> __device__ __forceinline__ void fetch_piece(Piece<T>& w, const T* __restrict__ W, int ld, int o0, int outs, int k0, int len) {
    const int lane = forgotten(threadIdx.x & 63), r = lane & 31;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int sm = (threadIdx.x >> 6) + 4 * j, s = sm >> 1, m = sm & 1;
        int o = o0 + 32 * ((r >> 2) & 1) + 16 * m + 4 * (r >> 3) + (r & 3), k = k0 + 32 * (lane >> 5) + 8 * s;
        o = o < outs ? o : outs - 1;
        if (DX) {      // eight rows of W at one column
            if (k0 + 64 <= len) {      // (one vector offset, the rows as scalar bases)
                const uint32_t at = k * ld + o;
#pragma unroll
                for (int i = 0; i < 8; ++i) w.v[j][i] = (W + i * ld)[at];
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i) w.v[j][i] = W[(uint32_t)((k + i < len ? k + i : len - 1) * ld + o)];
            }
        } else {       // eight columns of one row, in 16-byte pieces that end with the row
            constexpr int VE = 16 / (int)sizeof(T);
#pragma unroll
            for (int q = 0; q < 8 / VE; ++q) {
                const int c = k + q * VE;
                *reinterpret_cast<vec16*>(&w.v[j][q * VE]) = *reinterpret_cast<const vec16*>(W + (uint32_t)(o * ld + (c < len ? c : len - VE)));
            }
        }
    }
}
template <typename T, int P> __device__ __forceinline__ void put_piece(vec16* dst, const Piece<T>& w, int o0, int outs, int k0, int len) {
    const int lane = forgotten(threadIdx.x & 63), r = lane & 31;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int sm = (threadIdx.x >> 6) + 4 * j, s = sm >> 1, m = sm & 1;
        const int o = o0 + 32 * ((r >> 2) & 1) + 16 * m + 4 * (r >> 3) + (r & 3), k = k0 + 32 * (lane >> 5) + 8 * s;
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = o < outs && k + i < len ? as_float(w.v[j][i]) : 0.f;
        bf16x8_t p[P];
        to_planes(v, p);
#pragma unroll
        for (int q = 0; q < P; ++q) dst[(sm * P + q) * 64 + lane] = __builtin_bit_cast(vec16, p[q]);
    }
}

// For a wave that `holds_nan`: its 32 rows of 64 output columns from c0 on, lane = its node's half as in Tile.  The look costs one
// multiply-add per output (128 -> 64 of 64 K rows: below the runs' difference).
template <bool DX> __device__ __forceinline__ void rows_again(const LinArgs& a, int o, int c0, const Rows& rows, int lane) {
    const int L = DX ? a.M : a.K, C = DX ? a.K : a.M, n = lane & 31;
    if (n >= rows.left) return;
    const int64_t row = rows.first + n;
    for (int i = 0; i < 32; ++i) {
        const int c = c0 + 32 * (lane >> 5) + i;
        if (c >= C) return;
        float t = !DX && a.bias[o] ? reinterpret_cast<const float*>(a.bias[o])[c] : 0.f;
        for (int j = DX ? 0 : o; j < (DX ? a.nw : o + 1); ++j) {
            const float *x = reinterpret_cast<const float*>(a.A[DX ? j : 0]) + row * L, *W = reinterpret_cast<const float*>(a.W[j]);
            for (int k = 0; k < L; ++k) t = fmaf(x[k], DX ? W[k * a.K + c] : W[c * a.K + k], t);
        }
        reinterpret_cast<float*>(a.out[o])[row * C + c] = t;
    }
}

// (float32: 80 KB, two workgroups per CU)
template <typename T> constexpr int lin_lds() { return 2 * kFragVecs<Num<T>::P> * 16 + kWaves * RowShape<T>::kVecs * 16; }

// panel: 128 rows; share: `per` of the 64-column pieces of all outputs
template <typename T, bool DX, bool RESIDENT> __device__ __forceinline__ void tiles_block(const LinArgs& a, const int per, const int panel, const int share, unsigned char* smem) {
    constexpr int P = Num<T>::P, FV = kFragVecs<P>;
    vec16* w = reinterpret_cast<vec16*>(smem);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    vec16* stage = w + 2 * FV + wave * RowShape<T>::kVecs;
    const int L = DX ? a.M : a.K, C = DX ? a.K : a.M, nl = (L + 63) / 64, nk = (DX ? a.nw : 1) * nl, nc = (C + 63) / 64;
    const int first = share * per, all = (DX ? 1 : a.nw) * nc, end = first + per < all ? first + per : all;
    const Rows rows((int64_t)panel * kWaves + wave, a.N);
    Frags<P> f[RESIDENT ? 2 : 1];
    Raw<T> raw;
    const auto ask_rows = [&](int k) { fetch_cols(raw, reinterpret_cast<const T*>(a.A[k / nl]), L, (k % nl) * 64, rows, lane); };
    const auto operands = [&](Frags<P>& to) {
        Tile t;
        settle<T, false>(t, raw, stage, rows, lane);
        make_frags(to, t);
    };
    ask_rows(0);
    Piece<T> next;
    const auto ask = [&](int t, int k) { fetch_piece<T, DX>(next, reinterpret_cast<const T*>(a.W[DX ? k / nl : t / nc]), a.K, (t % nc) * 64, C, (k % nl) * 64, L); };
    if constexpr (RESIDENT) {
        operands(f[0]);
        if (nk == 2) {
            ask_rows(1);
            operands(f[1]);
        }
    }
    ask(first, 0);
    int turn = 0;
    for (int t = first; t < end; ++t) {
        const int o = t / nc, c0 = (t - o * nc) * 64;
        Tile acc;
        zero(acc);
        if (!DX && a.bias[o]) {
            constexpr int VE = 16 / (int)sizeof(T);
#pragma unroll
            for (int i = 0; i < 32 / VE; ++i) {
                const int c = c0 + 32 * (lane >> 5) + VE * i;
                float v[VE];
                unpack16(*reinterpret_cast<const vec16*>(reinterpret_cast<const T*>(a.bias[o]) + (c < C ? c : C - VE)), v, (const T*)nullptr);
#pragma unroll
                for (int e = 0; e < VE; ++e) acc.set(i * VE + e, v[e]);
            }
        }
        for (int k = 0; k < nk; ++k, turn ^= 1) {
            vec16* const mine = w + turn * FV;      // last read in the step before the one before: every wave has passed the barrier since
            put_piece<T, P>(mine, next, c0, C, (k % nl) * 64, L);
            if (k + 1 < nk) ask(t, k + 1);
            else if (t + 1 < end) ask(t + 1, 0);
            if constexpr (!RESIDENT) {
                operands(f[0]);
                if (k + 1 < nk || t + 1 < end) ask_rows(k + 1 < nk ? k + 1 : 0);
            }
            __syncthreads();
            if (RESIDENT && k == 1) gemm_apart<P>(acc, f[RESIDENT ? 1 : 0], mine, lane);
            else gemm_apart<P>(acc, f[0], mine, lane);
        }
        bool again = false;
        if constexpr (P == 3) again = holds_nan([&](int i) { return acc.get(i); }, 32);
        put_cols(reinterpret_cast<T*>(a.out[o]), C, c0, acc, stage, rows, lane);
        if constexpr (P == 3)
            if (again) {
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // (the rows as they were first are on their way)
                rows_again<DX>(a, o, c0, rows, lane);
            }
    }
}

template <typename T, bool DX, bool RESIDENT> __global__ __launch_bounds__(kThreads, 2) void k_linear_tiles(const LinArgs a, const int per) {
    extern __shared__ __align__(16) unsigned char smem[];
    tiles_block<T, DX, RESIDENT>(a, per, blockIdx.x, blockIdx.y, smem);
}
// One output of 64 columns, and the packing of a model's parameters, which that output does not depend on: as a launch of its own the packing is
// 5 to 6 us of a few dozen workgroups with nothing beside them.  128 -> 64 and the parameters of four layers, us, two launches / one: float32 4 K rows
// 6.0 + 8.9 / 9.6, 37605 5.1 + 14.2 / 13.0, 64 K 5.8 + 16.8 / 19.5, bf16 64 K (GT) 5.6 + 8.3 / 11.4.
template <typename T> __global__ __launch_bounds__(kThreads, 2) void k_linear_tiles_and_pack(const LinArgs a, const PackArgs p, const int packers) {
    extern __shared__ __align__(16) unsigned char smem[];
    if ((int)blockIdx.x < packers) pack_block<T, kThreads>(p, blockIdx.x);
    else tiles_block<T, false, true>(a, 1, blockIdx.x - packers, 0, smem);
}

template <typename T, bool DX, bool RESIDENT> int launch(const LinArgs& a, hipStream_t st) {
    static std::atomic<uint64_t> done{0};
    constexpr int lds = lin_lds<T>();
    if (int rc = allow_lds(reinterpret_cast<const void*>(&k_linear_tiles<T, DX, RESIDENT>), lds, done)) return rc;
    // two workgroups per CU: below that the columns are shared out
    const int64_t panels = (a.N + 32 * kWaves - 1) / (32 * kWaves);
    const int all = (DX ? 1 : a.nw) * (((DX ? a.K : a.M) + 63) / 64), splits = (int)std::min<int64_t>(all, std::max<int64_t>(1, 512 / panels)), per = (all + splits - 1) / splits;
    hipLaunchKernelGGL((k_linear_tiles<T, DX, RESIDENT>), dim3((unsigned)panels, (unsigned)((all + per - 1) / per)), dim3(kThreads), lds, st, a, per);
    TGT_HIP_CHECK(hipGetLastError());
    return TGT_OK;
}
template <typename T, bool DX> int run(const LinArgs& a, hipStream_t st) {
    return (DX ? a.nw * ((a.M + 63) / 64) : (a.K + 63) / 64) <= 2 ? launch<T, DX, true>(a, st) : launch<T, DX, false>(a, st);
}

// ---- weight gradients -------------------------------------------------------------------------------------------------
// A workgroup keeps one 64-row piece of one dW_j against XT 64-column pieces of x in registers, one 32 x 32 block per wave, over
// its share of 64-node panels.  The panel's rows arrive coalesced, are cut into bf16 planes on their way to LDS and are read back
// transposed by the products (node_tile.h); the next panel is asked for before the products of this one.  Bound by the traffic
// of x and dy: with two pieces of x at a time dy is read once per 128 columns of x.  XT = 1 where x has 64 columns or less.
constexpr int kPanelBytes = 64 * 128;      // one plane of one operand

template <typename T, int XT> __global__ __launch_bounds__(XT * 256) void k_gradw_tiles(const GradWArgs a) {
    constexpr int P = Num<T>::P, NWV = 4 * XT, RPW = 64 / NWV, PP = RowShape<T>::kPieces, PER = RowShape<T>::kPer, ACC = RPW / PER, VE = 16 / (int)sizeof(T), NT = 1 + XT;
    extern __shared__ __align__(16) unsigned char smem[];      // [NT][P][kPanelBytes]: dy, then x
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int groups = ((a.K + 63) / 64 + XT - 1) / XT, mts = (a.M + 63) / 64;
    const int m = blockIdx.y / groups, g = blockIdx.y - m * groups, j = m / mts, m0 = (m - j * mts) * 64, k0 = g * XT * 64;
    const T* src[NT];
    int ld[NT], col[NT];
    src[0] = reinterpret_cast<const T*>(a.dy[j]); ld[0] = a.M; col[0] = m0;
#pragma unroll
    for (int t = 1; t < NT; ++t) { src[t] = reinterpret_cast<const T*>(a.x); ld[t] = a.K; col[t] = k0 + 64 * (t - 1); }
    const int q = lane % PP, r0 = wave * RPW + lane / PP;      // this lane's 16-byte piece and first row of a panel
    const int64_t panels = (a.N + 63) / 64;
    vec16 raw[NT][ACC];
    const auto fetch = [&](int64_t p) {
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const int c = col[t] + q * VE;
#pragma unroll
            for (int i = 0; i < ACC; ++i) {
                const int64_t r = p * 64 + r0 + i * PER;
                raw[t][i] = *reinterpret_cast<const vec16*>(src[t] + (r < a.N ? r : a.N - 1) * ld[t] + (c < ld[t] ? c : ld[t] - VE));
            }
        }
    };
    float sums[VE];
#pragma unroll
    for (int e = 0; e < VE; ++e) sums[e] = 0.f;
    float16_t acc, small;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = small[i] = 0.f;
    const int block = wave & 3, base_dy = operand_base(block >> 1, lane), base_x = operand_base(block & 1, lane);
    const unsigned char* const x_planes = smem + (1 + wave / 4) * P * kPanelBytes;
    int64_t p = blockIdx.x;
    if (p < panels) fetch(p);
    for (; p < panels; p += gridDim.x) {
        __syncthreads();      // the panel before has been used
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const bool in = col[t] + q * VE < ld[t];
#pragma unroll
            for (int i = 0; i < ACC; ++i) {
                const int r = r0 + i * PER;
                if (!in || p * 64 + r >= a.N) raw[t][i] = vec16{0u, 0u, 0u, 0u};
                float v[VE];
                unpack16(raw[t][i], v, (const T*)nullptr);
                if (t == 0) {
#pragma unroll
                    for (int e = 0; e < VE; ++e) sums[e] += v[e];
                }
                unsigned char* const at = smem + t * P * kPanelBytes + r * 128 + (((q * VE / 8) ^ (r & 7)) << 4);
                if constexpr (P == 1) *reinterpret_cast<vec16*>(at) = raw[t][i];
                else {
                    uint32_t w[3][4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) cut3(v[e], w[0][e], w[1][e], w[2][e]);
#pragma unroll
                    for (int s = 0; s < P; ++s)
                        *reinterpret_cast<uint2*>(at + s * kPanelBytes + 8 * (q & 1)) =
                            make_uint2(__builtin_amdgcn_perm(w[s][1], w[s][0], 0x07060302u), __builtin_amdgcn_perm(w[s][3], w[s][2], 0x07060302u));
                }
            }
        }
        __syncthreads();
        if (p + gridDim.x < panels) fetch(p + gridDim.x);
        node_product<P, kPanelBytes, true>(acc, smem, x_planes, base_dy, base_x, &small);
    }
    if constexpr (P == 3) acc += small;
    const int64_t per = (int64_t)a.M * a.K + a.M;
    float* const mine = a.partial + ((int64_t)blockIdx.x * a.nw + j) * per;
    const int k = k0 + 64 * (wave / 4) + 32 * (block & 1) + (lane & 31);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int o = m0 + 32 * (block >> 1) + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
        if (o < a.M && k < a.K) mine[(int64_t)o * a.K + k] = acc[i];
    }
    if constexpr (P == 3)
        if (holds_nan([&](int i) { return acc[i]; }, 16) && k < a.K) {      // as in rows_again: this worker's share of the nodes
            const float *x = reinterpret_cast<const float*>(a.x) + k, *dy = reinterpret_cast<const float*>(a.dy[j]);
            for (int i = 0; i < 16; ++i) {
                const int o = m0 + 32 * (block >> 1) + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
                if (o >= a.M) break;
                float t = 0.f;
                for (int64_t q0 = blockIdx.x; q0 < panels; q0 += gridDim.x)
                    for (int64_t r = q0 * 64; r < a.N && r < q0 * 64 + 64; ++r) t = fmaf(dy[r * a.M + o], x[r * a.K], t);
                mine[(int64_t)o * a.K + k] = t;
            }
        }
    if (g == 0) {      // column sums of dy: over the lanes of a piece, then over the waves
        float* const part = reinterpret_cast<float*>(smem);
        __syncthreads();
#pragma unroll
        for (int e = 0; e < VE; ++e) {
#pragma unroll
            for (int off = PP; off < 64; off <<= 1) sums[e] += __shfl_xor(sums[e], off);
            if (lane < PP) part[wave * 64 + q * VE + e] = sums[e];
        }
        __syncthreads();
        if (threadIdx.x < 64 && m0 + (int)threadIdx.x < a.M) {
            float s = 0.f;
#pragma unroll
            for (int w = 0; w < NWV; ++w) s += part[w * 64 + threadIdx.x];
            mine[(int64_t)a.M * a.K + m0 + threadIdx.x] = s;
        }
    }
}

template <typename T, int XT> int launch_gradw(const GradWArgs& a, int workers, hipStream_t st) {
    static std::atomic<uint64_t> done{0};
    constexpr int lds = (1 + XT) * Num<T>::P * kPanelBytes;
    if (int rc = allow_lds(reinterpret_cast<const void*>(&k_gradw_tiles<T, XT>), lds, done)) return rc;
    const int groups = ((a.K + 63) / 64 + XT - 1) / XT;
    hipLaunchKernelGGL((k_gradw_tiles<T, XT>), dim3((unsigned)workers, (unsigned)(a.nw * ((a.M + 63) / 64) * groups)), dim3(XT * 256), lds, st, a);
    TGT_HIP_CHECK(hipGetLastError());
    return TGT_OK;
}

}  // namespace

int gradw_tiles(const GradWArgs& a, int workers, int dtype, hipStream_t st) {
    // (one piece of x at a time where there is only one)
    if (dtype == TGT_DTYPE_F32) return a.K <= 64 ? launch_gradw<float, 1>(a, workers, st) : launch_gradw<float, 2>(a, workers, st);
    return a.K <= 64 ? launch_gradw<nbf16, 1>(a, workers, st) : launch_gradw<nbf16, 2>(a, workers, st);
}

template <typename T> static int launch_with_pack(const LinArgs& a, const tgt_node_pack_args& p, hipStream_t st) {
    static std::atomic<uint64_t> done{0};
    constexpr int lds = lin_lds<T>();
    if (int rc = allow_lds(reinterpret_cast<const void*>(&k_linear_tiles_and_pack<T>), lds, done)) return rc;
    const PackArgs args = pack_args(p, 0, 0);
    const int packers = pack_blocks(args, kThreads);
    hipLaunchKernelGGL((k_linear_tiles_and_pack<T>), dim3((unsigned)((a.N + 32 * kWaves - 1) / (32 * kWaves) + packers)), dim3(kThreads), lds, st, a, args, packers);
    TGT_HIP_CHECK(hipGetLastError());
    return TGT_OK;
}
// (one column piece of a weight that stays in registers, what one launch can be told; 64 -> 64 has kernels of its own in linear.hip)
int packs_beside(const LinArgs& a, const tgt_node_pack_args* pack, int dtype, bool& fits) {
    if (int rc = check_pack(pack, dtype)) return rc;
    fits = a.N > 0 && a.M == 64 && a.K != 64 && a.K <= 128 && pack->n_mats <= kPackMats && pack->n_vecs <= kPackVecs;
    return TGT_OK;
}
int linear_tiles_and_pack(const LinArgs& a, const tgt_node_pack_args& pack, int dtype, hipStream_t st) {
    return dtype == TGT_DTYPE_F32 ? launch_with_pack<float>(a, pack, st) : launch_with_pack<nbf16>(a, pack, st);
}

int linear_tiles(const LinArgs& a, bool dx, int dtype, hipStream_t st) {
    if (dtype == TGT_DTYPE_F32) return dx ? run<float, true>(a, st) : run<float, false>(a, st);
    return dx ? run<nbf16, true>(a, st) : run<nbf16, false>(a, st);
}

}  // namespace tgt
