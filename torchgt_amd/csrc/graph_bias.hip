// The graph-level attention bias and the shortest-path preprocessing behind it.
//
//   tgt_graph_attn_bias_fwd / _bwd   GraphAttnBias.forward, simple edge-type branch
//                                    (models/graphormer_graph_level.py:94-156) and the
//                                    gradients of its three embedding tables
//   tgt_floyd_warshall               floyd_warshall of data/algos.pyx:9-54 (distance and
//                                    intermediate-node matrices) for a batch of small graphs
//
// The reference builds the [b, H, S+1, S+1] bias with six ATen passes over tensors of
// that size (clone, repeat, two embedding lookups + permutes, slice adds); here one
// kernel reads the ids once and writes the bias once.  The backward folds the bias
// gradient into the (tiny) tables: every workgroup accumulates in LDS and the
// workgroup partials are added in a fixed order.
#include "common.h"
#include <algorithm>
#include <type_traits>

namespace tgt {
namespace {

struct gbf16 { uint16_t x; };
__device__ __forceinline__ float ldf(const float* p) { return *p; }
__device__ __forceinline__ float ldf(const gbf16* p) { return __uint_as_float(((uint32_t)p->x) << 16); }
__device__ __forceinline__ void stf(float* p, float v) { *p = v; }
__device__ __forceinline__ void stf(gbf16* p, float v) {
    const __bf16 b = static_cast<__bf16>(v);
    p->x = __builtin_bit_cast(uint16_t, b);
}

constexpr int kMaxHeads = 32;

struct BiasArgs {
    const void* attn_bias;        // [b, S1, S1]
    const int64_t* spatial_pos;   // [b, s, s]
    const int64_t* edge_type;     // [b, s, s, F]
    const void* spatial_table;    // [num_spatial, H]
    const void* edge_table;       // [num_edges, H]
    const void* virtual_dist;     // [H]
    int b, s, H, F, num_spatial, num_edges;
};

__device__ __forceinline__ int clamp_id(int64_t v, int n) { return v < 0 ? 0 : (v >= n ? n - 1 : (int)v); }

// one thread per (graph, row i, column j) of the [S1, S1] bias, all heads
template <typename T>
__global__ __launch_bounds__(256) void k_graph_bias_fwd(BiasArgs a, T* __restrict__ out) {
    const int S1 = a.s + 1;
    const int64_t total = (int64_t)a.b * S1 * S1;
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= total) return;
    const int j = (int)(t % S1), i = (int)((t / S1) % S1);
    const int64_t g = t / ((int64_t)S1 * S1);
    const float base = 2.f * ldf(reinterpret_cast<const T*>(a.attn_bias) + t);    // the clone plus the final re-add (:104, :153)
    const T* sp_tab = reinterpret_cast<const T*>(a.spatial_table);
    const T* e_tab = reinterpret_cast<const T*>(a.edge_table);
    const T* vd = reinterpret_cast<const T*>(a.virtual_dist);
    const bool inner = i >= 1 && j >= 1;
    const bool virt = i == 0 || j == 0;          // (i >= 1, j == 0) and the whole row 0 (:116-117)
    int sp = 0;
    const int64_t* et = nullptr;
    if (inner) {
        const int64_t pos = (g * a.s + (i - 1)) * a.s + (j - 1);
        sp = clamp_id(a.spatial_pos[pos], a.num_spatial);
        et = a.edge_type + pos * a.F;
    }
    const float inv_f = 1.f / (float)a.F;
    for (int h = 0; h < a.H; ++h) {
        float v = base;
        if (inner) {
            v += ldf(sp_tab + sp * a.H + h);
            float e = 0.f;
            for (int f = 0; f < a.F; ++f) e += ldf(e_tab + clamp_id(et[f], a.num_edges) * a.H + h);
            v += e * inv_f;                      // mean over the edge features (:150)
        }
        if (virt) v += ldf(vd + h);
        stf(out + ((g * a.H + h) * S1 + i) * S1 + j, v);
    }
}

// Position (graph, row, column) of a thread in the [b, S1, S1] index space and its step from one
// iteration of a grid-stride loop to the next, without a 64-bit division per iteration.
struct BiasPos {
    int64_t g;
    int i, j;
};
struct BiasStep {
    int64_t dg;
    int di, dj;
};
__device__ __forceinline__ BiasPos bias_pos(int64_t t, int S1) {
    const int64_t plane = (int64_t)S1 * S1;
    BiasPos p;
    p.g = t / plane;
    const int ij = (int)(t - p.g * plane);
    p.i = ij / S1;
    p.j = ij - p.i * S1;
    return p;
}
__device__ __forceinline__ BiasStep bias_step(int64_t stride, int S1) {
    const BiasPos p = bias_pos(stride, S1);
    return BiasStep{p.g, p.i, p.j};
}
__device__ __forceinline__ void bias_advance(BiasPos& p, const BiasStep& d, int S1) {
    p.j += d.dj;
    if (p.j >= S1) { p.j -= S1; ++p.i; }
    p.i += d.di;
    if (p.i >= S1) { p.i -= S1; ++p.g; }
    p.g += d.dg;
}

// The same for eight heads and tables that fit LDS: the tables are converted to float once per
// workgroup, a position reads its table rows with 16-byte LDS loads instead of one global load per
// head and feature, and the global loads of a position (bias, ids) are issued together.  Same
// arithmetic in the same order as the kernel above.
template <typename T>
__global__ __launch_bounds__(256) void k_graph_bias_fwd8(BiasArgs a, T* __restrict__ out) {
    constexpr int H = 8;
    extern __shared__ float4 tab4[];
    float* tab = reinterpret_cast<float*>(tab4);
    const int n_sp = a.num_spatial * H, n_e = a.num_edges * H;
    {
        const T* sp_tab = reinterpret_cast<const T*>(a.spatial_table);
        const T* e_tab = reinterpret_cast<const T*>(a.edge_table);
        const T* vd = reinterpret_cast<const T*>(a.virtual_dist);
        for (int k = threadIdx.x; k < n_sp + n_e + H; k += 256)
            tab[k] = k < n_sp ? ldf(sp_tab + k) : (k < n_sp + n_e ? ldf(e_tab + (k - n_sp)) : ldf(vd + (k - n_sp - n_e)));
    }
    __syncthreads();
    const float4* t_sp = tab4;
    const float4* t_e = tab4 + n_sp / 4;
    const float4* t_v = t_e + n_e / 4;
    const int S1 = a.s + 1, F = a.F;
    const int64_t plane = (int64_t)S1 * S1;
    const int64_t total = (int64_t)a.b * plane;
    const float inv_f = 1.f / (float)F;
    const T* __restrict__ bias = reinterpret_cast<const T*>(a.attn_bias);
    const int64_t stride = (int64_t)gridDim.x * 256;
    const BiasStep step = bias_step(stride, S1);
    BiasPos p = bias_pos((int64_t)blockIdx.x * 256 + threadIdx.x, S1);
    for (int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x; t < total; t += stride, bias_advance(p, step, S1)) {
        const int64_t g = p.g;
        const int i = p.i, j = p.j, ij = i * S1 + j;
        const bool inner = i >= 1 && j >= 1;
        const int64_t pos = inner ? (g * a.s + (i - 1)) * a.s + (j - 1) : 0;
        const T braw = bias[t];
        float v[H];
        if (a.s > 0) {
            const int64_t spr = a.spatial_pos[pos];
            float e[H];
#pragma unroll
            for (int h = 0; h < H; ++h) e[h] = 0.f;
            for (int f0 = 0; f0 < F; f0 += 4) {
                int64_t er[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) er[u] = a.edge_type[pos * F + min(f0 + u, F - 1)];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    if (f0 + u < F) {
                        const int id = clamp_id(er[u], a.num_edges);
                        const float4 lo = t_e[id * 2], hi = t_e[id * 2 + 1];
                        e[0] += lo.x; e[1] += lo.y; e[2] += lo.z; e[3] += lo.w;
                        e[4] += hi.x; e[5] += hi.y; e[6] += hi.z; e[7] += hi.w;
                    }
                }
            }
            const int sp = clamp_id(spr, a.num_spatial);
            const float4 lo = t_sp[sp * 2], hi = t_sp[sp * 2 + 1];
            const float s8[H] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
            const float base = 2.f * ldf(&braw);
#pragma unroll
            for (int h = 0; h < H; ++h) {
                float x = base;
                if (inner) { x += s8[h]; x += e[h] * inv_f; }
                v[h] = x;
            }
        } else {
            const float base = 2.f * ldf(&braw);
#pragma unroll
            for (int h = 0; h < H; ++h) v[h] = base;
        }
        if (!inner) {
            const float4 lo = t_v[0], hi = t_v[1];
            v[0] += lo.x; v[1] += lo.y; v[2] += lo.z; v[3] += lo.w;
            v[4] += hi.x; v[5] += hi.y; v[6] += hi.z; v[7] += hi.w;
        }
        T* __restrict__ o = out + g * H * plane + ij;
#pragma unroll
        for (int h = 0; h < H; ++h) stf(o + h * plane, v[h]);
    }
}

// Table gradients.  Each workgroup keeps the three tables in LDS ([num_spatial + num_edges + 1][H]
// floats), walks its share of the positions and writes one partial.  Row 0 of the two
// embedding tables is the padding index: it receives no gradient (nn.Embedding padding_idx=0).
// All loads of a position (ids, then the gradient of eight heads at a time) are issued without a
// lane-dependent branch around them: out-of-range lanes read a clamped address and add nothing.
// Shortest-path ids are few and small (most pairs of a graph are two to four hops apart), and an LDS
// float atomic costs a few cycles per active lane whatever the address: with up to eight heads the
// ids 1..NHOT are summed in registers (one compare per id, one select + add per id and head), added
// over the wave at the end and put into LDS by one lane; only the rare other ids, the edge types
// (most pairs are not edges: id 0) and the virtual-node row and column use atomics per position.
constexpr int kBiasFeat = 4;      // edge features handled per pass over the heads (1 when there is only one)
constexpr int kBiasHot = 5;       // spatial ids 1..5 (self, one to four hops) are summed in registers

// What one lane reads for one position and one pass (up to kBiasFeat edge features, eight heads), kept
// as loaded: converting or clamping a value where it is fetched would make the wave wait for it there.
// NS gradients of one and the same bias (the layers of a model share it) are read side by side and added in float.
template <typename T> struct BiasGrads { const T* p[4]; };
template <int FC> struct BiasIds {
    int64_t spr, er[FC];
    int64_t g;
    int ij;
    bool valid, inner;
};
template <int FC>
__device__ __forceinline__ void bias_ids(const BiasArgs& a, const BiasPos& p, bool valid, int f0, BiasIds<FC>& x) {
    x.valid = valid;
    x.g = valid ? p.g : 0;                           // past the end: element 0, nothing is added
    const int i = valid ? p.i : 0, j = valid ? p.j : 0;
    x.ij = i * (a.s + 1) + j;
    x.inner = valid && i >= 1 && j >= 1;
    const int64_t pos = x.inner ? (x.g * a.s + (i - 1)) * a.s + (j - 1) : 0;
    x.spr = 0;
#pragma unroll
    for (int u = 0; u < FC; ++u) x.er[u] = 0;
    if (a.s > 0) {
        x.spr = a.spatial_pos[pos];
#pragma unroll
        for (int u = 0; u < FC; ++u) x.er[u] = a.edge_type[pos * a.F + min(f0 + u, a.F - 1)];
    }
}

// sp, e: what the position's gradient goes to (0: nowhere)
template <typename T, int FC, int NS>
struct BiasFetch {
    int sp, e[FC];
    bool virt;
    T raw[NS][8];
};
template <typename T, int FC, int NS>
__device__ __forceinline__ void bias_targets(const BiasArgs& a, const BiasIds<FC>& id, int f0, BiasFetch<T, FC, NS>& x) {
    x.sp = id.inner && f0 == 0 ? clamp_id(id.spr, a.num_spatial) : 0;
#pragma unroll
    for (int u = 0; u < FC; ++u) x.e[u] = id.inner && f0 + u < a.F ? clamp_id(id.er[u], a.num_edges) : 0;
    x.virt = id.valid && !id.inner && f0 == 0;
}
template <typename T, int FC, int NS>
__device__ __forceinline__ void bias_grads(const BiasArgs& a, const BiasGrads<T>& dout, int64_t at, int h0, BiasFetch<T, FC, NS>& x) {
    const int64_t plane = (int64_t)(a.s + 1) * (a.s + 1);
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        const T* __restrict__ dg = dout.p[k] + at;          // head h of this position: dg[h * plane]
#pragma unroll
        for (int u = 0; u < 8; ++u) x.raw[k][u] = dg[(int64_t)min(h0 + u, a.H - 1) * plane];
    }
}

template <typename T, int NHOT, int FC, int NS>
__device__ __forceinline__ void bias_consume(const BiasArgs& a, const BiasFetch<T, FC, NS>& x, int h0, float* acc_sp, float* acc_e,
                                             float* acc_v, float (&hot)[NHOT > 0 ? NHOT : 1][8]) {
    const int H = a.H;
    const bool cold = x.sp > NHOT;
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        v[u] = ldf(&x.raw[0][u]);
#pragma unroll
        for (int k = 1; k < NS; ++k) v[u] += ldf(&x.raw[k][u]);
    }
    if (NHOT > 0) {
#pragma unroll
        for (int r = 0; r < NHOT; ++r) {
            const bool hit = x.sp == r + 1;
#pragma unroll
            for (int u = 0; u < 8; ++u) hot[r][u] += hit ? v[u] : 0.f;
        }
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        const int h = h0 + u;
        if (h < H && v[u] != 0.f) {              // masked positions carry exact zeros
            if (cold) atomicAdd(&acc_sp[x.sp * H + h], v[u]);
#pragma unroll
            for (int w = 0; w < FC; ++w)
                if (x.e[w] > 0) atomicAdd(&acc_e[x.e[w] * H + h], v[u]);
            if (x.virt) atomicAdd(&acc_v[h], v[u]);
        }
    }
}

// ONEPASS: H <= 8 and F <= FC, one fetch per position; the gradients of the next position and the ids of the one behind it are
// asked for before the current one is consumed.  A batch of graphs is padded to its largest, and padding has id 0 everywhere, whose
// rows receive no gradient: a lane of such a position reads the address of the wave's last lane that adds something, and a wave of nothing
// else one element and goes on.  The same 256 graphs in float32 with 3 gradients 102 us read in full, 74 so, 1 gradient 55 and 48; padding is 44 % of their rows.
template <typename T, int NHOT, bool ONEPASS, int FC, int NS>
__global__ __launch_bounds__(256) void k_graph_bias_bwd(BiasArgs a, BiasGrads<T> dout, float* __restrict__ partial,
                                                        int copies) {
    extern __shared__ float acc_all[];
    const int n_acc = (a.num_spatial + a.num_edges + 1) * a.H;
    for (int k = threadIdx.x; k < n_acc * copies; k += 256) acc_all[k] = 0.f;
    __syncthreads();
    // neighbouring lanes add into different copies of the tables
    float* acc = acc_all + (threadIdx.x % copies) * n_acc;
    float* acc_sp = acc;
    float* acc_e = acc + a.num_spatial * a.H;
    float* acc_v = acc_e + a.num_edges * a.H;
    const int H = a.H, F = a.F;
    const int64_t total = (int64_t)a.b * (a.s + 1) * (a.s + 1);
    const int64_t stride = (int64_t)gridDim.x * 256;
    float hot[NHOT > 0 ? NHOT : 1][8];
#pragma unroll
    for (int r = 0; r < (NHOT > 0 ? NHOT : 1); ++r)
#pragma unroll
        for (int u = 0; u < 8; ++u) hot[r][u] = 0.f;
    if (total == 0) {
    } else if (ONEPASS) {
        BiasFetch<T, FC, NS> cur, nxt;
        BiasIds<FC> ids;
        const BiasStep step = bias_step(stride, a.s + 1);
        int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
        BiasPos p = bias_pos(t, a.s + 1);
        const int64_t heads = (int64_t)H * (a.s + 1) * (a.s + 1);
        const auto ask_ids = [&](int64_t at) { bias_ids(a, p, at < total, 0, ids); bias_advance(p, step, a.s + 1); };
        int64_t at = 0;      // of the position whose targets are known
        const auto targets = [&](BiasFetch<T, FC, NS>& x) -> uint64_t {
            bias_targets(a, ids, 0, x);
            bool adds = x.virt || x.sp > 0;
#pragma unroll
            for (int u = 0; u < FC; ++u) adds |= x.e[u] > 0;
            const uint64_t any = __ballot(adds);
            const int64_t own = ids.g * heads + ids.ij;
            const int last = any ? 63 - __builtin_clzll(any) : 0;
            const uint64_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)own, last), hi = (uint32_t)__builtin_amdgcn_readlane((int)(own >> 32), last);
            at = adds ? own : (any ? (int64_t)(hi << 32 | lo) : 0);
            return any;
        };
        // (the ids first: loads are waited for in their order)
        ask_ids(t);
        uint64_t cur_any = targets(cur);
        ask_ids(t + stride);
        bias_grads(a, dout, at, 0, cur);
        for (; t - threadIdx.x < total; t += stride) {
            const uint64_t nxt_any = targets(nxt);
            ask_ids(t + 2 * stride);
            bias_grads(a, dout, at, 0, nxt);
            if (cur_any) bias_consume<T, NHOT, FC, NS>(a, cur, 0, acc_sp, acc_e, acc_v, hot);
            cur = nxt;
            cur_any = nxt_any;
        }
    } else {
        for (int64_t t0 = (int64_t)blockIdx.x * 256; t0 < total; t0 += stride)
            for (int f0 = 0; f0 < F; f0 += FC)
                for (int h0 = 0; h0 < H; h0 += 8) {
                    BiasIds<FC> ids;
                    BiasFetch<T, FC, NS> x;
                    bias_ids(a, bias_pos(t0 + threadIdx.x, a.s + 1), t0 + threadIdx.x < total, f0, ids);
                    bias_grads(a, dout, ids.g * H * (a.s + 1) * (a.s + 1) + ids.ij, h0, x);
                    // the spatial id counts once per head pass, in the first feature pass
                    bias_targets(a, ids, f0, x);
                    bias_consume<T, NHOT, FC, NS>(a, x, h0, acc_sp, acc_e, acc_v, hot);
                }
    }
    if (NHOT > 0) {
        // the wave's sums of the ids kept in registers (NHOT > 0 only with H <= 8: one pass over the heads)
#pragma unroll
        for (int r = 0; r < NHOT; ++r)
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                float x = hot[r][u];
#pragma unroll
                for (int off = 32; off >= 1; off >>= 1) x += __shfl_xor(x, off);
                if (threadIdx.x % 64 == 0 && u < H && r + 1 < a.num_spatial) atomicAdd(&acc_sp[(r + 1) * H + u], x);
            }
    }
    __syncthreads();
    const float inv_f = 1.f / (float)F;                       // mean over the edge features (:150)
    const int e_lo = a.num_spatial * H, e_hi = e_lo + a.num_edges * H;
    for (int k = threadIdx.x; k < n_acc; k += 256) {
        float t = 0.f;
        for (int c = 0; c < copies; ++c) t += acc_all[c * n_acc + k];       // copies in order
        partial[(int64_t)blockIdx.x * n_acc + k] = k >= e_lo && k < e_hi ? t * inv_f : t;
    }
}

// The same for bfloat16 gradients, one edge feature and eight heads, on the matrix cores: a table row's gradient is the product of the
// positions that look it up, as zeros and ones, with their gradients.  A wave takes 120 consecutive positions of a graph's [S1, S1] plane; 8 spatial
// ids, 7 edge ids and the virtual node are 16 rows of zeros and ones, built from the ids in registers, 16 more spatial ids another 16 where
// they occur; the columns are 16 (gradient, head).  One times a bfloat16 is exact, the sums are float, in four sets.  Other ids go to LDS atomics
// as above, and so does a wave's whole share when one of its sums is no number: zero times infinity is none either.  A column arrives as 64 whole
// dwords, one a lane, from the one that holds its first element (every other plane of an odd S1 begins inside a dword), and goes through LDS to
// the lanes of the products (loaded in the products' order, a line per lane, the address unit alone took 75 us).
// Bound by memory: a row of padding still has its virtual node's element.  256 graphs of up to 128 nodes (44 % of the rows padding), 40 spatial
// and 64 edge ids, with the reduction, us, the kernel above before / this one: 1 gradient 48 / 34, 2 59 / 42, 3 70 / 51, 4 93 / 60 (at five terabytes
// a second); behind the layers that write the three gradients 86 / 69.  rms error of the spatial table against 64 bits, four draws of each: 2.7e-8 / 2.7e-8.
constexpr int kRowsSp = 24, kRowsE = 7;      // ids 1 .. with a matrix row
constexpr uint32_t kVirtCode = 0xffffu;      // (ids are below 32768: the tables fit LDS)
constexpr int kChunk = 120;                               // (the 128 of a product would need a 65th dword of an odd column)
constexpr int kBiasMinSide = 11, kBiasMaxSide = 1625;     // a plane of one chunk; S1^3 < 2^32: the division by S1 as a multiplication
constexpr size_t kBiasMaxLds = 80 * 1024;                 // two workgroups per CU
constexpr int kColumn = 68;                               // dwords of a column in LDS: 16 columns in different banks
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
template <int NS> constexpr int bias_mm_lds() { return 4 * (NS * 8 * kColumn * 4 + 2 * 128 * 2); }      // four waves: columns, codes

// Orders a wave's LDS writes before its own later reads (and the other way round): the hardware runs them in order, this keeps the compiler to it.
__device__ __forceinline__ void wave_sync_lds() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int NS>
__global__ __launch_bounds__(256, 4) void k_graph_bias_bwd_mm(BiasArgs a, BiasGrads<gbf16> dout, float* __restrict__ partial, int, int chunks, uint32_t inv_s1) {
    constexpr int G = (NS + 1) / 2;
    extern __shared__ __align__(16) float mm_lds[];      // the waves' columns and codes, then the tables
    float* const acc_all = mm_lds + bias_mm_lds<NS>() / 4;
    constexpr int H = 8;
    const int S1 = a.s + 1, plane = S1 * S1, n_acc = (a.num_spatial + a.num_edges + 1) * H;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), c16 = lane & 15, oct = lane >> 4;
    uint32_t* const columns = reinterpret_cast<uint32_t*>(mm_lds) + wave * (bias_mm_lds<NS>() / 16);
    uint16_t* const codes = reinterpret_cast<uint16_t*>(columns + NS * 8 * kColumn);      // [2][128]
    for (int k = threadIdx.x; k < bias_mm_lds<NS>() / 4 + n_acc; k += 256) mm_lds[k] = 0.f;
    __syncthreads();
    float *const acc_sp = acc_all, *const acc_e = acc_sp + a.num_spatial * H, *const acc_v = acc_e + a.num_edges * H;
    // position k * 64 + lane of a chunk: the last chunk of a plane ends with it, what it shares with the one before adds nothing
    struct At { int p, i, j; bool in, inner; };
    const auto first_of = [&](int r) { return min(r * kChunk, plane - kChunk); };
    const auto position = [&](int r, int k, bool there) {
        At x;
        const int q = 64 * k + lane;
        x.p = first_of(r) + q;
        x.i = (int)__umulhi((uint32_t)x.p, inv_s1);
        x.j = x.p - x.i * S1;
        x.in = there && q < kChunk && x.p >= r * kChunk;
        x.inner = x.in && x.i >= 1 && x.j >= 1;
        return x;
    };
    struct Chunk { int64_t g; int r; };
    const int total_waves = gridDim.x * 4, dg = total_waves / chunks, dr = total_waves - dg * chunks;
    const auto advance = [&](Chunk& c) {
        c.r += dr; c.g += dg;
        if (c.r >= chunks) { c.r -= chunks; ++c.g; }
    };
    const int w0 = blockIdx.x * 4 + wave;
    const Chunk begin{w0 / chunks, w0 % chunks};
    struct Ids { int64_t sp[2], e[2]; bool in[2], inner[2]; };
    const auto ask_ids = [&](const Chunk& c, Ids& x) {
        const bool there = c.g < a.b;
        const int64_t base = there ? c.g * a.s * a.s : 0;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const At at = position(c.r, k, there);
            const uint32_t pos = at.inner ? (at.i - 1) * a.s + at.j - 1 : 0;
            x.in[k] = at.in;
            x.inner[k] = at.inner;
            x.sp[k] = (a.spatial_pos + base)[pos];
            x.e[k] = (a.edge_type + base)[pos];
        }
    };
    struct Targets { uint32_t sp[2], e[2]; uint64_t any[2]; };
    const auto targets = [&](const Ids& id, Targets& x) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            x.sp[k] = id.inner[k] ? (uint32_t)clamp_id(id.sp[k], a.num_spatial) : 0u;
            x.e[k] = id.inner[k] ? (uint32_t)clamp_id(id.e[k], a.num_edges) : (id.in[k] ? kVirtCode : 0u);
            x.any[k] = __ballot((x.sp[k] | x.e[k]) != 0u);
        }
    };
    uint32_t raw[NS][8];
    const auto ask_grads = [&](const Chunk& c, const Targets& x) {
        // the dwords of octets that add nothing are read where the nearest octet below that does lies, those in front of the first at the first
        const auto octets_of = [](uint64_t m) {
            m |= m >> 4; m |= m >> 2; m |= m >> 1;
            m &= 0x0101010101010101ull;
            return (uint32_t)((m * 0x0102040810204080ull) >> 56);
        };
        uint32_t octets = octets_of(x.any[0]) | octets_of(x.any[1]) << 8;
        octets |= octets << 1;      // (an odd column's dword at the end of an octet is the first of the next)
        const uint32_t below = octets & ((2u << (lane >> 2)) - 1u);
        const int from = below ? 31 - __clz((int)below) : __ffs((int)octets) - 1;
        const uint32_t at = (uint32_t)(4 * from + (lane & 3)) * 4u;
        const uint64_t off = 2 * (c.g * 8 * plane + first_of(c.r));
#pragma unroll
        for (int n = 0; n < NS; ++n)
#pragma unroll
            for (int odd_head = 0; odd_head < 2; ++odd_head) {
                const uint64_t start = reinterpret_cast<uint64_t>(dout.p[n]) + off + (odd_head ? 2 * plane : 0);
                const uint32_t mine = min(at, 2u * kChunk - 4u + ((uint32_t)start & 2u) * 2u);      // no dword without an element of the chunk
                uint64_t base = start & ~(uint64_t)3;
#pragma unroll
                for (int h = odd_head; h < 8; h += 2, base += 4u * (uint32_t)plane)      // (memory, said aloud: of a number the compiler makes a flat load)
                    raw[n][h] = *reinterpret_cast<const __attribute__((address_space(1))) uint32_t*>((const __attribute__((address_space(1))) char*)base + mine);
            }
    };
    const u16x2 want0 = c16 < 8 ? (uint16_t)(1 + c16) : (c16 == 15 ? (uint16_t)kVirtCode : (uint16_t)(c16 - 7)), want1 = (uint16_t)(9 + c16);
    const uint16_t *const from0 = codes + (c16 < 8 ? 0 : 128) + 8 * oct, *const from1 = codes + 8 * oct;
    const auto ones = [](const uint16_t* from, u16x2 want) {
        uint4 ids = *reinterpret_cast<const uint4*>(from), out;
        const auto one = [&](uint32_t v) {      // 1.0 where the code is the wanted one
            u16x2 off;      // (by hand: three instructions a pair, not the five of two compares)
            asm("v_pk_min_u16 %0, %1, %2" : "=v"(off) : "v"((u16x2)(__builtin_bit_cast(u16x2, v) ^ want)), "v"((u16x2)(uint16_t)1));
            return __builtin_bit_cast(uint32_t, (u16x2)(off * (uint16_t)0xc080 + (uint16_t)0x3f80));
        };
        out.x = one(ids.x); out.y = one(ids.y); out.z = one(ids.z); out.w = one(ids.w);
        return __builtin_bit_cast(bf16x8, out);
    };
    floatx4 sums[4][G], far_sums[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
        far_sums[g] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < 4; ++k) sums[k][g] = far_sums[g];
    }
    // this lane's column in the products, and whether it begins inside a dword in a chunk that does not
    const uint32_t* mine[G];
    uint32_t odd[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
        const int n = c16 < 8 || 2 * g + 1 >= NS ? 2 * g : 2 * g + 1;      // (without a gradient: another's)
        mine[g] = columns + (n * 8 + (c16 & 7)) * kColumn;
        const gbf16* p = n == 2 * g ? dout.p[2 * g] : dout.p[2 * g + 1 < NS ? 2 * g + 1 : 2 * g];
        odd[g] = (uint32_t)(reinterpret_cast<uintptr_t>(p) >> 1) + (uint32_t)((c16 & 7) * plane);
    }
    const auto put = [&](const Targets& x) {
#pragma unroll
        for (int n = 0; n < NS; ++n)
#pragma unroll
            for (int h = 0; h < 8; ++h) columns[(n * 8 + h) * kColumn + lane] = raw[n][h];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            codes[64 * k + lane] = (uint16_t)x.sp[k];
            codes[128 + 64 * k + lane] = (uint16_t)x.e[k];
        }
        wave_sync_lds();
    };
    const auto consume = [&](const Chunk& c, uint64_t far, uint64_t cold) {
        const uint32_t chunk_odd = (uint32_t)first_of(c.r);      // (eight planes are whole dwords)
        uint32_t shift[G];
#pragma unroll
        for (int g = 0; g < G; ++g) shift[g] = 16 * ((odd[g] + chunk_odd) & 1u);
        const auto octet = [&](int k, int g) {
            const uint32_t* from = mine[g] + 16 * k + 4 * oct;
            const uint4 w = *reinterpret_cast<const uint4*>(from);
            const uint32_t next = from[4];
            return uint4{__builtin_amdgcn_alignbit(w.y, w.x, shift[g]), __builtin_amdgcn_alignbit(w.z, w.y, shift[g]), __builtin_amdgcn_alignbit(w.w, w.z, shift[g]),
                         __builtin_amdgcn_alignbit(next, w.w, shift[g])};
        };
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const bf16x8 ones0 = ones(from0 + 32 * k, want0);
            bf16x8 v[G];
#pragma unroll
            for (int g = 0; g < G; ++g) {
                v[g] = __builtin_bit_cast(bf16x8, octet(k, g));
                sums[k][g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones0, v[g], sums[k][g], 0, 0, 0);
            }
            if (far) {
                const bf16x8 ones1 = ones(from1 + 32 * k, want1);
#pragma unroll
                for (int g = 0; g < G; ++g) far_sums[g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones1, v[g], far_sums[g], 0, 0, 0);
            }
        }
        if (cold) {
            // ids without a row: a lane's eight positions, the gradients' sum of a head in the lower eight of sixteen lanes
#pragma unroll 1
            for (int k = 0; k < 4; ++k) {
                uint4 w[G];
#pragma unroll
                for (int g = 0; g < G; ++g) w[g] = octet(k, g);
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const uint32_t sp = codes[32 * k + 8 * oct + u], e = codes[128 + 32 * k + 8 * oct + u];
                    float sum = 0.f;
#pragma unroll
                    for (int g = 0; g < G; ++g) {
                        const uint32_t pair = u < 4 ? (u < 2 ? w[g].x : w[g].y) : (u < 6 ? w[g].z : w[g].w);
                        sum += c16 < 8 || 2 * g + 1 < NS ? __uint_as_float(u & 1 ? pair & 0xffff0000u : pair << 16) : 0.f;
                    }
                    sum += __shfl_xor(sum, 8);
                    if (c16 < 8 && sum != 0.f) {
                        if (sp > kRowsSp) atomicAdd(&acc_sp[sp * H + c16], sum);
                        if (e > kRowsE && e != kVirtCode) atomicAdd(&acc_e[e * H + c16], sum);
                    }
                }
            }
        }
        wave_sync_lds();
    };
    {
        // while a chunk's products are made, the next one's gradients and the ids of the one behind it are on their way
        Ids ids;
        Targets cur, nxt;
        Chunk c = begin, c1 = begin;
        ask_ids(c, ids);
        targets(ids, cur);
        advance(c1);
        ask_ids(c1, ids);
        if (cur.any[0] | cur.any[1]) ask_grads(c, cur);
        while (c.g < a.b) {
            targets(ids, nxt);
            Chunk c2 = c1;
            advance(c2);
            ask_ids(c2, ids);
            const bool adds = cur.any[0] | cur.any[1];
            const uint32_t most = max(cur.sp[0], cur.sp[1]);
            const uint64_t far = __ballot(most > 8), cold = __ballot(most > kRowsSp || (uint16_t)(cur.e[0] + 1) > kRowsE + 1 || (uint16_t)(cur.e[1] + 1) > kRowsE + 1);
            if (adds) put(cur);
            if (nxt.any[0] | nxt.any[1]) ask_grads(c1, nxt);
            if (adds) consume(c, far, cold);
            cur = nxt;
            c = c1;
            c1 = c2;
        }
    }
    // row 4 oct + t of a block in register t
    bool number = true;
#pragma unroll
    for (int g = 0; g < G; ++g) {
        sums[0][g] = (sums[0][g] + sums[1][g]) + (sums[2][g] + sums[3][g]);
#pragma unroll
        for (int t = 0; t < 4; ++t) number &= fabsf(sums[0][g][t]) < __builtin_inff() && fabsf(far_sums[g][t]) < __builtin_inff();
    }
    if (__ballot(!number) == 0) {
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int row = 16 * m + 4 * oct + t;
                float v = 0.f;
#pragma unroll
                for (int g = 0; g < G; ++g) v += c16 < 8 || 2 * g + 1 < NS ? (m == 0 ? sums[0][g][t] : far_sums[g][t]) : 0.f;
                v += __shfl_xor(v, 8);
                if (c16 >= 8) continue;
                const int sp = row < 8 ? row + 1 : (row < 16 ? 0 : row - 7), e = row < 16 ? row - 7 : 0;      // (e 8: the virtual node)
                if (sp > 0) { if (sp < a.num_spatial) atomicAdd(&acc_sp[sp * H + c16], v); }
                else if (e < 8) { if (e < a.num_edges) atomicAdd(&acc_e[e * H + c16], v); }
                else atomicAdd(&acc_v[c16], v);
            }
    } else {
        for (Chunk c = begin; c.g < a.b; advance(c)) {
            Ids id;
            ask_ids(c, id);
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const At at = position(c.r, k, true);
                const int sp = at.inner ? clamp_id(id.sp[k], a.num_spatial) : 0, e = at.inner ? clamp_id(id.e[k], a.num_edges) : 0;
                if (!at.in) continue;
                for (int h = 0; h < H; ++h) {
                    float v = 0.f;
                    for (int n = 0; n < NS; ++n) v += ldf(dout.p[n] + (c.g * H + h) * plane + at.p);
                    if (v == 0.f) continue;
                    if (sp > 0 && sp <= kRowsSp) atomicAdd(&acc_sp[sp * H + h], v);
                    if (e > 0 && e <= kRowsE) atomicAdd(&acc_e[e * H + h], v);
                    if (!at.inner) atomicAdd(&acc_v[h], v);
                }
            }
        }
    }
    __syncthreads();
    for (int k = threadIdx.x; k < n_acc; k += 256) partial[(int64_t)blockIdx.x * n_acc + k] = acc_all[k];      // (one feature: its mean is itself)
}

// Sum of the workgroup partials in a fixed order: 64 slices of the workers per entry, then the slices.
template <typename T>
__global__ __launch_bounds__(256) void k_graph_bias_reduce(const float* __restrict__ partial, int workers, int n_sp, int n_e,
                                                           int n_v, T* __restrict__ d_sp, T* __restrict__ d_e,
                                                           T* __restrict__ d_v) {
    __shared__ float part[64][4];
    const int n = n_sp + n_e + n_v;
    const int kl = threadIdx.x % 4, slice = threadIdx.x / 4;
    const int k = blockIdx.x * 4 + kl;
    float t = 0.f;
    if (k < n)
        for (int w = slice; w < workers; w += 64 * 8) {      // eight loads at a time: one by one 1024 workers took 8 us
            float v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = w + 64 * u < workers ? partial[(int64_t)(w + 64 * u) * n + k] : 0.f;
#pragma unroll
            for (int u = 0; u < 8; ++u) t += v[u];
        }
    part[slice][kl] = t;
    __syncthreads();
    if (slice != 0 || k >= n) return;
    t = 0.f;
#pragma unroll
    for (int c = 0; c < 64; ++c) t += part[c][kl];
    if (k < n_sp) stf(d_sp + k, t);
    else if (k < n_sp + n_e) stf(d_e + (k - n_sp), t);
    else stf(d_v + (k - n_sp - n_e), t);
}

constexpr int kBiasWorkers = 1024;
constexpr int kBiasCopies = 16;

int bias_check(int b, int s, int H, int F, int num_spatial, int num_edges, int dtype, const char* who) {
    if (b < 0 || s < 0 || H < 1 || F < 1 || num_spatial < 1 || num_edges < 1 ||
        (dtype != TGT_DTYPE_F32 && dtype != TGT_DTYPE_BF16)) {
        set_error("%s: bad size or dtype", who);
        return TGT_ERR_INVALID_ARG;
    }
    if (H > kMaxHeads) {
        set_error("%s: at most %d heads", who, kMaxHeads);
        return TGT_ERR_UNSUPPORTED;
    }
    return TGT_OK;
}

// One workgroup per graph.  Distances (uint16: at most 2 * 510) live in LDS; the intermediate nodes (int16) too
// for graphs of up to 128 nodes, beyond that they are kept in the output array itself (every (i, j) has one
// owner thread, so nobody else reads them).  Within one k the k-th row and column do not change
// (M[k][k] = 0), so all (i, j) of a step can be relaxed at once and give exactly the sequential result.
constexpr int kFwMax = 256;
constexpr int kFwLdsPath = 128;      // largest graph whose intermediate nodes fit in LDS beside the distances
constexpr int kFwInf = 510;          // data/algos.pyx:30

// 1024 threads: thread (r, j) = (tid / COLS, tid % COLS) owns column j of rows r, r + 1024 / COLS, ...: no
// division per element, row i's M[i][k] is one LDS word for all lanes of a row, M[k][j] runs along the lanes.
template <int COLS, bool PATH_IN_LDS>
__global__ __launch_bounds__(1024) void k_floyd_warshall(const uint8_t* __restrict__ adj, const int32_t* __restrict__ n_nodes,
                                                         int n_max, int32_t* __restrict__ dist, int32_t* __restrict__ path) {
    extern __shared__ uint16_t lds[];
    const int g = blockIdx.x;
    const int n = n_nodes ? min(max(n_nodes[g], 0), n_max) : n_max;      // a count outside [0, n_max] is clamped
    uint16_t* M = lds;                                   // [n][n]
    int16_t* P = reinterpret_cast<int16_t*>(lds + n * n);
    const uint8_t* A = adj + (int64_t)g * n_max * n_max;
    int32_t* D = dist + (int64_t)g * n_max * n_max;
    int32_t* Q = path + (int64_t)g * n_max * n_max;
    const int j = threadIdx.x % COLS, r = threadIdx.x / COLS;
    constexpr int kRows = 1024 / COLS;
    if (j < n)
        for (int i = r; i < n; i += kRows) {
            const uint16_t w = A[i * n_max + j];
            M[i * n + j] = i == j ? 0 : (w == 0 ? kFwInf : w);       // :27-32
            if (PATH_IN_LDS) P[i * n + j] = -1;
            else Q[i * n_max + j] = -1;
        }
    __syncthreads();
    for (int k = 0; k < n; ++k) {
        if (j < n && j != k) {
            const uint16_t kj = M[k * n + j];
            for (int i = r; i < n; i += kRows) {
                const uint16_t c = M[i * n + k] + kj;
                if (M[i * n + j] > c && i != k) {        // row k and column k never improve through k
                    M[i * n + j] = c;
                    if (PATH_IN_LDS) P[i * n + j] = (int16_t)k;
                    else Q[i * n_max + j] = k;
                }
            }
        }
        __syncthreads();
    }
    if (j < n)
        for (int i = r; i < n; i += kRows) {
            const bool far = M[i * n + j] >= kFwInf;     // :49-53
            D[i * n_max + j] = far ? kFwInf : M[i * n + j];
            if (PATH_IN_LDS) Q[i * n_max + j] = far ? kFwInf : P[i * n + j];
            else if (far) Q[i * n_max + j] = kFwInf;
        }
}

}  // namespace
}  // namespace tgt

extern "C" {

int tgt_graph_attn_bias_fwd(const void* d_attn_bias, const int64_t* d_spatial_pos, const int64_t* d_edge_type, int F,
                            const void* d_spatial_table, int num_spatial, const void* d_edge_table, int num_edges,
                            const void* d_virtual_dist, int b, int s, int H, int dtype, void* d_out, void* stream) {
    using namespace tgt;
    const int rc = bias_check(b, s, H, F, num_spatial, num_edges, dtype, "tgt_graph_attn_bias_fwd");
    if (rc != TGT_OK) return rc;
    if (b == 0) return TGT_OK;
    if (!d_attn_bias || !d_spatial_table || !d_edge_table || !d_virtual_dist || !d_out ||
        (s > 0 && (!d_spatial_pos || !d_edge_type))) {
        set_error("tgt_graph_attn_bias_fwd: null pointer");
        return TGT_ERR_INVALID_ARG;
    }
    BiasArgs a{d_attn_bias, d_spatial_pos, d_edge_type, d_spatial_table, d_edge_table, d_virtual_dist,
               b, s, H, F, num_spatial, num_edges};
    const int64_t total = (int64_t)b * (s + 1) * (s + 1);
    const dim3 grid((unsigned)((total + 255) / 256));
    hipStream_t st = (hipStream_t)stream;
    KernelTimer timer(KS_GRAPH_BIAS_FWD, st);
    const size_t tab_bytes = sizeof(float) * (size_t)(num_spatial + num_edges + 1) * H;
    if (H == 8 && tab_bytes <= 32 * 1024) {
        const dim3 g8((unsigned)std::min<int64_t>((total + 255) / 256, 4096));
        if (dtype == TGT_DTYPE_F32) hipLaunchKernelGGL((k_graph_bias_fwd8<float>), g8, dim3(256), tab_bytes, st, a, (float*)d_out);
        else hipLaunchKernelGGL((k_graph_bias_fwd8<gbf16>), g8, dim3(256), tab_bytes, st, a, (gbf16*)d_out);
    } else if (dtype == TGT_DTYPE_F32) {
        hipLaunchKernelGGL((k_graph_bias_fwd<float>), grid, dim3(256), 0, st, a, (float*)d_out);
    } else {
        hipLaunchKernelGGL((k_graph_bias_fwd<gbf16>), grid, dim3(256), 0, st, a, (gbf16*)d_out);
    }
    TGT_HIP_CHECK(hipGetLastError());
    return TGT_OK;
}

int64_t tgt_graph_attn_bias_bwd_workspace_bytes(int num_spatial, int num_edges, int H) {
    if (num_spatial < 1 || num_edges < 1 || H < 1) return 0;
    return (int64_t)sizeof(float) * tgt::kBiasWorkers * (num_spatial + num_edges + 1) * H;
}

int tgt_graph_attn_bias_bwd_sum(const void* const* d_douts, int n_douts, const int64_t* d_spatial_pos, const int64_t* d_edge_type, int F,
                            int num_spatial, int num_edges, int b, int s, int H, int dtype, void* d_dspatial_table,
                            void* d_dedge_table, void* d_dvirtual_dist, void* d_workspace, int64_t workspace_bytes,
                            void* stream) {
    using namespace tgt;
    const int rc = bias_check(b, s, H, F, num_spatial, num_edges, dtype, "tgt_graph_attn_bias_bwd");
    if (rc != TGT_OK) return rc;
    if (!d_dspatial_table || !d_dedge_table || !d_dvirtual_dist ||
        !d_douts || n_douts < 1 || n_douts > 4 || (b > 0 && ((s > 0 && (!d_spatial_pos || !d_edge_type))))) {
        set_error("tgt_graph_attn_bias_bwd: null pointer, or not 1 to 4 gradients");
        return TGT_ERR_INVALID_ARG;
    }
    for (int k = 0; k < n_douts; ++k)
        if (b > 0 && !d_douts[k]) {
            set_error("tgt_graph_attn_bias_bwd: null pointer");
            return TGT_ERR_INVALID_ARG;
        }
    const int n_acc = (num_spatial + num_edges + 1) * H;
    if ((size_t)n_acc * sizeof(float) > 128 * 1024) {
        set_error("tgt_graph_attn_bias_bwd: (num_spatial + num_edges + 1) * H = %d table entries exceed the %d kept on chip",
                  n_acc, 128 * 1024 / 4);
        return TGT_ERR_UNSUPPORTED;
    }
    if (!d_workspace || workspace_bytes < tgt_graph_attn_bias_bwd_workspace_bytes(num_spatial, num_edges, H)) {
        set_error("tgt_graph_attn_bias_bwd: workspace of %lld bytes needed, got %lld",
                  (long long)tgt_graph_attn_bias_bwd_workspace_bytes(num_spatial, num_edges, H), (long long)workspace_bytes);
        return TGT_ERR_WORKSPACE;
    }
    BiasArgs a{nullptr, d_spatial_pos, d_edge_type, nullptr, nullptr, nullptr, b, s, H, F, num_spatial, num_edges};
    const int64_t total = (int64_t)b * (s + 1) * (s + 1);
    int workers = (int)std::max<int64_t>(1, std::min<int64_t>((total + 255) / 256, kBiasWorkers));
    hipStream_t st = (hipStream_t)stream;
    KernelTimer timer(KS_GRAPH_BIAS_BWD, st);
    float* partial = (float*)d_workspace;
    int copies = kBiasCopies;
    while (copies > 1 && (size_t)n_acc * copies * sizeof(float) > 16 * 1024) copies /= 2;      // more workgroups per CU beat more copies
    size_t lds = (size_t)n_acc * copies * sizeof(float);
    const unsigned rgrid = (unsigned)((n_acc + 3) / 4);
    auto launch = [&](auto kernel, auto reduce, auto dout, auto* dsp, auto* de, auto* dv, auto... more) -> int {
        if (lds > 48 * 1024)
            TGT_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                              128 * 1024));
        hipLaunchKernelGGL(kernel, dim3(workers), dim3(256), lds, st, a, dout, partial, copies, more...);
        hipLaunchKernelGGL(reduce, dim3(rgrid), dim3(256), 0, st, (const float*)partial, workers, num_spatial * H, num_edges * H, H,
                           dsp, de, dv);
        return TGT_OK;
    };
    // registers for the frequent ids need one pass over the heads; the prefetching loop one pass over the features too
    const int variant = H > 8 ? 0 : (F > kBiasFeat ? 1 : (F > 1 ? 2 : 3));
    if (n_douts > 1 && variant != 3) {
        set_error("tgt_graph_attn_bias_bwd_sum: several gradients with at most 8 heads and one edge feature only");
        return TGT_ERR_UNSUPPORTED;
    }
    int lrc;
    auto run = [&](auto tag) -> int {
        using T = decltype(tag);
        auto* red = &k_graph_bias_reduce<T>;
        BiasGrads<T> dout;
        for (int k = 0; k < 4; ++k) dout.p[k] = (const T*)d_douts[k < n_douts ? k : 0];
        T *dsp = (T*)d_dspatial_table, *de = (T*)d_dedge_table, *dv = (T*)d_dvirtual_dist;
        if constexpr (std::is_same<T, gbf16>::value) {
            // Tables that leave room for two workgroups per CU: 512 spatial and 64 edge ids 67 us without the matrix cores, 52 with them (three gradients
            // 91, 66), 512 and 1537 159 and 73; with less room a CU would be left to one.
            const size_t mm_lds = (n_douts == 4 ? bias_mm_lds<4>() : n_douts == 3 ? bias_mm_lds<3>() : n_douts == 2 ? bias_mm_lds<2>() : bias_mm_lds<1>()) + (size_t)n_acc * sizeof(float);
            if (variant == 3 && H == 8 && b > 0 && s + 1 >= kBiasMinSide && s + 1 <= kBiasMaxSide && mm_lds <= kBiasMaxLds) {
                const int chunks = ((s + 1) * (s + 1) + kChunk - 1) / kChunk;
                const uint32_t inv_s1 = (uint32_t)((((uint64_t)1 << 32) + s) / (uint32_t)(s + 1));
                workers = (int)std::min<int64_t>(std::min<int64_t>(((int64_t)b * chunks + 3) / 4, kBiasWorkers), (int64_t)num_cus() * (int64_t)(160 * 1024 / mm_lds));      // one round
                lds = mm_lds;
                const auto mm = [&](auto kernel) { return launch(kernel, red, dout, dsp, de, dv, chunks, inv_s1); };
                return n_douts == 4 ? mm(&k_graph_bias_bwd_mm<4>) : n_douts == 3 ? mm(&k_graph_bias_bwd_mm<3>) : n_douts == 2 ? mm(&k_graph_bias_bwd_mm<2>) : mm(&k_graph_bias_bwd_mm<1>);
            }
        }
        if (n_douts == 4) return launch(&k_graph_bias_bwd<T, kBiasHot, true, 1, 4>, red, dout, dsp, de, dv);
        if (n_douts == 3) return launch(&k_graph_bias_bwd<T, kBiasHot, true, 1, 3>, red, dout, dsp, de, dv);
        if (n_douts == 2) return launch(&k_graph_bias_bwd<T, kBiasHot, true, 1, 2>, red, dout, dsp, de, dv);
        return variant == 3   ? launch(&k_graph_bias_bwd<T, kBiasHot, true, 1, 1>, red, dout, dsp, de, dv)
               : variant == 2 ? launch(&k_graph_bias_bwd<T, kBiasHot, true, kBiasFeat, 1>, red, dout, dsp, de, dv)
               : variant == 1 ? launch(&k_graph_bias_bwd<T, kBiasHot, false, kBiasFeat, 1>, red, dout, dsp, de, dv)
                              : launch(&k_graph_bias_bwd<T, 0, false, kBiasFeat, 1>, red, dout, dsp, de, dv);
    };
    lrc = dtype == TGT_DTYPE_F32 ? run(float()) : run(gbf16());
    if (lrc != TGT_OK) return lrc;
    TGT_HIP_CHECK(hipGetLastError());
    return TGT_OK;
}

int tgt_graph_attn_bias_bwd(const void* d_dout, const int64_t* d_spatial_pos, const int64_t* d_edge_type, int F,
                            int num_spatial, int num_edges, int b, int s, int H, int dtype, void* d_dspatial_table,
                            void* d_dedge_table, void* d_dvirtual_dist, void* d_workspace, int64_t workspace_bytes,
                            void* stream) {
    return tgt_graph_attn_bias_bwd_sum(&d_dout, 1, d_spatial_pos, d_edge_type, F, num_spatial, num_edges, b, s, H, dtype, d_dspatial_table,
                                       d_dedge_table, d_dvirtual_dist, d_workspace, workspace_bytes, stream);
}

int tgt_floyd_warshall(const uint8_t* d_adj, const int32_t* d_n_nodes, int num_graphs, int n_max, int32_t* d_dist,
                       int32_t* d_path, void* stream) {
    using namespace tgt;
    if (num_graphs < 0 || n_max < 1 || (num_graphs > 0 && (!d_adj || !d_dist || !d_path))) {
        set_error("tgt_floyd_warshall: null pointer or bad size");
        return TGT_ERR_INVALID_ARG;
    }
    if (n_max > kFwMax) {
        set_error("tgt_floyd_warshall: graphs of up to %d nodes (got n_max = %d)", kFwMax, n_max);
        return TGT_ERR_UNSUPPORTED;
    }
    if (num_graphs == 0) return TGT_OK;
    hipStream_t st = (hipStream_t)stream;
    if (n_max <= kFwLdsPath) {
        const size_t lds = (size_t)n_max * n_max * 4;
        static bool raised = false;
        if (!raised && lds > 48 * 1024) {
            TGT_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_floyd_warshall<128, true>),
                                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)(kFwLdsPath * kFwLdsPath * 4)));
            raised = true;
        }
        hipLaunchKernelGGL((k_floyd_warshall<128, true>), dim3(num_graphs), dim3(1024), lds, st, d_adj, d_n_nodes, n_max, d_dist,
                           d_path);
    } else {
        const size_t lds = (size_t)n_max * n_max * 2;      // up to 128 KB of the CU's 160
        static bool raised = false;
        if (!raised) {
            TGT_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_floyd_warshall<256, false>),
                                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)(kFwMax * kFwMax * 2)));
            raised = true;
        }
        hipLaunchKernelGGL((k_floyd_warshall<256, false>), dim3(num_graphs), dim3(1024), lds, st, d_adj, d_n_nodes, n_max, d_dist,
                           d_path);
    }
    TGT_HIP_CHECK(hipGetLastError());
    return TGT_OK;
}

}  // extern "C"
