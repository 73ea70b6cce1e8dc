// Input features of the graph-level model: GraphNodeFeature.forward
// (models/graphormer_graph_level.py:18-60) and the gradients of its four embedding tables.
//
//   out[g, 0, :]     = graph_token
//   out[g, 1 + i, :] = sum_f atom_table[x[g, i, f]] + in_degree_table[in_degree[g, i]]
//                      + out_degree_table[out_degree[g, i]]
//
// The reference runs three embedding lookups, a sum over the features, two adds, a repeat and a
// concatenation; here one kernel reads the ids and writes every output row once.  The backward adds the output gradient
// into float copies of the tables (row 0 of the three lookup tables is the padding index and gets none) and a
// last kernel adds the copies up and hands the sums over in the caller's type.
//
// With a few dozen atom types every table row is shared by hundreds of node rows, and atomics on one address serialise
// (55 us for the 33 K rows of 256 padded graphs into one copy, 43 with the fill into 64, in LDS as slow as in memory).  Tables that
// fit a workgroup's LDS twice are summed there without atomics: a wave has a table to itself.  Larger ones are added to
// with vector-memory atomics, neighbouring workgroups into different copies (up to 64, at most 16 MB in all): their results agree to
// rounding between runs, not bit for bit.
#include "common.h"
#include <algorithm>

namespace tgt {
namespace {

struct nbf16 { uint16_t x; };
__device__ __forceinline__ float ldf(const float* p) { return *p; }
__device__ __forceinline__ float ldf(const nbf16* p) { return __uint_as_float(((uint32_t)p->x) << 16); }
__device__ __forceinline__ void stf(float* p, float v) { *p = v; }
__device__ __forceinline__ void stf(nbf16* p, float v) {
    const __bf16 b = static_cast<__bf16>(v);
    p->x = __builtin_bit_cast(uint16_t, b);
}
__device__ __forceinline__ int clamp_id(int64_t v, int n) { return v < 0 ? 0 : (v >= n ? n - 1 : (int)v); }

struct NodeFeatArgs {
    const int64_t* x;            // [b, s, Fx]
    const int64_t* in_degree;    // [b, s]
    const int64_t* out_degree;   // [b, s]
    int b, s, Fx, C, num_atoms, num_in, num_out;
    int pad_rows;                // 1: row 0 of the atom table is a padding index (no gradient); 0: an ordinary row
    int has_degree, has_token;   // without degrees: the atom sum alone; without token: s rows per graph, no row 0
};

// one thread per (graph, node, channel), channel fastest
template <typename T>
__global__ __launch_bounds__(256) void k_node_feature_fwd(NodeFeatArgs a, const T* __restrict__ atom, const T* __restrict__ tin,
                                                          const T* __restrict__ tout, const T* __restrict__ token,
                                                          T* __restrict__ out) {
    const int rows = a.s + a.has_token;
    const int64_t total = (int64_t)a.b * rows * a.C;
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= total) return;
    const int c = (int)(t % a.C);
    const int64_t row = t / a.C;
    const int node = (int)(row % rows) + 1 - a.has_token;             // 0 = the graph token's row
    const int64_t g = row / rows;
    float v;
    if (node == 0) {
        v = ldf(token + c);                                           // (:52-56)
    } else {
        const int64_t p = g * a.s + (node - 1);
        v = 0.f;
        for (int f = 0; f < a.Fx; ++f) v += ldf(atom + (int64_t)clamp_id(a.x[p * a.Fx + f], a.num_atoms) * a.C + c);   // (:45)
        if (a.has_degree) {
            v += ldf(tin + (int64_t)clamp_id(a.in_degree[p], a.num_in) * a.C + c);                                      // (:46-50)
            v += ldf(tout + (int64_t)clamp_id(a.out_degree[p], a.num_out) * a.C + c);
        }
    }
    stf(out + t, v);
}

// The same, 16 bytes of a row per thread: C a multiple of them, every table and `out` 16-byte aligned, fewer than 2^31 threads.  Bound by the two
// dependent reads of a row's ids and table rows; with a thread per channel every lane divided 64-bit numbers four times and wrote 2 bytes.
// 33 K rows of 64 channels, bf16: 11.3 / 4.4 us.
template <typename T> constexpr int kFeatVec = 16 / (int)sizeof(T);
template <typename T> struct FeatVec { T e[kFeatVec<T>]; };
template <typename T>
__global__ __launch_bounds__(256) void k_node_feature_fwd_vec(NodeFeatArgs a, const T* __restrict__ atom, const T* __restrict__ tin, const T* __restrict__ tout,
                                                              const T* __restrict__ token, T* __restrict__ out) {
    constexpr int V = kFeatVec<T>;
    const uint32_t rows = a.s + a.has_token, per = a.C / V, t = blockIdx.x * 256u + threadIdx.x, row = t / per, c = t % per * V;
    if (row >= (uint32_t)a.b * rows) return;
    const uint32_t g = row / rows;
    const int node = (int)(row % rows) + 1 - a.has_token;
    const auto ask = [&](const T* table, int r) { return *reinterpret_cast<const uint4*>(table + (int64_t)r * a.C + c); };
    uint4 u;
    if (node == 0) u = ask(token, 0);
    else {
        const int64_t p = (int64_t)g * a.s + (node - 1);
        float v[V];
#pragma unroll
        for (int i = 0; i < V; ++i) v[i] = 0.f;
        const auto add = [&](const uint4& w) {
            const FeatVec<T> x = __builtin_bit_cast(FeatVec<T>, w);
#pragma unroll
            for (int i = 0; i < V; ++i) v[i] += ldf(x.e + i);
        };
        int64_t din = 0, dout = 0;
        if (a.has_degree) { din = a.in_degree[p]; dout = a.out_degree[p]; }
        for (int f = 0; f < a.Fx; ++f) add(ask(atom, clamp_id(a.x[p * a.Fx + f], a.num_atoms)));
        if (a.has_degree) {
            const uint4 x = ask(tin, clamp_id(din, a.num_in)), y = ask(tout, clamp_id(dout, a.num_out));
            add(x);
            add(y);
        }
        FeatVec<T> o;
#pragma unroll
        for (int i = 0; i < V; ++i) stf(o.e + i, v[i]);
        u = __builtin_bit_cast(uint4, o);
    }
    *reinterpret_cast<uint4*>(out + (int64_t)row * a.C + c) = u;
}

__global__ __launch_bounds__(256) void k_fill_zero(float* __restrict__ p, int64_t n) {
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (t < n) p[t] = 0.f;
}

// One wave per output row (lane = channel, channels beyond 64 in further passes): the ids of a row are read once
// by the whole wave, the row's position in the batch costs one division.  acc is the float copy of the tables in
// memory: float [num_atoms + num_in + num_out + 1][C].
template <typename T>
__device__ __forceinline__ void node_feature_bwd_row(const NodeFeatArgs& a, const T* __restrict__ dout, int64_t row, int lane,
                                                     float* acc) {
    const int rows = a.s + a.has_token;
    const int64_t g = row / rows;
    const int node = (int)(row - g * rows) + 1 - a.has_token;
    float* acc_in = acc + (int64_t)a.num_atoms * a.C;
    float* acc_out = acc_in + (int64_t)a.num_in * a.C;
    float* acc_tok = acc_out + (int64_t)a.num_out * a.C;
    const T* d_row = dout + row * a.C;
    if (node == 0) {
        for (int c = lane; c < a.C; c += 64) {
            const float d = ldf(d_row + c);
            if (d != 0.f) atomicAdd(acc_tok + c, d);
        }
        return;
    }
    const int64_t p = g * a.s + (node - 1);
    int ii = 0, io = 0;
    if (a.has_degree) {
        ii = clamp_id(a.in_degree[p], a.num_in);
        io = clamp_id(a.out_degree[p], a.num_out);
    }
    for (int c = lane; c < a.C; c += 64) {
        const float d = ldf(d_row + c);
        if (d == 0.f) continue;
        for (int f = 0; f < a.Fx; ++f) {
            const int id = clamp_id(a.x[p * a.Fx + f], a.num_atoms);
            if (id >= a.pad_rows) atomicAdd(acc + (int64_t)id * a.C + c, d);        // row 0 = padding index
        }
        if (ii > 0) atomicAdd(acc_in + (int64_t)ii * a.C + c, d);
        if (io > 0) atomicAdd(acc_out + (int64_t)io * a.C + c, d);
    }
}

template <typename T>
__global__ __launch_bounds__(256) void k_node_feature_bwd(NodeFeatArgs a, const T* __restrict__ dout, float* __restrict__ acc,
                                                          int copies, int64_t n_acc) {
    const int64_t n_rows = (int64_t)a.b * (a.s + a.has_token);
    const int64_t row = (int64_t)blockIdx.x * 4 + threadIdx.x / 64;
    // neighbouring workgroups add into different copies of the sums: rows that many positions share serialise less
    if (row < n_rows) node_feature_bwd_row(a, dout, row, threadIdx.x % 64, acc + (blockIdx.x % copies) * n_acc);
}

// Tables in LDS.  A workgroup takes a run of rows for all tables: wave w adds the rows of set w / tables to that set's copy of table w % tables,
// lane = channel, so nobody else writes there and the sums come in row order.  Bound by that chain, one LDS read, add and write per row, and
// by the loads in front of it, sixteen rows at a time.  33 K rows of 64 channels, tables of 64 + 64 + 64 + 1 rows: 20 us, and 5
// for the sum of 256 copies; with atomics 33, 6 for their fill and 4.
constexpr int kFeatRows = 16, kFeatSets = 4;
template <typename T>
__global__ __launch_bounds__(64 * 3 * kFeatSets) void k_node_feature_bwd_lds(NodeFeatArgs a, const T* __restrict__ dout, float* __restrict__ partial,
                                                                             int n_acc, int tables, int sets) {
    extern __shared__ __align__(16) float sums[];      // [sets][n_acc]
    const bool fours = n_acc % 4 == 0;
    if (fours) {
#pragma unroll 4
        for (int i = threadIdx.x; i < sets * n_acc / 4; i += blockDim.x) reinterpret_cast<float4*>(sums)[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    } else
        for (int i = threadIdx.x; i < sets * n_acc; i += blockDim.x) sums[i] = 0.f;
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), table = wave % tables, set = wave / tables;
    float* mine = sums + set * n_acc;
    float* token = mine + (a.num_atoms + a.num_in + a.num_out) * a.C;
    const int64_t* ids = a.x;
    int F = a.Fx, num = a.num_atoms, least = a.pad_rows;
    if (table == 1) { ids = a.in_degree; F = 1; num = a.num_in; least = 1; mine += a.num_atoms * a.C; }
    if (table == 2) { ids = a.out_degree; F = 1; num = a.num_out; least = 1; mine += (a.num_atoms + a.num_in) * a.C; }
    if (a.s == 0) F = 0;      // token rows only
    const int rows = a.s + a.has_token, n_rows = a.b * rows, per = (n_rows + gridDim.x - 1) / gridDim.x;
    const int r0 = per * blockIdx.x, r1 = min(r0 + per, n_rows), last = a.b * a.s - 1;
    // every load of sixteen rows is asked for before the first is used, also where there is nothing to add (another row's is read then)
    for (int row = r0 + kFeatRows * set; row < r1; row += kFeatRows * sets) {
        const int g0 = (uint32_t)row / (uint32_t)rows;
        int at = row - g0 * rows, p = g0 * a.s + at - a.has_token;      // the row's place in its graph, the position of its ids
        int pos[kFeatRows];
        bool node[kFeatRows];
#pragma unroll
        for (int u = 0; u < kFeatRows; ++u) {
            node[u] = !(a.has_token && at == 0);
            pos[u] = max(0, min(p, last));
            at = at + 1 == rows ? 0 : at + 1;
            p += !(a.has_token && at == 0);
        }
        for (int c = lane; c < a.C; c += 64) {
            float d[kFeatRows];
#pragma unroll
            for (int u = 0; u < kFeatRows; ++u) d[u] = ldf(dout + (int64_t)min(row + u, r1 - 1) * a.C + c);
            for (int f = 0; f < F; ++f) {
                int64_t id[kFeatRows];
#pragma unroll
                for (int u = 0; u < kFeatRows; ++u) id[u] = ids[(int64_t)pos[u] * F + f];
#pragma unroll
                for (int u = 0; u < kFeatRows; ++u) {
                    const int to = clamp_id(id[u], num);
                    if (row + u < r1 && node[u] && to >= least) mine[to * a.C + c] += d[u];
                }
            }
            if (table == 0) {
#pragma unroll
                for (int u = 0; u < kFeatRows; ++u)
                    if (row + u < r1 && !node[u]) token[c] += d[u];
            }
        }
    }
    __syncthreads();
    float* __restrict__ out = partial + (int64_t)blockIdx.x * n_acc;
    if (fours) {
#pragma unroll 2
        for (int i = threadIdx.x; i < n_acc / 4; i += blockDim.x) {
            float4 t[kFeatSets];
#pragma unroll
            for (int k = 0; k < kFeatSets; ++k) t[k] = reinterpret_cast<const float4*>(sums)[(k < sets ? k : 0) * (n_acc / 4) + i];
#pragma unroll
            for (int k = 1; k < kFeatSets; ++k)
                if (k < sets) { t[0].x += t[k].x; t[0].y += t[k].y; t[0].z += t[k].z; t[0].w += t[k].w; }
            reinterpret_cast<float4*>(out)[i] = t[0];
        }
    } else
        for (int i = threadIdx.x; i < n_acc; i += blockDim.x) {
            float t = sums[i];
            for (int k = 1; k < sets; ++k) t += sums[k * n_acc + i];
            out[i] = t;
        }
}

// Sum of the copies, handed over in the caller's type.  64 entries per workgroup along the lanes; the four waves take
// every fourth copy each (sixteen loads in flight per lane) and their partial sums are added in wave order.
template <typename T>
__global__ __launch_bounds__(256) void k_node_feature_finish(const float* __restrict__ acc, int64_t n_atom, int64_t n_in,
                                                             int64_t n_out, int64_t n_tok, int copies, T* __restrict__ d_atom,
                                                             T* __restrict__ d_in, T* __restrict__ d_out, T* __restrict__ d_tok) {
    __shared__ float part[4][64];
    const int64_t n_acc = n_atom + n_in + n_out + n_tok;
    const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
    const int64_t t = (int64_t)blockIdx.x * 64 + lane;
    float v = 0.f;
    if (t < n_acc) {
        for (int c0 = wave; c0 < copies; c0 += 64) {
            float x[16];
#pragma unroll
            for (int u = 0; u < 16; ++u) x[u] = c0 + 4 * u < copies ? acc[(int64_t)(c0 + 4 * u) * n_acc + t] : 0.f;
#pragma unroll
            for (int u = 0; u < 16; u += 4) v += (x[u] + x[u + 1]) + (x[u + 2] + x[u + 3]);
        }
    }
    part[wave][lane] = v;
    __syncthreads();
    if (wave != 0 || t >= n_acc) return;
    v = (part[0][lane] + part[1][lane]) + (part[2][lane] + part[3][lane]);
    if (t < n_atom) stf(d_atom + t, v);
    else if (t < n_atom + n_in) stf(d_in + (t - n_atom), v);
    else if (t < n_atom + n_in + n_out) stf(d_out + (t - n_atom - n_in), v);
    else stf(d_tok + (t - n_atom - n_in - n_out), v);
}

// Copies of the tables in a workgroup's LDS (0: none): two to four, at less than a CU's 160 KB.  One alone leaves the chain of a table's rows to one wave:
// 33 K rows, tables of 321 and 579 rows of 64 channels 50 and 57 us whatever the ids; with atomics 30 and 33 where all rows are used alike, 71 and
// 71 where four of each table are.  Two, of 257 rows: 33, atomics 30 and 121.
inline int node_feat_sets(int64_t n_acc) {
    const int sets = (int)std::min<int64_t>(kFeatSets, (156 << 10) / (n_acc * (int64_t)sizeof(float)));
    return sets >= 2 ? sets : 0;
}
// Copies of the float sums in memory, 16 MB in all at most.  From LDS: one per workgroup, a workgroup per CU at most (rows are counted in 32 bits
// there).  With atomics: at most 64.
inline int node_feat_copies(int64_t n_acc) {
    const int64_t fit = std::max<int64_t>(1, (16 << 20) / (n_acc * (int64_t)sizeof(float)));
    if (node_feat_sets(n_acc) > 0) return (int)std::min<int64_t>(num_cus(), fit);
    int copies = 64;
    while (copies > fit) copies /= 2;
    return copies;
}

int node_feat_check(int b, int s, int Fx, int C, int num_atoms, int num_in, int num_out, int dtype, const char* who) {
    if (b < 0 || s < 0 || Fx < 1 || C < 1 || num_atoms < 1 || num_in < 1 || num_out < 1 ||
        (dtype != TGT_DTYPE_F32 && dtype != TGT_DTYPE_BF16)) {
        set_error("%s: bad size or dtype", who);
        return TGT_ERR_INVALID_ARG;
    }
    return TGT_OK;
}

}  // namespace
}  // namespace tgt

namespace tgt {
namespace {

int node_feature_fwd_impl(NodeFeatArgs a, const void* d_atom_table, const void* d_in_table, const void* d_out_table,
                          const void* d_graph_token, int dtype, void* d_out, void* stream) {
    const int64_t total = (int64_t)a.b * (a.s + a.has_token) * a.C;
    if (total == 0) return TGT_OK;
    const dim3 grid((unsigned)((total + 255) / 256));
    hipStream_t st = (hipStream_t)stream;
    const int vec = dtype == TGT_DTYPE_F32 ? kFeatVec<float> : kFeatVec<nbf16>;
    const auto where = [](const void* p) { return reinterpret_cast<uintptr_t>(p); };      // (what is not in use is not read)
    const uintptr_t ends = where(d_atom_table) | where(d_out) | (a.has_degree ? where(d_in_table) | where(d_out_table) : 0) | (a.has_token ? where(d_graph_token) : 0);
    if (a.C % vec == 0 && ends % 16 == 0 && total / vec <= INT32_MAX) {
        const dim3 few((unsigned)((total / vec + 255) / 256));
        if (dtype == TGT_DTYPE_F32)
            hipLaunchKernelGGL((k_node_feature_fwd_vec<float>), few, dim3(256), 0, st, a, (const float*)d_atom_table, (const float*)d_in_table, (const float*)d_out_table,
                               (const float*)d_graph_token, (float*)d_out);
        else
            hipLaunchKernelGGL((k_node_feature_fwd_vec<nbf16>), few, dim3(256), 0, st, a, (const nbf16*)d_atom_table, (const nbf16*)d_in_table, (const nbf16*)d_out_table,
                               (const nbf16*)d_graph_token, (nbf16*)d_out);
    } else if (dtype == TGT_DTYPE_F32)
        hipLaunchKernelGGL((k_node_feature_fwd<float>), grid, dim3(256), 0, st, a, (const float*)d_atom_table, (const float*)d_in_table,
                           (const float*)d_out_table, (const float*)d_graph_token, (float*)d_out);
    else
        hipLaunchKernelGGL((k_node_feature_fwd<nbf16>), grid, dim3(256), 0, st, a, (const nbf16*)d_atom_table, (const nbf16*)d_in_table,
                           (const nbf16*)d_out_table, (const nbf16*)d_graph_token, (nbf16*)d_out);
    TGT_HIP_CHECK(hipGetLastError());
    return TGT_OK;
}

// acc layout: [num_atoms][C], [num_in][C], [num_out][C], [1][C]; tables that are not in use have num = 0 rows here
int node_feature_bwd_impl(NodeFeatArgs a, const void* d_dout, int dtype, void* d_datom, void* d_din, void* d_dout_table,
                          void* d_dtoken, float* acc, void* stream) {
    hipStream_t st = (hipStream_t)stream;
    const int64_t n_atom = (int64_t)a.num_atoms * a.C, n_in = a.has_degree ? (int64_t)a.num_in * a.C : 0,
                  n_out = a.has_degree ? (int64_t)a.num_out * a.C : 0, n_tok = a.has_token ? a.C : 0;
    const int64_t n_acc = n_atom + n_in + n_out + n_tok;
    if (!a.has_degree) a.num_in = a.num_out = 0;          // the kernel's offsets of the sums that follow the atom table
    const int64_t n_rows = (int64_t)a.b * (a.s + a.has_token);
    int copies = node_feat_copies(n_acc);
    if (const int sets = node_feat_sets(n_acc); sets > 0 && n_rows + kFeatRows * kFeatSets <= INT32_MAX) {
        // a workgroup for every sixteen rows of each set, at most one per copy
        copies = (int)std::min<int64_t>(copies, (n_rows + kFeatRows * sets - 1) / (kFeatRows * sets));
        if (copies > 0) {
            const int tables = a.has_degree ? 3 : 1, lds = (int)(sets * n_acc * sizeof(float));
            static std::atomic<uint64_t> done[2];
            const auto run = [&](auto kernel, const auto* dout, std::atomic<uint64_t>& d) {
                if (int rc = allow_lds(reinterpret_cast<const void*>(kernel), 156 << 10, d)) return rc;
                hipLaunchKernelGGL(kernel, dim3(copies), dim3(64 * tables * sets), lds, st, a, dout, acc, (int)n_acc, tables, sets);
                return (int)TGT_OK;
            };
            const int rc = dtype == TGT_DTYPE_F32 ? run(&k_node_feature_bwd_lds<float>, (const float*)d_dout, done[0])
                                                  : run(&k_node_feature_bwd_lds<nbf16>, (const nbf16*)d_dout, done[1]);
            if (rc != TGT_OK) return rc;
        }
    } else {
        hipLaunchKernelGGL(k_fill_zero, dim3((unsigned)((n_acc * copies + 255) / 256)), dim3(256), 0, st, acc, n_acc * copies);
        const dim3 grid((unsigned)((n_rows + 3) / 4));
        if (n_rows > 0) {
            if (dtype == TGT_DTYPE_F32) hipLaunchKernelGGL((k_node_feature_bwd<float>), grid, dim3(256), 0, st, a, (const float*)d_dout, acc, copies, n_acc);
            else hipLaunchKernelGGL((k_node_feature_bwd<nbf16>), grid, dim3(256), 0, st, a, (const nbf16*)d_dout, acc, copies, n_acc);
        }
    }
    const dim3 fgrid((unsigned)((n_acc + 63) / 64));
    if (dtype == TGT_DTYPE_F32)
        hipLaunchKernelGGL((k_node_feature_finish<float>), fgrid, dim3(256), 0, st, (const float*)acc, n_atom, n_in, n_out, n_tok, copies,
                           (float*)d_datom, (float*)d_din, (float*)d_dout_table, (float*)d_dtoken);
    else
        hipLaunchKernelGGL((k_node_feature_finish<nbf16>), fgrid, dim3(256), 0, st, (const float*)acc, n_atom, n_in, n_out, n_tok, copies,
                           (nbf16*)d_datom, (nbf16*)d_din, (nbf16*)d_dout_table, (nbf16*)d_dtoken);
    TGT_HIP_CHECK(hipGetLastError());
    return TGT_OK;
}

}  // namespace
}  // namespace tgt

extern "C" {

int tgt_graph_node_feature_fwd(const int64_t* d_x, const int64_t* d_in_degree, const int64_t* d_out_degree, int Fx,
                               const void* d_atom_table, int num_atoms, const void* d_in_table, int num_in,
                               const void* d_out_table, int num_out, const void* d_graph_token, int b, int s, int C, int dtype,
                               void* d_out, void* stream) {
    using namespace tgt;
    const int rc = node_feat_check(b, s, Fx, C, num_atoms, num_in, num_out, dtype, "tgt_graph_node_feature_fwd");
    if (rc != TGT_OK) return rc;
    if (b == 0) return TGT_OK;
    if (!d_atom_table || !d_in_table || !d_out_table || !d_graph_token || !d_out || (s > 0 && (!d_x || !d_in_degree || !d_out_degree))) {
        set_error("tgt_graph_node_feature_fwd: null pointer");
        return TGT_ERR_INVALID_ARG;
    }
    NodeFeatArgs a{d_x, d_in_degree, d_out_degree, b, s, Fx, C, num_atoms, num_in, num_out, 1, 1, 1};
    return node_feature_fwd_impl(a, d_atom_table, d_in_table, d_out_table, d_graph_token, dtype, d_out, stream);
}

int64_t tgt_graph_node_feature_bwd_workspace_bytes(int num_atoms, int num_in, int num_out, int C) {
    if (num_atoms < 1 || num_in < 1 || num_out < 1 || C < 1) return 0;
    const int64_t n_acc = ((int64_t)num_atoms + num_in + num_out + 1) * C;
    return (int64_t)sizeof(float) * n_acc * tgt::node_feat_copies(n_acc);
}

int tgt_graph_node_feature_bwd(const void* d_dout, const int64_t* d_x, const int64_t* d_in_degree, const int64_t* d_out_degree,
                               int Fx, int num_atoms, int num_in, int num_out, int b, int s, int C, int dtype, void* d_datom_table,
                               void* d_din_table, void* d_dout_table, void* d_dgraph_token, void* d_workspace,
                               int64_t workspace_bytes, void* stream) {
    using namespace tgt;
    const int rc = node_feat_check(b, s, Fx, C, num_atoms, num_in, num_out, dtype, "tgt_graph_node_feature_bwd");
    if (rc != TGT_OK) return rc;
    if (!d_datom_table || !d_din_table || !d_dout_table || !d_dgraph_token ||
        (b > 0 && (!d_dout || (s > 0 && (!d_x || !d_in_degree || !d_out_degree))))) {
        set_error("tgt_graph_node_feature_bwd: null pointer");
        return TGT_ERR_INVALID_ARG;
    }
    const int64_t need = tgt_graph_node_feature_bwd_workspace_bytes(num_atoms, num_in, num_out, C);
    if (!d_workspace || workspace_bytes < need) {
        set_error("tgt_graph_node_feature_bwd: workspace of %lld bytes needed, got %lld", (long long)need, (long long)workspace_bytes);
        return TGT_ERR_WORKSPACE;
    }
    NodeFeatArgs a{d_x, d_in_degree, d_out_degree, b, s, Fx, C, num_atoms, num_in, num_out, 1, 1, 1};
    return node_feature_bwd_impl(a, d_dout, dtype, d_datom_table, d_din_table, d_dout_table, d_dgraph_token, (float*)d_workspace, stream);
}

int tgt_embedding_sum_fwd(const int64_t* d_x, int Fx, const void* d_table, int num_rows, int b, int s, int C, int dtype, void* d_out,
                          void* stream) {
    using namespace tgt;
    const int rc = node_feat_check(b, s, Fx, C, num_rows, 1, 1, dtype, "tgt_embedding_sum_fwd");
    if (rc != TGT_OK) return rc;
    if (b == 0 || s == 0) return TGT_OK;
    if (!d_table || !d_out || !d_x) {
        set_error("tgt_embedding_sum_fwd: null pointer");
        return TGT_ERR_INVALID_ARG;
    }
    NodeFeatArgs a{d_x, nullptr, nullptr, b, s, Fx, C, num_rows, 1, 1, 0, 0, 0};
    return node_feature_fwd_impl(a, d_table, nullptr, nullptr, nullptr, dtype, d_out, stream);
}

int64_t tgt_embedding_sum_bwd_workspace_bytes(int num_rows, int C) {
    if (num_rows < 1 || C < 1) return 0;
    const int64_t n_acc = (int64_t)num_rows * C;
    return (int64_t)sizeof(float) * n_acc * tgt::node_feat_copies(n_acc);
}

int tgt_embedding_sum_bwd(const void* d_dout, const int64_t* d_x, int Fx, int num_rows, int b, int s, int C, int dtype, void* d_dtable,
                          void* d_workspace, int64_t workspace_bytes, void* stream) {
    using namespace tgt;
    const int rc = node_feat_check(b, s, Fx, C, num_rows, 1, 1, dtype, "tgt_embedding_sum_bwd");
    if (rc != TGT_OK) return rc;
    if (!d_dtable || (b > 0 && s > 0 && (!d_dout || !d_x))) {
        set_error("tgt_embedding_sum_bwd: null pointer");
        return TGT_ERR_INVALID_ARG;
    }
    const int64_t need = tgt_embedding_sum_bwd_workspace_bytes(num_rows, C);
    if (!d_workspace || workspace_bytes < need) {
        set_error("tgt_embedding_sum_bwd: workspace of %lld bytes needed, got %lld", (long long)need, (long long)workspace_bytes);
        return TGT_ERR_WORKSPACE;
    }
    NodeFeatArgs a{d_x, nullptr, nullptr, b, s, Fx, C, num_rows, 1, 1, 0, 0, 0};
    return node_feature_bwd_impl(a, d_dout, dtype, d_dtable, nullptr, nullptr, nullptr, (float*)d_workspace, stream);
}

}  // extern "C"
