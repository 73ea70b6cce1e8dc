// Edge construction and ordering on the GPU: the integer side of the reference's
// batch preparation.
//
//   tgt_fix_edge_index      gt_sp/utils.py:34-50   (global node 0, edges to and from it)
//   tgt_sub_edge_index      gt_sp/utils.py:202-215 (edges among the nodes of a batch, renamed)
//   tgt_reformat_*          gt_sp/utils.py:319-359 (relabel by partition, cluster
//                           "blockize" of gt_sp/utils.py:223-305, stable sort by source)
//
// The reference does this with Python lists and per-edge appends (minutes at
// 18 M edges).  Here the per-edge work runs in kernels; the only host work is
// the k x k table of partition pairs and the block coordinates, which the
// reference draws from numpy's legacy MT19937 stream (np.random.seed(n) then
// np.random.randint) - restated below so the blocks are the same ones.
#include "common.h"
#include <vector>
#include <new>

namespace tgt {

// ---------------------------------------------------------------------------
// numpy legacy RandomState: MT19937 seeded with init_genrand, randint(0, high)
// by masked rejection on 32-bit outputs.
// ---------------------------------------------------------------------------
// A stream here is short (the blocks of one pair of partitions) and there is one per pair: state words are seeded and twisted when
// they are first needed, the same numbers as whole blocks of 624 (64 pairs: 180 us of host time with them).
class LegacyMT {
public:
    LegacyMT() = default;
    explicit LegacyMT(uint32_t s) { seed(s); }
    void seed(uint32_t s) { mt_[0] = s; }      // (of a new stream)
    uint32_t next() {
        const uint32_t UP = 0x80000000u, LO = 0x7fffffffu, MAG = 0x9908b0dfu;
        const int i = pos_, i1 = i + 1 < 624 ? i + 1 : 0, im = i + 397 < 624 ? i + 397 : i - 227;
        seeded(im > i1 ? im : i1);
        const uint32_t t = (mt_[i] & UP) | (mt_[i1] & LO);
        uint32_t y = mt_[i] = mt_[im] ^ (t >> 1) ^ ((t & 1u) ? MAG : 0u);
        pos_ = i1;
        y ^= y >> 11;
        y ^= (y << 7) & 0x9d2c5680u;
        y ^= (y << 15) & 0xefc60000u;
        y ^= y >> 18;
        return y;
    }
    // randint(0, high), high >= 1 and high - 1 < 2^32 - 1
    int64_t randint(int64_t high) {
        const uint64_t rng = (uint64_t)(high - 1);
        if (rng == 0) return 0;                       // no draw is consumed
        uint64_t mask = rng;
        mask |= mask >> 1; mask |= mask >> 2; mask |= mask >> 4; mask |= mask >> 8; mask |= mask >> 16;
        uint32_t v;
        do { v = next() & (uint32_t)mask; } while (v > rng);
        return (int64_t)v;
    }
    // The first state words of up to kTogether streams, side by side: a word is made of the one before it, so one stream waits for the
    // multiplier with every word (64 pairs of parts, 24 blocks each: 48 us of host time with the draws, 19 together).
    static constexpr int kTogether = 8;
    static void seed_together(LegacyMT* g, int n, int words) {
        uint32_t v[kTogether];
        for (int l = 0; l < kTogether; ++l) v[l] = l < n ? g[l].mt_[0] : 0u;
        words = words < 624 ? words : 624;
        for (int w = 1; w < words; ++w)
            for (int l = 0; l < kTogether; ++l) {
                v[l] = 1812433253u * (v[l] ^ (v[l] >> 30)) + (uint32_t)w;
                g[l].mt_[w] = v[l];
            }
        for (int l = 0; l < n; ++l) g[l].seeded_ = words > 1 ? words : 1;
    }
private:
    void seeded(int upto) {
        for (; seeded_ <= upto; ++seeded_) mt_[seeded_] = 1812433253u * (mt_[seeded_ - 1] ^ (mt_[seeded_ - 1] >> 30)) + (uint32_t)seeded_;
    }
    uint32_t mt_[624];
    int pos_ = 0, seeded_ = 1;
};

// ---------------------------------------------------------------------------
// kernels
// ---------------------------------------------------------------------------
__global__ void k_fix_edge_index(const int64_t* __restrict__ in, int64_t E0, int64_t n,
                                 int64_t* __restrict__ out) {
    const int64_t Eo = E0 + 2 * n;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= Eo) return;
    int64_t s, d;
    if (i < E0) { s = in[i] + 1; d = in[E0 + i] + 1; }
    else if (i < E0 + n) { s = i - E0 + 1; d = 0; }     // real node -> global node
    else { s = 0; d = i - E0 - n + 1; }                  // global node -> real node
    out[i] = s;
    out[Eo + i] = d;
}

// The lanes of a wave with the same key (key_bits of it matter) among those that take part
__device__ __forceinline__ uint64_t lanes_with(uint32_t key, int key_bits, bool in) {
    uint64_t same = __ballot(in);
    for (int b = 0; b < key_bits; ++b) {
        const bool bit = (key >> b) & 1u;
        const uint64_t bal = __ballot(bit);
        same &= bit ? bal : ~bal;
    }
    return same;
}
__device__ __forceinline__ uint64_t lower_lanes() { const int lane = threadIdx.x & 63; return lane == 0 ? 0ull : (~0ull >> (64 - lane)); }

// Range check and 32-bit ids of the parts, the counts of their first digits that the sort by part begins with (RadixSorter::Counts) and, as long
// as an id is one digit, the nodes of each part (cnt, cleared by the caller; more parts: k_count).  Neighbouring nodes are often in one part:
// equal digits of a wave are merged first.
template <int ITEMS>
__global__ __launch_bounds__(RadixSorter::kThreads) void k_check_partition(const int64_t* __restrict__ part, int64_t N, int k, uint32_t* __restrict__ p32,
                                                                           unsigned long long* __restrict__ flag, unsigned long long* __restrict__ cnt,
                                                                           const RadixSorter::Counts c) {
    constexpr int T = RadixSorter::kThreads;
    __shared__ uint32_t h[256];
    const int tid = threadIdx.x;
    h[tid] = 0;
    __syncthreads();
    const int64_t base = (int64_t)blockIdx.x * T * ITEMS + tid;
    for (int j = 0; j < ITEMS; j += 4) {
        int64_t p[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) p[u] = part[min(base + (j + u) * T, N - 1)];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int64_t i = base + (j + u) * T;
            const bool in = i < N;
            if (p[u] < 0 || p[u] >= k) {
                if (in) flag[0] = 1;
                p[u] = 0;
            }
            if (in) p32[i] = (uint32_t)p[u];
            const uint64_t same = lanes_with((uint32_t)p[u], 8, in);
            if (in && (same & lower_lanes()) == 0) atomicAdd(&h[p[u] & 255], (uint32_t)__popcll(same));
        }
    }
    __syncthreads();
    c.hist[0][(int64_t)tid * c.blocks + blockIdx.x] = h[tid];
    if (k <= 256 && h[tid]) atomicAdd(&cnt[tid], (unsigned long long)h[tid]);
}

// mapping[old] = new position; sorted[new] = old (as int64 for the caller)
__global__ void k_invert(const uint32_t* __restrict__ sorted_old, int64_t N, uint32_t* __restrict__ mapping,
                         int64_t* __restrict__ sorted_out) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    const uint32_t o = sorted_old[i];
    mapping[o] = (uint32_t)i;
    sorted_out[i] = (int64_t)o;
}

// Histogram of keys in [0, nbins).  The bins are few (k or k*k partition pairs) and neighbouring
// keys are often equal, so equal keys of a wave are first merged with ballots (one LDS add per
// distinct key and wave), workgroups count in LDS, and only non-empty bins reach global memory.
// Integer counts: the order of the additions does not matter.  keys(i, key, valid): of i, i + blockDim.x, ... (four).
constexpr int kCountLdsBins = 4096;
template <typename F> __device__ __forceinline__ void count_keys(const F& keys, int64_t n, int nbins, int key_bits, unsigned long long* __restrict__ cnt) {
    __shared__ uint32_t h[kCountLdsBins];
    const bool lds = nbins <= kCountLdsBins;
    if (lds) {
        for (int b = threadIdx.x; b < nbins; b += blockDim.x) h[b] = 0;
        __syncthreads();
    }
    const int64_t step = 4ll * gridDim.x * blockDim.x;
    const int64_t rounds = (n + step - 1) / step;          // the same for every thread: ballots need whole waves
    for (int64_t t = 0; t < rounds; ++t) {
        uint32_t key[4];
        bool valid[4];
        keys(t * step + 4ll * blockIdx.x * blockDim.x + threadIdx.x, key, valid);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const uint64_t same = lanes_with(key[u], key_bits, valid[u]);
            if (valid[u] && (same & lower_lanes()) == 0) {                    // lowest lane of its group of equal keys
                const uint32_t c = (uint32_t)__popcll(same);
                if (lds) atomicAdd(&h[key[u]], c);
                else atomicAdd(&cnt[key[u]], (unsigned long long)c);
            }
        }
    }
    if (lds) {
        __syncthreads();
        for (int b = threadIdx.x; b < nbins; b += blockDim.x)
            if (h[b]) atomicAdd(&cnt[b], (unsigned long long)h[b]);
    }
}

__global__ __launch_bounds__(256) void k_count(const uint32_t* __restrict__ keys, int64_t n, int nbins, int key_bits, unsigned long long* __restrict__ cnt) {
    count_keys([&](int64_t i, uint32_t (&key)[4], bool (&valid)[4]) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int64_t at = i + (int64_t)u * blockDim.x;
            valid[u] = at < n;
            key[u] = keys[min(at, n - 1)];
        }
    }, n, nbins, key_bits, cnt);
}
// Edges of every pair of parts (part[src] * k + part[dst]) and the range check of the endpoints (flagged, and taken as node 0).  The keys
// themselves (k_edge_keys) are written where edges are kept only: 0.39 M edges, 8 parts, the two passes 18 us with the gap between them.
__global__ __launch_bounds__(256) void k_count_pairs(const int64_t* __restrict__ src, const int64_t* __restrict__ dst, int64_t E, int64_t N, const uint32_t* __restrict__ p32,
                                                     int k, int key_bits, unsigned long long* __restrict__ cnt, unsigned long long* __restrict__ flag) {
    count_keys([&](int64_t i, uint32_t (&key)[4], bool (&valid)[4]) {
        int64_t s[4], d[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int64_t at = i + (int64_t)u * blockDim.x;
            valid[u] = at < E;
            s[u] = src[min(at, E - 1)]; d[u] = dst[min(at, E - 1)];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if ((s[u] < 0) | (s[u] >= N) | (d[u] < 0) | (d[u] >= N)) { flag[0] = 1; s[u] = 0; d[u] = 0; }
            key[u] = p32[s[u]] * (uint32_t)k + p32[d[u]];
        }
    }, E, k * k, key_bits, cnt);
}

// per-edge keys: pair = part[src]*k + part[dst], s32 = src, d32 = dst; an endpoint outside [0, N) is flagged and taken as node 0
__global__ void k_edge_keys(const int64_t* __restrict__ src, const int64_t* __restrict__ dst, int64_t E, int64_t N,
                            const uint32_t* __restrict__ p32, int k, uint32_t* __restrict__ pair,
                            uint32_t* __restrict__ s32, uint32_t* __restrict__ d32, unsigned long long* __restrict__ flag) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= E) return;
    int64_t s64 = src[i], d64 = dst[i];
    if ((s64 < 0) | (s64 >= N) | (d64 < 0) | (d64 >= N)) { flag[0] = 1; s64 = 0; d64 = 0; }
    const uint32_t s = (uint32_t)s64, d = (uint32_t)d64;
    s32[i] = s;
    d32[i] = d;
    pair[i] = p32[s] * (uint32_t)k + p32[d];
}

// out[i] = table[idx[i]]
__global__ void k_gather_u32(const uint32_t* __restrict__ table, const uint32_t* __restrict__ idx, int64_t n,
                             uint32_t* __restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = table[idx[i]];
}

// relabelled endpoints of the edges order[lo + t], t < cnt, written at out_off + t
__global__ void k_emit_raw(const uint32_t* __restrict__ order, int64_t lo, int64_t cnt,
                           const uint32_t* __restrict__ s32, const uint32_t* __restrict__ d32,
                           const uint32_t* __restrict__ mapping, int64_t out_off, uint32_t* __restrict__ ns,
                           uint32_t* __restrict__ nd) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= cnt) return;
    const uint32_t e = order ? order[lo + t] : (uint32_t)(lo + t);
    ns[out_off + t] = mapping[s32[e]];
    nd[out_off + t] = mapping[d32[e]];
}

// dense bs x bs block, pairs (a, b) row-major (gt_sp/utils.py:218-220); one workgroup per block
struct Block { int64_t off; uint32_t r0, c0; };
__global__ void k_emit_blocks(const Block* __restrict__ blocks, int bs, uint32_t* __restrict__ ns, uint32_t* __restrict__ nd) {
    const Block b = blocks[blockIdx.x];
    const int64_t off = b.off;
    const uint32_t r0 = b.r0, c0 = b.c0;
    for (int p = threadIdx.x; p < bs * bs; p += blockDim.x) {
        ns[off + p] = r0 + (uint32_t)(p / bs);
        nd[off + p] = c0 + (uint32_t)(p % bs);
    }
}

// The same where nothing but blocks is emitted (block b begins at b bs bs), in the tiles of the sort by new source, with the counts of its
// first digits (RadixSorter::Counts)
template <int ITEMS>
__global__ __launch_bounds__(RadixSorter::kThreads) void k_emit_all_blocks(const Block* __restrict__ blocks, int bs, int64_t n, uint32_t* __restrict__ ns, uint32_t* __restrict__ nd,
                                                                           const RadixSorter::Counts c) {
    constexpr int T = RadixSorter::kThreads;
    __shared__ uint32_t h[256];
    const int tid = threadIdx.x;
    h[tid] = 0;
    __syncthreads();
    const uint32_t per = (uint32_t)bs * (uint32_t)bs;
#pragma unroll 4
    for (int j = 0; j < ITEMS; ++j) {
        const uint32_t at = blockIdx.x * (uint32_t)(T * ITEMS) + j * T + tid;      // (n is below 2^31)
        if (at >= n) break;
        const Block b = blocks[at / per];
        const uint32_t p = at % per, s = b.r0 + p / (uint32_t)bs;
        ns[at] = s;
        nd[at] = b.c0 + p % (uint32_t)bs;
        atomicAdd(&h[s & 255u], 1u);
    }
    __syncthreads();
    c.hist[0][(int64_t)tid * c.blocks + blockIdx.x] = h[tid];
}

__global__ void k_write_raw(const uint32_t* __restrict__ ns, const uint32_t* __restrict__ nd, int64_t off,
                            int64_t cnt, int64_t dst_off, int64_t E_raw, int64_t* __restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= cnt) return;
    out[dst_off + i] = (int64_t)ns[off + i];
    out[E_raw + dst_off + i] = (int64_t)nd[off + i];
}

__global__ void k_write_sorted(const uint32_t* __restrict__ keys_sorted, const uint32_t* __restrict__ order,
                               const uint32_t* __restrict__ nd, int64_t n, int64_t* __restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    out[i] = (int64_t)keys_sorted[i];
    out[n + i] = (int64_t)nd[order[i]];
}

static inline unsigned nblk(int64_t n, int t = 256) { return (unsigned)((n + t - 1) / t); }

}  // namespace tgt

struct tgt_reformat {
    int64_t N = 0, E_out = 0;
    tgt::RadixSorter sorter;      // the edges sorted by new source (stable): keys and order ...
    const uint32_t *keys = nullptr, *order = nullptr;
    tgt::DevBuf nd;               // ... and the new destinations in emission order
    tgt::DevBuf mapping;          // uint32 [N], old id -> new id
    tgt::DevBuf sorted_indices;   // int64 [N], new id -> old id
    std::vector<int32_t> tiles;   // (first source, first destination) of every emitted block, emission order
    int64_t E_raw = 0;            // edges kept as they are (the sparsity > p branch, or everything if !blockize)
    tgt::DevBuf raw;              // int64 [2, E_raw], relabelled, emission order
    std::vector<tgt::Block> blocks;      // feeds an asynchronous copy, which `copied` marks the end of
    hipEvent_t copied = nullptr;
    ~tgt_reformat() {
        if (!copied) return;
        (void)hipEventSynchronize(copied);
        (void)hipEventDestroy(copied);
    }
};

namespace tgt {

static int reformat_impl(const int64_t* d_src, const int64_t* d_dst, int64_t E, int64_t N,
                         const int64_t* d_part, int k, int bs, int blockize, hipStream_t st, tgt_reformat* R) {
    R->N = N;
    DevBuf report, p32, pair, s32, d32;
    RadixSorter node_sorter;
    int rc = node_sorter.init(N, st);
    if (rc) return rc;
    const size_t eb = sizeof(uint32_t) * (size_t)(E ? E : 1);
    // flag, nodes per part, edges per pair of parts: cleared and read back in one go
    const size_t words = (1 + (size_t)k + (size_t)k * k + 1) / 2 * 2;      // (16 bytes at a time: else it takes two launches to clear them)
    TGT_HIP_CHECK(report.alloc(sizeof(unsigned long long) * words, st));
    TGT_HIP_CHECK(p32.alloc(sizeof(uint32_t) * N, st));
    TGT_HIP_CHECK(R->mapping.alloc(sizeof(uint32_t) * N, st));
    TGT_HIP_CHECK(R->sorted_indices.alloc(sizeof(int64_t) * N, st));
    const DevBuf& mapping = R->mapping;
    unsigned long long *const flag = report.as<unsigned long long>(), *const cnt_nodes = flag + 1, *const cnt_pairs = cnt_nodes + k;
    TGT_HIP_CHECK(hipMemsetAsync(report.p, 0, sizeof(unsigned long long) * words, st));
    const RadixSorter::Counts node_counts = node_sorter.counts(N, 1);
    hipLaunchKernelGGL(node_counts.items == RadixSorter::kFewItems ? &k_check_partition<RadixSorter::kFewItems> : &k_check_partition<RadixSorter::kManyItems>,
                       dim3(node_counts.blocks), dim3(RadixSorter::kThreads), 0, st, d_part, N, k, p32.as<uint32_t>(), flag, cnt_nodes, node_counts);
    const auto count_grid = [](int64_t n) { return dim3((unsigned)std::min<int64_t>(512, (n + 1023) / 1024)); };
    if (k > 256) hipLaunchKernelGGL(k_count, count_grid(N), dim3(256), 0, st, p32.as<uint32_t>(), N, k, bits_for(k), cnt_nodes);
    // the edges' keys: for those that are kept as they are
    const auto edge_keys = [&]() -> int {
        TGT_HIP_CHECK(pair.alloc(eb, st));
        TGT_HIP_CHECK(s32.alloc(eb, st));
        TGT_HIP_CHECK(d32.alloc(eb, st));
        hipLaunchKernelGGL(k_edge_keys, dim3(nblk(E)), dim3(256), 0, st, d_src, d_dst, E, N, p32.as<uint32_t>(), k,
                           pair.as<uint32_t>(), s32.as<uint32_t>(), d32.as<uint32_t>(), flag);
        return TGT_OK;
    };
    if (E > 0 && !blockize) {
        if ((rc = edge_keys()) != TGT_OK) return rc;
    } else if (E > 0) {
        hipLaunchKernelGGL(k_count_pairs, count_grid(E), dim3(256), 0, st, d_src, d_dst, E, N, p32.as<uint32_t>(), k, bits_for((int64_t)k * k), cnt_pairs, flag);
    }
    std::vector<unsigned long long> h_report(words);
    TGT_HIP_CHECK(hipMemcpyAsync(h_report.data(), report.p, sizeof(unsigned long long) * words, hipMemcpyDeviceToHost, st));
    TGT_HIP_CHECK(hipStreamSynchronize(st));
    if (h_report[0]) {
        set_error("partition id outside [0, %d) or edge endpoint outside [0, %lld)", k, (long long)N);
        return TGT_ERR_INDEX_RANGE;
    }
    const unsigned long long *const h_nodes = h_report.data() + 1, *const h_pairs = h_nodes + k;
    // relabel: parts in order, members in ascending old id (gt_sp/utils.py:329-335) = stable sort by part
    const uint32_t *ks = nullptr, *vs = nullptr;
    rc = node_sorter.sort(p32.as<uint32_t>(), nullptr, N, bits_for(k), st, &ks, &vs, true);
    if (rc) return rc;
    hipLaunchKernelGGL(k_invert, dim3(nblk(N)), dim3(256), 0, st, vs, N, R->mapping.as<uint32_t>(),
                       R->sorted_indices.as<int64_t>());

    // ---- what to emit, in the reference's order ------------------------------
    struct RawSlice { int64_t lo, cnt, out_off; };
    struct Stream { size_t block0; int i, j, n; uint32_t seed; };      // the blocks of one pair of parts, drawn from a stream of their own
    std::vector<RawSlice> raws;
    std::vector<Block>& blocks = R->blocks;
    int64_t E_out = 0;
    if (!blockize) {
        E_out = E;
    } else {
        // run lengths of equal (part_src, part_dst) in sorted order, stored COMPACTLY in the order
        // of the non-empty pairs and read back as [i*k+j] (gt_sp/utils.py:237-246,270)
        std::vector<int64_t> counts((size_t)k * k, 0), cum((size_t)k * k + 1, 0), offs(k, 0);
        size_t w = 0;
        for (size_t pq = 0; pq < (size_t)k * k; ++pq)
            if (h_pairs[pq]) counts[w++] = (int64_t)h_pairs[pq];
        for (size_t pq = 0; pq < (size_t)k * k; ++pq) cum[pq + 1] = cum[pq] + counts[pq];
        for (int i = 1; i < k; ++i) offs[i] = offs[i - 1] + (int64_t)h_nodes[i - 1];
        int64_t keep_cnt = 0;
        std::vector<Stream> streams;
        streams.reserve(std::min<size_t>((size_t)k * k, 4096));
        const double per_block = (double)bs * (double)bs;
        for (int i = 0; i < k; ++i) {
            for (int j = 0; j < k; ++j) {
                const int64_t ni = (int64_t)h_nodes[i], nj = (int64_t)h_nodes[j];
                const int64_t total = ni * nj;
                if (total == 0) {
                    set_error("partition %d or %d is empty (the reference divides by zero here)", i, j);
                    return TGT_ERR_INVALID_ARG;
                }
                const int64_t c = counts[(size_t)i * k + j];
                const double sparsity = (double)c / (double)total;
                if (sparsity > 1.0) {                       // p is hard-wired to 1 (gt_sp/utils.py:344)
                    raws.push_back(RawSlice{cum[(size_t)i * k + j], c, E_out});
                    E_out += c;
                } else {
                    const int nb = (int)(sparsity * (double)total / per_block) + 1;
                    if (ni >= bs && nj >= bs) {
                        streams.push_back(Stream{blocks.size(), i, j, nb, (uint32_t)keep_cnt});      // np.random.seed(keep_cnt)
                        for (int b = 0; b < nb; ++b) blocks.push_back(Block{E_out + (int64_t)b * bs * bs, 0, 0});
                        keep_cnt += nb;
                        E_out += (int64_t)nb * bs * bs;
                    }
                }
            }
        }
        for (size_t s0 = 0; s0 < streams.size(); s0 += LegacyMT::kTogether) {
            const int n = (int)std::min<size_t>(LegacyMT::kTogether, streams.size() - s0);
            LegacyMT rng[LegacyMT::kTogether];
            int most = 0;
            for (int l = 0; l < n; ++l) {
                rng[l].seed(streams[s0 + l].seed);
                most = std::max(most, streams[s0 + l].n);
            }
            // draw d reads words d + 1 and d + 397; two draws a block, some of them twice (what is not there yet is made when it is asked for)
            LegacyMT::seed_together(rng, n, 400 + (int)std::min<int64_t>(3ll * most, 624));
            for (int l = 0; l < n; ++l) {
                const Stream& s = streams[s0 + l];
                const int64_t rows = (int64_t)h_nodes[s.i] / bs, cols = (int64_t)h_nodes[s.j] / bs;
                for (int b = 0; b < s.n; ++b) {
                    const int64_t br = rng[l].randint(rows), bc = rng[l].randint(cols);
                    blocks[s.block0 + b].r0 = (uint32_t)(br * bs + offs[s.i]);
                    blocks[s.block0 + b].c0 = (uint32_t)(bc * bs + offs[s.j]);
                }
            }
        }
    }
    if (E_out > 0x7fff0000LL) { set_error("reordered edge list does not fit 31 bits"); return TGT_ERR_INVALID_ARG; }
    R->E_out = E_out;
    DevBuf ns, &nd = R->nd;
    TGT_HIP_CHECK(ns.alloc(sizeof(uint32_t) * (size_t)(E_out ? E_out : 1), st));
    TGT_HIP_CHECK(nd.alloc(sizeof(uint32_t) * (size_t)(E_out ? E_out : 1), st));
    RadixSorter& sorter = R->sorter;
    rc = sorter.init(E_out > E ? E_out : E, st);
    if (rc) return rc;
    bool counted = false;      // the first digits of the sort by new source

    if (!blockize) {
        if (E > 0)
            hipLaunchKernelGGL(k_emit_raw, dim3(nblk(E)), dim3(256), 0, st, (const uint32_t*)nullptr, (int64_t)0, E,
                               s32.as<uint32_t>(), d32.as<uint32_t>(), mapping.as<uint32_t>(), (int64_t)0,
                               ns.as<uint32_t>(), nd.as<uint32_t>());
    } else {
        if (!raws.empty()) {
            // edges sorted by ((part_src, part_dst), (src, dst)) (gt_sp/utils.py:230-235): LSD over
            // dst, src, pair with the stable sort
            DevBuf tmp, order;
            if (E > 0 && (rc = edge_keys()) != TGT_OK) return rc;
            TGT_HIP_CHECK(tmp.alloc(eb, st));
            TGT_HIP_CHECK(order.alloc(eb, st));
            const uint32_t *ko = nullptr, *vo = nullptr;
            rc = sorter.sort(d32.as<uint32_t>(), nullptr, E, bits_for(N), st, &ko, &vo);
            if (rc) return rc;
            hipLaunchKernelGGL(k_gather_u32, dim3(nblk(E)), dim3(256), 0, st, s32.as<uint32_t>(), vo, E,
                               tmp.as<uint32_t>());
            TGT_HIP_CHECK(hipMemcpyAsync(order.p, vo, eb, hipMemcpyDeviceToDevice, st));
            rc = sorter.sort(tmp.as<uint32_t>(), order.as<uint32_t>(), E, bits_for(N), st, &ko, &vo);
            if (rc) return rc;
            hipLaunchKernelGGL(k_gather_u32, dim3(nblk(E)), dim3(256), 0, st, pair.as<uint32_t>(), vo, E,
                               tmp.as<uint32_t>());
            TGT_HIP_CHECK(hipMemcpyAsync(order.p, vo, eb, hipMemcpyDeviceToDevice, st));
            rc = sorter.sort(tmp.as<uint32_t>(), order.as<uint32_t>(), E, bits_for((int64_t)k * k), st, &ko, &vo);
            if (rc) return rc;
            for (const RawSlice& r : raws)
                if (r.cnt > 0)
                    hipLaunchKernelGGL(k_emit_raw, dim3(nblk(r.cnt)), dim3(256), 0, st, vo, r.lo, r.cnt,
                                       s32.as<uint32_t>(), d32.as<uint32_t>(), mapping.as<uint32_t>(), r.out_off,
                                       ns.as<uint32_t>(), nd.as<uint32_t>());
        }
        if (!blocks.empty()) {
            DevBuf d_blocks;
            TGT_HIP_CHECK(d_blocks.alloc(sizeof(Block) * blocks.size(), st));
            TGT_HIP_CHECK(hipMemcpyAsync(d_blocks.p, blocks.data(), sizeof(Block) * blocks.size(), hipMemcpyHostToDevice, st));
            TGT_HIP_CHECK(hipEventCreateWithFlags(&R->copied, hipEventDisableTiming));
            TGT_HIP_CHECK(hipEventRecord(R->copied, st));
            counted = raws.empty();
            const RadixSorter::Counts c = sorter.counts(E_out, 1);
            if (counted)
                hipLaunchKernelGGL(c.items == RadixSorter::kFewItems ? &k_emit_all_blocks<RadixSorter::kFewItems> : &k_emit_all_blocks<RadixSorter::kManyItems>, dim3(c.blocks),
                                   dim3(RadixSorter::kThreads), 0, st, d_blocks.as<Block>(), bs, E_out, ns.as<uint32_t>(), nd.as<uint32_t>(), c);
            else
                hipLaunchKernelGGL(k_emit_blocks, dim3((unsigned)blocks.size()), dim3(256), 0, st, d_blocks.as<Block>(), bs, ns.as<uint32_t>(), nd.as<uint32_t>());
        }
    }
    // the blocks as a tile list and the edges kept as they are, for the block attention path
    R->tiles.reserve(2 * blocks.size());
    for (const Block& b : blocks) {
        R->tiles.push_back((int32_t)b.r0);
        R->tiles.push_back((int32_t)b.c0);
    }
    {
        int64_t e_raw = blockize ? 0 : E;
        for (const RawSlice& r : raws) e_raw += r.cnt;
        R->E_raw = e_raw;
        TGT_HIP_CHECK(R->raw.alloc(sizeof(int64_t) * 2 * (size_t)(e_raw ? e_raw : 1), st));
        if (!blockize) {
            if (E > 0)
                hipLaunchKernelGGL(k_write_raw, dim3(nblk(E)), dim3(256), 0, st, ns.as<uint32_t>(), nd.as<uint32_t>(),
                                   (int64_t)0, E, (int64_t)0, e_raw, R->raw.as<int64_t>());
        } else {
            int64_t pos = 0;
            for (const RawSlice& r : raws) {
                if (r.cnt > 0)
                    hipLaunchKernelGGL(k_write_raw, dim3(nblk(r.cnt)), dim3(256), 0, st, ns.as<uint32_t>(),
                                       nd.as<uint32_t>(), r.out_off, r.cnt, pos, e_raw, R->raw.as<int64_t>());
                pos += r.cnt;
            }
        }
    }
    // stable sort by new source (gt_sp/utils.py:354-356)
    if (E_out > 0) {
        rc = sorter.sort(ns.as<uint32_t>(), nullptr, E_out, bits_for(N), st, &R->keys, &R->order, counted);
        if (rc) return rc;
    }
    TGT_HIP_CHECK(hipGetLastError());
    return TGT_OK;
}

// The batch node behind every row of the reordered batch: idx[old id], without the `tokens` global nodes in front of the old ids
// (at most one: the first member of its part, wherever that part lies)
__global__ void k_batch_rows(const int64_t* __restrict__ sorted, int64_t N, const uint32_t* __restrict__ mapping, const int64_t* __restrict__ idx, int tokens,
                             int64_t* __restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    const int64_t token = tokens ? (int64_t)mapping[0] : N;      // the global node's new place
    if (i != token) out[i > token ? i - 1 : i] = idx[sorted[i] - tokens];
}

// ---------------------------------------------------------------------------
// Sub-graph of a node batch (gen_sub_edge_index, gt_sp/utils.py:202-215): the
// sequence of torch_geometric 2.0.0 calls
//   remove_self_loops(edge_index)              keep edges with src != dst, in order
//   add_self_loops(.., num_nodes=N)            append (i, i) for i = 0..N-1
//   subgraph(idx_batch, .., relabel_nodes=True, num_nodes=N)
//                                              keep edges with both ends in the batch, in
//                                              order, and rename node idx_batch[p] to p
// as one order-preserving compaction over the E edges followed by the N
// self-loops.  A node that occurs more than once in idx_batch takes its LAST
// position (what the sequential index assignment n_idx[subset] = arange gives).
// ---------------------------------------------------------------------------
constexpr int kSubItems = 1024;     // items of a tile of the compaction

__global__ void k_sub_fill(int32_t* __restrict__ pos, int64_t N, uint32_t* __restrict__ member, int64_t words, int* __restrict__ bad) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0) *bad = 0;
    if (i < N) pos[i] = -1;
    if (i < words) member[i] = 0;
}

// member: one bit per node of the batch
__global__ void k_sub_positions(const int64_t* __restrict__ idx, int64_t S, int64_t N, int32_t* __restrict__ pos,
                                uint32_t* __restrict__ member, int* __restrict__ bad) {
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= S) return;
    const int64_t v = idx[p];
    if (v < 0 || v >= N) { atomicOr(bad, 1); return; }
    atomicMax(&pos[v], (int32_t)p);
    atomicOr(&member[v >> 5], 1u << (v & 31));
}

// The endpoints of item i (< E: edge i; E + v: the self-loop of node v).  An index past the end reads the last item's.
__device__ __forceinline__ void sub_ends(const int64_t* __restrict__ ei, int64_t E, int64_t total, int64_t i, int64_t& s, int64_t& d) {
    i = min(i, total - 1);
    const bool edge = i < E;
    const int64_t at = edge ? i : 0;
    if (E > 0) { s = ei[at]; d = ei[E + at]; }
    if (!edge) s = d = i - E;
}

// First pass: the kept items of every tile of kSubItems, as one bit per item and their number.  A wave takes a tile.  Two look-ups in a random place
// for every edge are what this pass waits for when they go to the position table (a request to L2 per lane: 35 us for 3.1 M edges and
// 256 K nodes, whose 16 bytes per edge take 10); whether a node is in the batch is one bit, and the bits of up to 1 M nodes stay in a
// CU's LDS (IN_LDS): 15 us.  The loads of eight rounds go out before the first is used.
constexpr int kSubWords = kSubItems / 64, kSubRounds = 8, kSubWaves = 16;
template <bool IN_LDS>
__global__ __launch_bounds__(64 * kSubWaves) void k_sub_mark(const int64_t* __restrict__ ei, int64_t E, int64_t N, const uint32_t* __restrict__ member,
                                                             int words, int tiles, uint32_t* __restrict__ counts, uint64_t* __restrict__ keep_bits,
                                                             int* __restrict__ bad) {
    extern __shared__ __align__(16) uint32_t in_lds[];
    if (IN_LDS) {
        for (int i = threadIdx.x; i < words / 4; i += 64 * kSubWaves) reinterpret_cast<uint4*>(in_lds)[i] = reinterpret_cast<const uint4*>(member)[i];
        __syncthreads();
    }
    const uint32_t* bits = IN_LDS ? in_lds : member;
    const int lane = threadIdx.x & 63;
    const int64_t total = E + N;
    for (int tile = blockIdx.x * kSubWaves + (threadIdx.x >> 6); tile < tiles; tile += gridDim.x * kSubWaves) {
        uint64_t mine = 0;      // lane w: word w
        uint32_t kept = 0;
#pragma unroll 1
        for (int r0 = 0; r0 < kSubWords; r0 += kSubRounds) {
            const int64_t i0 = (int64_t)tile * kSubItems + r0 * 64 + lane;
            int64_t s[kSubRounds], d[kSubRounds];
#pragma unroll
            for (int r = 0; r < kSubRounds; ++r) sub_ends(ei, E, total, i0 + r * 64, s[r], d[r]);
#pragma unroll
            for (int r = 0; r < kSubRounds; ++r) {
                const int64_t i = i0 + r * 64;
                const bool in = s[r] >= 0 && s[r] < N && d[r] >= 0 && d[r] < N;
                if (!in && i < E) atomicOr(bad, 2);
                const uint32_t a = bits[in ? s[r] >> 5 : 0] >> (s[r] & 31), b = bits[in ? d[r] >> 5 : 0] >> (d[r] & 31);
                const uint64_t m = __ballot(in && i < total && (a & b & 1u) && (i >= E || s[r] != d[r]));
                mine = lane == r0 + r ? m : mine;
                kept += (uint32_t)__popcll(m);
            }
        }
        if (lane < kSubWords) keep_bits[(int64_t)tile * kSubWords + lane] = mine;
        if (lane == 0) counts[tile] = kept;
    }
}

// Second pass: the kept items in item order, behind the tile's offset.  Every wave of a tile's workgroup reads all of its words, a lane each,
// whose prefix is where a word's items go; only kept items look at their endpoints and positions.
__global__ __launch_bounds__(256) void k_sub_write(const int64_t* __restrict__ ei, int64_t E, int64_t N, const int32_t* __restrict__ pos,
                                                   const uint32_t* __restrict__ offsets, const uint64_t* __restrict__ keep_bits,
                                                   int64_t* __restrict__ out, int64_t capacity) {
    constexpr int kRounds = kSubWords / 4;      // words of a wave: wave, 4 + wave, ...
    static_assert(kSubWords % 4 == 0 && kSubWords <= 64, "a lane per word");
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t total = E + N, item0 = (int64_t)blockIdx.x * kSubItems + threadIdx.x;
    const uint64_t mine = lane < kSubWords ? keep_bits[(int64_t)blockIdx.x * kSubWords + lane] : 0ull;
    const uint32_t n = (uint32_t)__popcll(mine);
    uint32_t before = n;      // kept items up to this lane's word
#pragma unroll
    for (int off = 1; off < kSubWords; off <<= 1) {
        const uint32_t x = __shfl_up(before, off);
        if (lane >= off) before += x;
    }
    before += offsets[blockIdx.x] - n;
    int64_t s[kRounds], d[kRounds];
    uint64_t m[kRounds];
#pragma unroll
    for (int r = 0; r < kRounds; ++r) {
        m[r] = __shfl(mine, 4 * r + wave);
        s[r] = d[r] = -1;
        if ((m[r] >> lane) & 1ull) sub_ends(ei, E, total, item0 + r * 256, s[r], d[r]);
    }
#pragma unroll
    for (int r = 0; r < kRounds; ++r) {
        const uint32_t first = __shfl(before, 4 * r + wave);
        if (s[r] >= 0) {
            const int64_t o = (int64_t)first + __popcll(m[r] & ((1ull << lane) - 1ull));
            out[o] = pos[s[r]];
            out[capacity + o] = pos[d[r]];
        }
    }
}

// exclusive prefix of the workgroup counts in place (one workgroup), total to counts[n]
__global__ __launch_bounds__(256) void k_sub_scan(uint32_t* __restrict__ counts, int n) {
    __shared__ uint32_t part[256];
    const int tid = threadIdx.x;
    const int chunk = (n + 255) / 256;
    const int b = min(tid * chunk, n), e = min(b + chunk, n);
    uint32_t sum = 0;
    for (int i = b; i < e; ++i) sum += counts[i];
    part[tid] = sum;
    __syncthreads();
    for (int off = 1; off < 256; off <<= 1) {
        const uint32_t x = tid >= off ? part[tid - off] : 0u;
        __syncthreads();
        part[tid] += x;
        __syncthreads();
    }
    uint32_t run = tid ? part[tid - 1] : 0u;
    for (int i = b; i < e; ++i) {
        const uint32_t x = counts[i];
        counts[i] = run;
        run += x;
    }
    if (tid == 255) counts[n] = part[255];
}

static int sub_edge_index_impl(const int64_t* d_ei, int64_t E, int64_t N, const int64_t* d_idx, int64_t S,
                               int64_t* d_out, int64_t capacity, bool packed, int64_t* h_num, hipStream_t st) {
    const int64_t total = E + N;
    const int nblocks = (int)((total + kSubItems - 1) / kSubItems);
    const int64_t words = (N + 127) / 128 * 4;      // of the members' bits, in whole vectors
    DevBuf pos, counts, bits, member;      // counts: per tile, their total, the error flag
    TGT_HIP_CHECK(pos.alloc(sizeof(int32_t) * (size_t)N, st));
    TGT_HIP_CHECK(counts.alloc(sizeof(uint32_t) * (size_t)(nblocks + 2), st));
    TGT_HIP_CHECK(bits.alloc(sizeof(uint64_t) * (size_t)nblocks * kSubWords, st));
    TGT_HIP_CHECK(member.alloc(sizeof(uint32_t) * (size_t)words, st));
    int* const bad = counts.as<int>() + nblocks + 1;
    hipLaunchKernelGGL(k_sub_fill, dim3(nblk(std::max(N, words))), dim3(256), 0, st, pos.as<int32_t>(), N, member.as<uint32_t>(), words, bad);
    if (S > 0)
        hipLaunchKernelGGL(k_sub_positions, dim3(nblk(S)), dim3(256), 0, st, d_idx, S, N, pos.as<int32_t>(),
                           member.as<uint32_t>(), bad);
    {
        // a workgroup per CU; with the bits elsewhere (more than 1 M nodes) twice as many waves cover the requests
        constexpr int kMost = 128 << 10;
        const bool in_lds = words * (int64_t)sizeof(uint32_t) <= kMost;
        const int grid = (int)std::min<int64_t>((int64_t)num_cus() * (in_lds ? 1 : 2), (nblocks + kSubWaves - 1) / kSubWaves);
        static std::atomic<uint64_t> done;
        const auto run = [&](auto kernel, int lds) {
            hipLaunchKernelGGL(kernel, dim3(grid), dim3(64 * kSubWaves), lds, st, d_ei, E, N, (const uint32_t*)member.as<uint32_t>(), (int)words, nblocks,
                               counts.as<uint32_t>(), bits.as<uint64_t>(), bad);
        };
        if (in_lds) {
            if (int rc = allow_lds(reinterpret_cast<const void*>(&k_sub_mark<true>), kMost, done)) return rc;
            run(&k_sub_mark<true>, (int)(words * sizeof(uint32_t)));
        } else run(&k_sub_mark<false>, 0);
    }
    hipLaunchKernelGGL(k_sub_scan, dim3(1), dim3(256), 0, st, counts.as<uint32_t>(), nblocks);
    TGT_HIP_CHECK(hipGetLastError());
    uint32_t back[2] = {0, 0};
    TGT_HIP_CHECK(hipMemcpyAsync(back, counts.as<uint32_t>() + nblocks, sizeof(back), hipMemcpyDeviceToHost, st));
    TGT_HIP_CHECK(hipStreamSynchronize(st));
    const uint32_t n_keep = back[0], h_bad = back[1];
    if (h_bad) {
        set_error("tgt_sub_edge_index: %s outside [0, %lld)", (h_bad & 1) ? "a batch node id is" : "an edge endpoint is",
                  (long long)N);
        return TGT_ERR_INDEX_RANGE;
    }
    *h_num = (int64_t)n_keep;
    if ((int64_t)n_keep > capacity) {
        set_error("tgt_sub_edge_index: %lld edges kept, room for %lld", (long long)n_keep, (long long)capacity);
        return TGT_ERR_WORKSPACE;
    }
    if (n_keep > 0) {
        hipLaunchKernelGGL(k_sub_write, dim3(nblocks), dim3(256), 0, st, d_ei, E, N, pos.as<int32_t>(),
                           counts.as<uint32_t>(), bits.as<uint64_t>(), d_out, packed ? (int64_t)n_keep : capacity);
        TGT_HIP_CHECK(hipGetLastError());
    }
    return TGT_OK;
}

}  // namespace tgt

extern "C" {

int tgt_fix_edge_index(const int64_t* d_edge_index, int64_t E0, int64_t num_node, int64_t* d_out, void* stream) {
    if (E0 < 0 || num_node < 0 || !d_out || (E0 > 0 && !d_edge_index)) {
        tgt::set_error("tgt_fix_edge_index: null pointer or negative size");
        return TGT_ERR_INVALID_ARG;
    }
    const int64_t Eo = E0 + 2 * num_node;
    if (Eo == 0) return TGT_OK;
    hipLaunchKernelGGL(tgt::k_fix_edge_index, dim3(tgt::nblk(Eo)), dim3(256), 0, (hipStream_t)stream, d_edge_index,
                       E0, num_node, d_out);
    TGT_HIP_CHECK(hipGetLastError());
    return TGT_OK;
}

static int sub_edge_index_entry(const int64_t* d_edge_index, int64_t E, int64_t N, const int64_t* d_idx_batch, int64_t S, int64_t* d_out, int64_t capacity, bool packed,
                                int64_t* h_num_edges, void* stream) {
    if (E < 0 || N < 1 || S < 0 || capacity < 0 || !h_num_edges || (E > 0 && !d_edge_index) || (S > 0 && !d_idx_batch) ||
        (capacity > 0 && !d_out)) {
        tgt::set_error("tgt_sub_edge_index: null pointer or bad size");
        return TGT_ERR_INVALID_ARG;
    }
    if (E > 0x7fff0000LL || N > 0x7fff0000LL || S > 0x7fff0000LL) {
        tgt::set_error("tgt_sub_edge_index: E, N and the batch size must fit 31 bits");
        return TGT_ERR_INVALID_ARG;
    }
    return tgt::sub_edge_index_impl(d_edge_index, E, N, d_idx_batch, S, d_out, capacity, packed, h_num_edges,
                                    (hipStream_t)stream);
}

int tgt_sub_edge_index(const int64_t* d_edge_index, int64_t E, int64_t N, const int64_t* d_idx_batch, int64_t S,
                       int64_t* d_out, int64_t capacity, int64_t* h_num_edges, void* stream) {
    return sub_edge_index_entry(d_edge_index, E, N, d_idx_batch, S, d_out, capacity, false, h_num_edges, stream);
}
int tgt_sub_edge_index_packed(const int64_t* d_edge_index, int64_t E, int64_t N, const int64_t* d_idx_batch, int64_t S,
                              int64_t* d_out, int64_t capacity, int64_t* h_num_edges, void* stream) {
    return sub_edge_index_entry(d_edge_index, E, N, d_idx_batch, S, d_out, capacity, true, h_num_edges, stream);
}

int tgt_np_legacy_randint(uint32_t seed, const int64_t* h_highs, int n, int64_t* h_out) {
    if (n < 0 || (n > 0 && (!h_highs || !h_out))) return TGT_ERR_INVALID_ARG;
    tgt::LegacyMT rng(seed);
    for (int i = 0; i < n; ++i) {
        if (h_highs[i] < 1 || h_highs[i] > 0xffffffffLL) return TGT_ERR_INVALID_ARG;
        h_out[i] = rng.randint(h_highs[i]);
    }
    return TGT_OK;
}

int tgt_reformat_create(const int64_t* d_src, const int64_t* d_dst, int64_t E, int64_t N,
                        const int64_t* d_partition_ids, int k, int block_size, int blockize, void* stream,
                        tgt_reformat_t** out) {
    if (!out || E < 0 || N < 1 || k < 1 || k > 4096 || block_size < 1 || !d_partition_ids ||
        (E > 0 && (!d_src || !d_dst))) {
        tgt::set_error("tgt_reformat_create: bad argument");
        return TGT_ERR_INVALID_ARG;
    }
    if (E > 0x7fff0000LL || N > 0x7fff0000LL) {
        tgt::set_error("tgt_reformat_create: E and N must fit 31 bits");
        return TGT_ERR_INVALID_ARG;
    }
    tgt_reformat* R = new (std::nothrow) tgt_reformat();
    if (!R) return TGT_ERR_INVALID_ARG;
    const int rc = tgt::reformat_impl(d_src, d_dst, E, N, d_partition_ids, k, block_size, blockize,
                                      (hipStream_t)stream, R);
    if (rc != TGT_OK) { delete R; return rc; }
    *out = R;
    return TGT_OK;
}

int64_t tgt_reformat_num_edges(const tgt_reformat_t* r) { return r ? r->E_out : -1; }

int tgt_reformat_export_edges(const tgt_reformat_t* r, int64_t* d_edge_index, void* stream) {
    if (!r || (r->E_out > 0 && !d_edge_index)) {
        tgt::set_error("tgt_reformat_export_edges: null pointer");
        return TGT_ERR_INVALID_ARG;
    }
    if (r->E_out > 0)
        hipLaunchKernelGGL(tgt::k_write_sorted, dim3(tgt::nblk(r->E_out)), dim3(256), 0, (hipStream_t)stream, r->keys, r->order, r->nd.as<uint32_t>(), r->E_out, d_edge_index);
    TGT_HIP_CHECK(hipGetLastError());
    return TGT_OK;
}

int tgt_reformat_export(const tgt_reformat_t* r, int64_t* d_edge_index, int64_t* d_sorted_indices, void* stream) {
    if (!r || !d_sorted_indices || (r->E_out > 0 && !d_edge_index)) {
        tgt::set_error("tgt_reformat_export: null pointer");
        return TGT_ERR_INVALID_ARG;
    }
    if (int rc = tgt_reformat_export_edges(r, d_edge_index, stream)) return rc;
    TGT_HIP_CHECK(hipMemcpyAsync(d_sorted_indices, r->sorted_indices.p, sizeof(int64_t) * r->N,
                                 hipMemcpyDeviceToDevice, (hipStream_t)stream));
    return TGT_OK;
}

int tgt_reformat_rows(const tgt_reformat_t* r, const int64_t* d_idx_batch, int tokens, int64_t* d_rows, void* stream) {
    if (!r || tokens < 0 || tokens > 1 || (r->N > tokens && (!d_idx_batch || !d_rows))) {
        tgt::set_error("tgt_reformat_rows: null pointer, or tokens not 0 or 1");
        return TGT_ERR_INVALID_ARG;
    }
    hipLaunchKernelGGL(tgt::k_batch_rows, dim3(tgt::nblk(r->N)), dim3(256), 0, (hipStream_t)stream, r->sorted_indices.as<int64_t>(), r->N, r->mapping.as<uint32_t>(),
                       d_idx_batch, tokens, d_rows);
    TGT_HIP_CHECK(hipGetLastError());
    return TGT_OK;
}

int64_t tgt_reformat_num_tiles(const tgt_reformat_t* r) { return r ? (int64_t)(r->tiles.size() / 2) : -1; }
int64_t tgt_reformat_num_raw_edges(const tgt_reformat_t* r) { return r ? r->E_raw : -1; }

int tgt_reformat_export_tiles(const tgt_reformat_t* r, int32_t* h_tiles, int64_t* d_raw_edge_index, void* stream) {
    if (!r || (!r->tiles.empty() && !h_tiles) || (r->E_raw > 0 && !d_raw_edge_index)) {
        tgt::set_error("tgt_reformat_export_tiles: null pointer");
        return TGT_ERR_INVALID_ARG;
    }
    for (size_t i = 0; i < r->tiles.size(); ++i) h_tiles[i] = r->tiles[i];
    if (r->E_raw > 0)
        TGT_HIP_CHECK(hipMemcpyAsync(d_raw_edge_index, r->raw.p, sizeof(int64_t) * 2 * r->E_raw,
                                     hipMemcpyDeviceToDevice, (hipStream_t)stream));
    return TGT_OK;
}

int tgt_reformat_destroy(tgt_reformat_t* r) {
    delete r;
    return TGT_OK;
}

}  // extern "C"
