// Graph plan: stable CSR-by-destination / CSC-by-source build and the
// degree-binned row schedule.
//
// Replaces, once per edge_index, what the reference redoes on every attention
// call: the per-edge gathers k[edge_index[0]], q[edge_index[1]] and the atomic
// scatter-adds over edge_index[1] (attn_module.py:146-147,180,185).  The sorted
// order is the stable one (ties keep the caller's edge order), the contract of
// the reference's edge sort (gt_sp/utils.py:354-356).
//
// The sort is a hand-written LSD radix sort (8-bit digits) whose ranking is
// position-based, so the result is bit-reproducible: integer LDS counters only
// count, they never decide an order.
#include "common.h"
#include <vector>
#include <new>
#include <mutex>
#include <utility>
#include <algorithm>
#include <stdlib.h>
#include <string.h>

namespace tgt {

static thread_local char g_err[512] = "";
void set_error(const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
}
const char* last_error() { return g_err; }

// ---------------------------------------------------------------------------
// kernels
// ---------------------------------------------------------------------------
// int64 endpoints -> uint32, with a range check (flag[0] = 1 on a bad index), and the counts of their first digits that both sorts begin
// with (RadixSorter::Counts: destinations, sources): a launch and a pass over the keys less.
template <int ITEMS>
__global__ __launch_bounds__(RadixSorter::kThreads) void k_convert_validate(const int64_t* __restrict__ src, const int64_t* __restrict__ dst, int64_t E, int64_t N,
                                                                            uint32_t* __restrict__ s32, uint32_t* __restrict__ d32, int* __restrict__ flag,
                                                                            const RadixSorter::Counts c) {
    constexpr int T = RadixSorter::kThreads;
    __shared__ uint32_t h[2][256];
    const int tid = threadIdx.x;
    h[0][tid] = h[1][tid] = 0;
    __syncthreads();
    const int64_t base = (int64_t)blockIdx.x * T * ITEMS + tid;
    for (int j = 0; j < ITEMS; j += 4) {
        int64_t s[4], d[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int64_t i = min(base + (j + u) * T, E - 1);
            s[u] = src[i]; d[u] = dst[i];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int64_t i = base + (j + u) * T;
            if (i >= E) continue;
            const bool bad = (s[u] < 0) | (s[u] >= N) | (d[u] < 0) | (d[u] >= N);
            if (bad) { flag[0] = 1; s[u] = 0; d[u] = 0; }
            s32[i] = (uint32_t)s[u];
            d32[i] = (uint32_t)d[u];
            atomicAdd(&h[0][d[u] & 255], 1u);      // (integer counts: order-free)
            atomicAdd(&h[1][s[u] & 255], 1u);
        }
    }
    __syncthreads();
#pragma unroll
    for (int v = 0; v < 2; ++v) c.hist[v][(int64_t)tid * c.blocks + blockIdx.x] = h[v][tid];
}

// The two views are made by the same launches (blockIdx.y: by destination, by source): a batch's edge list does not fill the
// chip with one of them, and a launch costs as much host time as such a kernel runs.
struct SideArrays {
    const uint32_t *keys[2], *order[2], *other[2];      // sorted keys, edge of a sorted position, the edges' other endpoints
    int32_t *rowptr[2], *col[2], *eid[2];
};

// rowptr[r] = first sorted position whose key is >= r (r = 0 .. N): one thread per row, binary
// search in the sorted keys (a thread per position walking the gap to the next key would leave
// all the work to one thread when the keys are few or far apart).
// The workgroups behind the first row_blocks: the endpoint and edge id of every sorted position, beside it.
__global__ __launch_bounds__(256) void k_fill_rowptr_and_col(const SideArrays a, int64_t E, int64_t N, int row_blocks) {
    if ((int)blockIdx.x >= row_blocks) {
        const uint32_t *__restrict__ eid = a.order[blockIdx.y], *__restrict__ other = a.other[blockIdx.y];
        const int64_t pos = (int64_t)(blockIdx.x - row_blocks) * blockDim.x + threadIdx.x;
        if (pos >= E) return;
        const uint32_t e = eid[pos];
        a.col[blockIdx.y][pos] = (int32_t)other[e];
        a.eid[blockIdx.y][pos] = (int32_t)e;
        return;
    }
    const uint32_t* __restrict__ keys = a.keys[blockIdx.y];
    int32_t* __restrict__ rowptr = a.rowptr[blockIdx.y];
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r > N) return;
    int64_t lo = 0, hi = E;            // answer in [lo, hi]
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if ((int64_t)keys[mid] < r) lo = mid + 1;
        else hi = mid;
    }
    rowptr[r] = (int32_t)lo;
}

// ---------------------------------------------------------------------------
// schedule kernels: rows are binned on the device, window by window; only per-window counts and the
// few long rows visit the host
// ---------------------------------------------------------------------------
constexpr int kSchedCats = kNumClass + 1;   // the wave classes, then "longer than a wave row"
constexpr int kSchedMaxWaves = 16;          // a window is one workgroup of up to 1024 threads, one per row

// skip_empty: rows without edges get no place in the schedule (-1)
__device__ __forceinline__ int sched_category(int len, int wave_row_max, bool skip_empty) {
    if (skip_empty && len == 0) return -1;
    if (len > wave_row_max) return kNumClass;
    if (len > 32) return 0;
    if (len > 16) return 1;
    if (len > 8) return 2;
    if (len > 4) return 3;
    return 4;
}

// Per side, written by the device and read back once: how many of everything the schedule holds.
// looked, near: rows whose middle edge was looked at, and those of them whose other endpoint is within kNearRows.
struct SchedHeader { int32_t n_wave, n_long, n_block, n_split, n_parts, n_groups, looked, near; };
// Whether the neighbours of most rows are near enough to meet in an XCD's L2: the graph is clustered or reordered, or small.  The rows are
// then sorted by length, for the backward's list with kind 6 (want_groups in sparse_attn.hip).  Without it the gathers are bound by the
// traffic behind the L2s and a row's own data, gathered by its self-loop and loaded by both views, should stay close in time: 64 K
// nodes without clusters, 0.5 M edges, bf16 35.4 us by classes, 38.4 as kind 6; 262 K nodes, 8.6 M edges 550 / 566.  From 16 000 rows on
// (8000 nodes, 0.26 M edges 17.6 / 18.7), and with ten edges a row unless rows are many (64 K nodes in 64 clusters, 0.5 M edges 32.4 / 33.5, 150 K nodes, 1.2 M edges 68.9 / 67.2).
constexpr int kNearRows = 8192, kNearWindows = 8;      // (every eighth window is asked)
constexpr int64_t kManyRows = 128 << 10, kDenseRows = 10;
static bool may_group(int64_t N, int64_t E) { return N >= 16000 && (E >= kDenseRows * N || N >= kManyRows); }
__host__ __device__ inline bool mostly_near(const SchedHeader& h) { return h.looked > 0 && 2 * (int64_t)h.near >= h.looked; }
struct BlockMeta;
// What the schedule kernels read and write, of both views (blockIdx.y)
struct SchedArgs {
    const int32_t *rowptr[2], *col[2];
    uint32_t *counts[2], *offs[2];
    SchedHeader* hdr[2];
    Item *items[2], *block_items[2];
    int32_t *long_rows[2], *row_item_off[2], *row_split_idx[2], *row_part_off[2], *split_row[2], *split_off[2], *split_grp[2], *part2split[2];
    BlockMeta* meta[2];
};

// How far the edges of every eighth window lead, for mostly_near: a row's middle edge stands for it.
__global__ __launch_bounds__(kWindowRows) void k_look_near(const SideArrays a, SchedHeader* hdr, int64_t N) {
    const int64_t r = (int64_t)blockIdx.x * kNearWindows * kWindowRows + threadIdx.x;
    const int32_t* __restrict__ rowptr = a.rowptr[blockIdx.y];
    const int start = r < N ? rowptr[r] : 0, len = r < N ? rowptr[r + 1] - start : 0;
    const bool asked = len >= kGroupRowMin;
    const bool is_near = asked && llabs((int64_t)a.col[blockIdx.y][start + len / 2] - r) <= kNearRows;
    const uint64_t ba = __ballot(asked), bn = __ballot(is_near);
    if ((threadIdx.x & 63) == 0 && ba) {      // (integer counts: order-free)
        atomicAdd(&hdr[blockIdx.y].looked, (int32_t)__popcll(ba));
        atomicAdd(&hdr[blockIdx.y].near, (int32_t)__popcll(bn));
    }
}

// counts[window * kSchedCats + cat] = rows of that category among the window's rows (blockDim.x rows).
__global__ void k_sched_count(const SchedArgs a, int64_t N, int wave_row_max, bool skip_empty) {
    const int32_t* __restrict__ rowptr = a.rowptr[blockIdx.y];
    uint32_t* __restrict__ counts = a.counts[blockIdx.y];
    __shared__ uint32_t c[kSchedCats];
    if (threadIdx.x < kSchedCats) c[threadIdx.x] = 0;
    __syncthreads();
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int cat = r < N ? sched_category(rowptr[r + 1] - rowptr[r], wave_row_max, skip_empty) : -1;
#pragma unroll
    for (int k = 0; k < kSchedCats; ++k) {
        const uint64_t b = __ballot(cat == k);
        if ((threadIdx.x & 63) == 0 && b) atomicAdd(&c[k], (uint32_t)__popcll(b));   // integer count: order-free
    }
    __syncthreads();
    if (threadIdx.x < kSchedCats) counts[(int64_t)blockIdx.x * kSchedCats + threadIdx.x] = c[threadIdx.x];
}

// offs[window, cat]: first position of the window's rows of a category - wave classes count through
// (window, class) in that order, long rows through the windows - and the two totals.  One workgroup per view.
__global__ __launch_bounds__(1024) void k_sched_scan(const SchedArgs a, int nwin) {
    const uint32_t* __restrict__ counts = a.counts[blockIdx.y];
    uint32_t* __restrict__ offs = a.offs[blockIdx.y];
    SchedHeader* __restrict__ hdr = a.hdr[blockIdx.y];
    __shared__ uint32_t sw[1024], sl[1024];
    const int tid = threadIdx.x;
    const int chunk = (nwin + 1023) / 1024;
    const int b = min(tid * chunk, nwin), e = min(b + chunk, nwin);
    uint32_t ws = 0, ls = 0;
    for (int w = b; w < e; ++w) {
        for (int c = 0; c < kNumClass; ++c) ws += counts[(int64_t)w * kSchedCats + c];
        ls += counts[(int64_t)w * kSchedCats + kNumClass];
    }
    sw[tid] = ws; sl[tid] = ls;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {
        const uint32_t x = tid >= off ? sw[tid - off] : 0u, y = tid >= off ? sl[tid - off] : 0u;
        __syncthreads();
        sw[tid] += x; sl[tid] += y;
        __syncthreads();
    }
    uint32_t rw = tid ? sw[tid - 1] : 0u, rl = tid ? sl[tid - 1] : 0u;
    for (int w = b; w < e; ++w) {
        for (int c = 0; c < kNumClass; ++c) { offs[(int64_t)w * kSchedCats + c] = rw; rw += counts[(int64_t)w * kSchedCats + c]; }
        offs[(int64_t)w * kSchedCats + kNumClass] = rl;
        rl += counts[(int64_t)w * kSchedCats + kNumClass];
    }
    if (tid == 1023) { hdr->n_wave = (int32_t)sw[1023]; hdr->n_long = (int32_t)sl[1023]; }
}

// Order of the rows of a category by length, longest first, in steps of the kernels' loops: four edges for rows that one lane group walks,
// sixteen for those of a whole wave.  Waves of a workgroup, and rows of a wave, then end together.
constexpr int kLongBin = 16, kLongBins = (kWaveRowMax - kGroupRowMax - 1) / kLongBin + 1, kGroupBin = 4;
constexpr int kSortBins = kLongBins + 6;
__device__ __forceinline__ int sort_bin(int len, int cat) {
    return cat == 0 ? max(kWaveRowMax - len, 0) / kLongBin : (cat == 1 ? kLongBins + (32 - len) / kGroupBin : (cat == 2 ? kLongBins + 4 + (16 - len) / kGroupBin : -1));
}

// Rows keep their order inside a (window, category): position = offs[window, cat] + rank among the
// window's rows - behind their order by length where neighbours are near.  Wave-class rows become wave items at items[position]; long rows are listed (row, first
// edge, length) for the kernels that cut them into workgroup items.
__global__ void k_sched_fill(const SchedArgs a, int64_t N, int wave_row_max, bool skip_empty, int64_t cap_long) {
    const bool by_length = mostly_near(*a.hdr[blockIdx.y]);
    const int32_t* __restrict__ rowptr = a.rowptr[blockIdx.y];
    const uint32_t* __restrict__ offs = a.offs[blockIdx.y];
    Item* __restrict__ items = a.items[blockIdx.y];
    int32_t* __restrict__ long_rows = a.long_rows[blockIdx.y];
    __shared__ uint32_t wave_cnt[kSchedMaxWaves][kSchedCats];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int start = 0, len = 0, cat = -1;
    if (r < N) {
        start = rowptr[r];
        len = rowptr[r + 1] - start;
        cat = sched_category(len, wave_row_max, skip_empty);
    }
    const uint64_t lower = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    uint32_t rank = 0;
#pragma unroll
    for (int k = 0; k < kSchedCats; ++k) {
        const uint64_t b = __ballot(cat == k);
        if (cat == k) rank = (uint32_t)__popcll(b & lower);
        if (lane == 0) wave_cnt[wave][k] = (uint32_t)__popcll(b);
    }
    __shared__ uint32_t wave_bin[kSchedMaxWaves][kSortBins];
    const int bin = by_length ? sort_bin(len, cat) : -1, bin0 = cat == 0 ? 0 : (cat == 1 ? kLongBins : kLongBins + 4);
    if (by_length) {
        if (bin >= 0) rank = 0;
        for (int k = 0; k < kSortBins; ++k) {
            const uint64_t b = __ballot(bin == k);
            if (bin == k) rank += (uint32_t)__popcll(b & lower);
            else if (bin > k && k >= bin0) rank += (uint32_t)__popcll(b);
            if (lane == 0) wave_bin[wave][k] = (uint32_t)__popcll(b);
        }
    }
    __syncthreads();
    if (cat < 0) return;
    uint32_t pos = offs[(int64_t)blockIdx.x * kSchedCats + cat] + rank;
    if (bin >= 0) {
        for (int w = 0; w < (int)(blockDim.x >> 6); ++w) {
            if (w == wave) continue;
            for (int k = bin0; k < bin; ++k) pos += wave_bin[w][k];
            if (w < wave) pos += wave_bin[w][bin];
        }
    } else {
        for (int w = 0; w < wave; ++w) pos += wave_cnt[w][cat];
    }
    if (cat < kNumClass) {
        items[pos] = Item{(int32_t)r, start, len, -1};
    } else if ((int64_t)pos < cap_long) {
        long_rows[3 * (int64_t)pos + 0] = (int32_t)r;
        long_rows[3 * (int64_t)pos + 1] = start;
        long_rows[3 * (int64_t)pos + 2] = len;
    }
}

// How a long row is cut (the same arithmetic on the device and wherever it is checked): balanced segments
// of at most block_seg edges; a row with more than spread_segs of those (a global node) gets segments of
// spread_seg edges instead, each scheduled next to the rows it gathers.
struct CutParams { int block_seg, spread_segs, spread_seg, combine_fan, window, near; };
__host__ __device__ inline void cut_row(const CutParams& cp, int len, int& nseg, int& seg, bool& spread) {
    nseg = (len + cp.block_seg - 1) / cp.block_seg;
    spread = nseg > cp.spread_segs;
    if (spread) nseg = (len + cp.spread_seg - 1) / cp.spread_seg;
    seg = (len + nseg - 1) / nseg;
}

// Long rows -> where their workgroup items, partial slots and combine groups start.  One workgroup per view: every
// thread takes a run of consecutive rows of the list (it is short: rows of more than a wave row's edges), the
// runs' totals are scanned in LDS, then every thread writes its rows.
__global__ __launch_bounds__(1024) void k_cut_rows(const SchedArgs a, CutParams cp) {
    const int32_t* __restrict__ long_rows = a.long_rows[blockIdx.y];
    SchedHeader* __restrict__ hdr = a.hdr[blockIdx.y];
    int32_t *__restrict__ row_item_off = a.row_item_off[blockIdx.y], *__restrict__ row_split_idx = a.row_split_idx[blockIdx.y],
            *__restrict__ row_part_off = a.row_part_off[blockIdx.y], *__restrict__ split_row = a.split_row[blockIdx.y],
            *__restrict__ split_off = a.split_off[blockIdx.y], *__restrict__ split_grp = a.split_grp[blockIdx.y];
    __shared__ uint32_t sh[4][1024];
    const int n_long = hdr->n_long;
    const int tid = threadIdx.x;
    const int chunk = (n_long + 1023) / 1024;
    const int b = min(tid * chunk, n_long), e = min(b + chunk, n_long);
    uint32_t items = 0, splits = 0, parts = 0, groups = 0;
    for (int i = b; i < e; ++i) {
        int nseg, seg;
        bool spread;
        cut_row(cp, long_rows[3 * i + 2], nseg, seg, spread);
        items += (uint32_t)nseg;
        if (nseg > 1) { splits += 1; parts += (uint32_t)nseg; }
        if (nseg > cp.combine_fan) groups += (uint32_t)((nseg + cp.combine_fan - 1) / cp.combine_fan);
    }
    sh[0][tid] = items; sh[1][tid] = splits; sh[2][tid] = parts; sh[3][tid] = groups;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {
        uint32_t x[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) x[k] = tid >= off ? sh[k][tid - off] : 0u;
        __syncthreads();
#pragma unroll
        for (int k = 0; k < 4; ++k) sh[k][tid] += x[k];
        __syncthreads();
    }
    // running totals in front of this thread's rows
    items = tid ? sh[0][tid - 1] : 0u; splits = tid ? sh[1][tid - 1] : 0u;
    parts = tid ? sh[2][tid - 1] : 0u; groups = tid ? sh[3][tid - 1] : 0u;
    for (int i = b; i < e; ++i) {
        int nseg, seg;
        bool spread;
        cut_row(cp, long_rows[3 * i + 2], nseg, seg, spread);
        const bool is_split = nseg > 1;
        row_item_off[i] = (int32_t)items;
        row_split_idx[i] = is_split ? (int32_t)splits : -1;
        row_part_off[i] = (int32_t)parts;
        if (is_split) {
            split_row[splits] = long_rows[3 * i];
            split_off[splits] = (int32_t)parts;
            split_grp[splits] = (int32_t)groups;
            splits += 1; parts += (uint32_t)nseg;
        }
        items += (uint32_t)nseg;
        if (nseg > cp.combine_fan) groups += (uint32_t)((nseg + cp.combine_fan - 1) / cp.combine_fan);
    }
    if (tid == 1023) {
        row_item_off[n_long] = (int32_t)sh[0][1023];
        split_off[sh[1][1023]] = (int32_t)sh[2][1023];
        split_grp[sh[1][1023]] = (int32_t)sh[3][1023];
        hdr->n_block = (int32_t)sh[0][1023];
        hdr->n_split = (int32_t)sh[1][1023];
        hdr->n_parts = (int32_t)sh[2][1023];
        hdr->n_groups = (int32_t)sh[3][1023];
    }
}

// What the host needs to know of a workgroup item to place it: the window it is scheduled with (where most of
// its other endpoints are), its edges, whether it is a short segment of a row that spans the graph.
struct BlockMeta { int32_t home, len, spread; };

// The window that an item is scheduled with: fifteen of its edges are asked for the window of their other endpoint, the one with
// the most others within `near` windows wins, the middle edge where nobody has more.  A single edge would do for rows whose
// endpoints all lie in one cluster; with one edge in five elsewhere it sends every fifth item - long rows hold half of the edges
// of a power-law graph - to an L2 that holds another cluster's rows.  The winner stays spread over the graph where the endpoints
// are (a median would pile all items up in the middle windows).  One edge / fifteen: 870 K nodes, 44 M edges, 64 clusters, bf16
// reads 5.3 + 13.9 / 4.5 + 11.9 GB through L2 misses forward + backward and takes 3443 / 3386 us; 100 K nodes, 3 M edges, 8
// clusters, float32 424 / 411 us; a graph without clusters (64 K nodes) 113 / 113 us.
constexpr int kVotes = 15;
__device__ __forceinline__ int home_window(const int32_t* __restrict__ col, int64_t first, int len, const CutParams& cp) {
    int w[kVotes];
#pragma unroll
    for (int k = 0; k < kVotes; ++k) w[k] = col[first + (int64_t)len * (2 * k + 1) / (2 * kVotes)] / cp.window;
    int best = w[kVotes / 2], most = 0;
#pragma unroll
    for (int k = 0; k < kVotes; ++k) {
        const int c = (k + kVotes / 2) % kVotes;      // the middle edge first: it wins ties
        int n = 0;
#pragma unroll
        for (int j = 0; j < kVotes; ++j) n += abs(w[j] - w[c]) <= cp.near ? 1 : 0;
        if (n > most) { most = n; best = w[c]; }
    }
    return best;
}

// One thread per workgroup item: finds its row in the offsets and writes the item.
__global__ void k_emit_items(const SchedArgs a, CutParams cp) {
    const int32_t* __restrict__ long_rows = a.long_rows[blockIdx.y];
    const SchedHeader* __restrict__ hdr = a.hdr[blockIdx.y];
    const int32_t *__restrict__ row_item_off = a.row_item_off[blockIdx.y], *__restrict__ row_split_idx = a.row_split_idx[blockIdx.y],
                  *__restrict__ row_part_off = a.row_part_off[blockIdx.y], *__restrict__ col = a.col[blockIdx.y];
    Item* __restrict__ block_items = a.block_items[blockIdx.y];
    BlockMeta* __restrict__ meta = a.meta[blockIdx.y];
    int32_t* __restrict__ part2split = a.part2split[blockIdx.y];
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= hdr->n_block) return;
    int lo = 0, hi = hdr->n_long - 1;               // last row whose first item is <= j
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (row_item_off[mid] <= j) lo = mid;
        else hi = mid - 1;
    }
    const int i = lo, sgm = j - row_item_off[i];
    const int r = long_rows[3 * i], b = long_rows[3 * i + 1], len = long_rows[3 * i + 2];
    int nseg, seg;
    bool spread;
    cut_row(cp, len, nseg, seg, spread);
    const int o = sgm * seg;
    const int l = (o + seg <= len) ? seg : (len - o);
    const int sidx = row_split_idx[i];
    const int part = sidx >= 0 ? row_part_off[i] + sgm : -1;
    block_items[j] = Item{r, b + o, l, part};
    meta[j] = BlockMeta{home_window(col, (int64_t)b + o, l, cp), l, spread ? 1 : 0};
    if (part >= 0) part2split[part] = sidx;
}

// A run: consecutive waves of the list of one XCD that do the same kind of thing, from wave `wave0` of the list.
//   rows:       the wave items [first, first + n) of one (window, class), rows_per_wave of them per wave
//   block item: workgroup item `first`; its four waves carry the same record
//   nothing:    padding to whole workgroups, and behind the end of a list; n waves
// code: descriptor code (kind, view), the XCD in bits 8 .. 10, the list in bits 11 and 12.
struct Run { int32_t wave0, first, n; uint32_t code; };
enum { LIST_FWD = 0, LIST_BWD = 1, LIST_BWD_GROUPED = 2, LIST_COUNT = 3 };
struct RecordLists { int32_t* recs[LIST_COUNT]; };
__host__ __device__ inline int32_t run_waves(uint32_t kind, int32_t n, int lpe) {
    if (kind == kDescBlock) return 4;
    if (kind == kDescNone) return n;
    const int ipw = rows_per_wave(lpe, (int)kind);
    return (n + ipw - 1) / ipw;
}

// One workgroup per run, for all lists of a shape; its sixteen waves write the run's wave records
// in turn (layout: WaveRec in common.h), the lanes of a wave one edge or bias row each.  Wave lw of
// XCD x's list is wave lw % 4 of that XCD's (lw / 4)-th workgroup, and workgroup b of the launch runs on XCD b mod 8:
// record ((lw / 4) * 8 + x) * 4 + lw % 4.  Everything a kernel uses of a record is written: no clearing pass.
// Bound by the two dependent reads (item, edges) of a record, which the waves of a long run repeat: four records of a wave are asked for
// together (64 K nodes, 0.53 M edges, 57 K records in 4.2 K runs of mostly 8 to 32: sixteen waves and one record at a time 33 us, four waves and four
// records 23).
constexpr int kRecordWaves = 4, kRecordStep = 4;
__global__ __launch_bounds__(64 * kRecordWaves) void k_build_records(const Run* __restrict__ runs, const Item* __restrict__ items_d,
                                                       const Item* __restrict__ items_s, const Item* __restrict__ bitems_d,
                                                       const Item* __restrict__ bitems_s, const int32_t* __restrict__ col_d,
                                                       const int32_t* __restrict__ eid_d, const int32_t* __restrict__ col_s,
                                                       const int32_t* __restrict__ eid_s, WaveRecLayout L, int lpe,
                                                       const RecordLists lists) {
    const Run run = runs[blockIdx.x];
    const int t = threadIdx.x & 63;
    const uint32_t kind = run.code & 7u, xcd = (run.code >> 8) & 7u;
    const bool src = (run.code & kDescSrcSide) != 0;
    const Item* items = src ? items_s : items_d;
    const int32_t* col = src ? col_s : col_d;
    const int32_t* eid = src ? eid_s : eid_d;
    int32_t* const recs = lists.recs[(run.code >> 11) & 3u];
    const int ipw = desc_is_rows(kind) ? rows_per_wave(lpe, (int)kind) : 1;
    const int S = desc_is_rows(kind) ? slots_for_class(lpe, (int)kind) : 1;
    const int groups = kWave / lpe, waves = run_waves(kind, run.n, lpe);
    const auto record = [&](int w) {
        const int lw = run.wave0 + w;
        return recs + (((int64_t)(lw >> 2) * 8 + xcd) * 4 + (lw & 3)) * L.stride;
    };
    if (!desc_is_rows(kind)) {
        for (int w = threadIdx.x >> 6; w < waves; w += kRecordWaves) {
            int32_t* out = record(w);
            if (t != 0) continue;
            if (kind == kDescNone) out[0] = (int32_t)kDescNone;
            else {
                const Item it = (src ? bitems_s : bitems_d)[run.first];
                out[0] = (int32_t)desc_code(kDescBlock, src, 0);
                out[4] = it.row; out[5] = it.start; out[6] = it.len; out[7] = it.part;
            }
        }
        return;
    }
    // the row of lane group g in the wave w; nothing behind the wave's last row (an item of it is read all the same)
    const auto row_of = [&](int w, int g) {
        const int i = g / S, last = run.n - 1 - w * ipw;
        Item it = items[run.first + w * ipw + min(i, last)];
        if (i > last) it = Item{0, 0, 0, -1};
        return it;
    };
    const auto step = [&](int w0, auto records) {
        constexpr int U = decltype(records)::value;
        int32_t* out[U];
        int wave[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            wave[u] = w0 + u * kRecordWaves;
            out[u] = record(wave[u]);
        }
        if (t < groups) {                               // every lane group's entries: a lane finds its row without knowing the class
            Item it[U];
#pragma unroll
            for (int u = 0; u < U; ++u) it[u] = row_of(wave[u], t);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (t == 0) out[u][0] = (int32_t)desc_code(kind, src, (uint32_t)min(ipw, run.n - wave[u] * ipw));
                out[u][L.off_row + t] = it[u].row;
                out[u][L.off_start + t] = it[u].start;
                out[u][L.off_len + t] = it[u].len;
            }
        }
        for (int k = t; k < 4 * groups; k += 64) {      // entry k: edge k % 4 of lane group k / 4
            Item it[U];
#pragma unroll
            for (int u = 0; u < U; ++u) it[u] = row_of(wave[u], k >> 2);
            int c[U], e[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int at = it[u].len > 0 ? it[u].start + min((k >> 2) % S + (k & 3) * S, it[u].len - 1) : 0;
                c[u] = col[at];
                e[u] = eid[at];
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                out[u][L.off_col + k] = it[u].len > 0 ? c[u] : 0;
                out[u][L.off_eid + k] = it[u].len > 0 ? e[u] : 0;
            }
        }
    };
    int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (; w + (kRecordStep - 1) * kRecordWaves < waves; w += kRecordWaves * kRecordStep) step(w, std::integral_constant<int, kRecordStep>{});
    if (w + kRecordWaves < waves) { step(w, std::integral_constant<int, 2>{}); w += 2 * kRecordWaves; }
    if (w < waves) step(w, std::integral_constant<int, 1>{});
}

// ---------------------------------------------------------------------------
// host helpers
// ---------------------------------------------------------------------------
// Sort edge ids by destination and by source (stable; first digits counted) and fill both views' rowptr / col / eid.
static int build_sides(const uint32_t* d32, const uint32_t* s32, int64_t E, int64_t N, RadixSorter& sorter, Side& dst, Side& src, hipStream_t st) {
    SideArrays a{};
    a.keys[0] = d32; a.keys[1] = s32;
    a.other[0] = s32; a.other[1] = d32;
    a.rowptr[0] = dst.rowptr; a.rowptr[1] = src.rowptr;
    a.col[0] = dst.col; a.col[1] = src.col;
    a.eid[0] = dst.eid; a.eid[1] = src.eid;
    if (E > 0) {
        const uint32_t* in[2] = {d32, s32};
        int rc = sorter.sort(in, nullptr, 2, E, bits_for(N), st, a.keys, a.order, true);
        if (rc) return rc;
    }
    const int T = 256;
    const int row_blocks = (int)((N + 1 + T - 1) / T);
    hipLaunchKernelGGL(k_fill_rowptr_and_col, dim3((unsigned)(row_blocks + (E + T - 1) / T), 2), dim3(T), 0, st, a, E, N, row_blocks);
    TGT_HIP_CHECK(hipGetLastError());
    return TGT_OK;
}

static int env_int(const char* name, int dflt) {
    const char* v = getenv(name);
    if (!v || !*v) return dflt;
    const int x = atoi(v);
    return x > 0 ? x : dflt;
}

// twice: large graphs (kManyRows) whose rows are short (kDenseRows) or whose neighbours are near (mostly_near).  Half as many windows to count and place (plan of
// 262 K nodes, 5 M edges 1.00 ms with 128 rows, 0.82 with 256), and forward + backward, 128 / 256 rows, us: 64 clusters, bf16 150 K nodes, 2.8 M edges 187 / 175,
// 262 K, 5 M 345 / 337, 870 K, 44 M 3000 / 2916, with a bias per edge and head 346 / 341, 671 / 664, 7186 / 7117; float32 357 / 356, 707 / 703, 5864 / 5855, with a
// bias 585 / 580, 1085 / 1083.  No clusters, eight edges a row: float32 228 / 226, 432 / 427, 1540 / 1547, bf16 124 / 124, 223 / 220, 841 / 840, with a bias 183 / 182,
// 337 / 335, 1233 / 1217; beside tiles 163 / 165, 161 / 161, 528 / 517.  Not where rows have nineteen far neighbours and more, of which a window's rows share few:
// float32 478 / 491, 882 / 896, 8758 / 8928, eight heads of 16 in bf16 150 K nodes 503 / 521 (eight of 8 246 / 249, 469 / 470, 4736 / 4764).
static int window_rows(bool twice) {
    int w = env_int("TGT_WINDOW_ROWS", twice ? 2 * tgt::kWindowRows : tgt::kWindowRows);
    w = (w + 63) / 64 * 64;
    return w > 64 * kSchedMaxWaves ? 64 * kSchedMaxWaves : w;
}

// Row schedule.  Rows are taken window by window (a window = window_rows() consecutive node ids).
// A row of up to kWaveRowMax edges is one wave item; the wave items of a window are grouped by length
// class (longest first) and keep row order inside a class, so the lanes of a wave see uniform lengths.
// A longer row is walked by whole workgroups: balanced segments, each a workgroup item that is
// scheduled with the window most of its other endpoints lie in (so that the rows a segment gathers
// are the ones the window's own rows load); if there is more than one segment their partial sums
// meet in the workspace.  All of it is made on the device; the host reads back the counts (one copy for
// both views, together with the range-check flag) and, if there are long rows, what it needs to place
// their workgroup items.
struct SideScratch {
    DevBuf rows;      // rows: per long row (row, first edge, length), its first split, partial slot and item
    int64_t cap_long = 0, cap_block = 0;
    CutParams cp{};
    int wave_row_max = 0, W = 0, nwin = 0;
};

// bounds known before anything is counted: a long row has more than wave_row_max edges, a row of len edges
// is cut into at most len / min(block_seg, spread_seg) + 1 segments
static int64_t cap_long_rows(int64_t N, int64_t E) { return std::min<int64_t>(N, E / (env_int("TGT_WAVE_ROW_MAX", tgt::kWaveRowMax) + 1)) + 1; }
static int64_t cap_block_items(int64_t N, int64_t E) {
    return E / std::max(1, std::min(env_int("TGT_BLOCK_SEG", tgt::kBlockSeg), env_int("TGT_SPREAD_SEG", tgt::kSpreadSeg))) + cap_long_rows(N, E) + 1;
}

// ints of the report in front of the per-window counts: two headers, the flag, padding
constexpr int kReportHead = 32;
constexpr int kReportFlag = 16;
// Room for as many workgroup items as there may be comes back with the report up to here: copying it all costs less than the second
// wait that a copy of the items there are needs.  256 KB are 1.4 M edges; plan of 64 K nodes, 0.4 M edges 336 -> 284 us, 1.3 M edges
// 359 -> 346; 262 K nodes, 1.6 M edges 571 -> 574; 524 K, 4.2 M 1187 -> 1207; 870 K, 17 M 3676 -> 3848.
constexpr size_t kOneCopyBytes = 256 << 10;

static int schedule_device(int64_t N, int64_t E, Side* const (&sides)[2], SideScratch (&scr)[2], int32_t* report, BlockMeta* metas, bool skip_empty,
                           int W, hipStream_t st) {
    SchedArgs a{};
    for (int i = 0; i < 2; ++i) {
        Side& side = *sides[i];
        SideScratch& sc = scr[i];
        // tuning overrides (experiments only; the defaults are the measured best)
        sc.wave_row_max = env_int("TGT_WAVE_ROW_MAX", tgt::kWaveRowMax);
        sc.cp.block_seg = env_int("TGT_BLOCK_SEG", tgt::kBlockSeg);
        sc.cp.spread_seg = env_int("TGT_SPREAD_SEG", tgt::kSpreadSeg);
        sc.cp.spread_segs = kSpreadSegs;
        sc.cp.combine_fan = kCombineFan;
        sc.W = W;
        sc.cp.window = sc.W;
        sc.nwin = (int)((N + sc.W - 1) / sc.W);
        sc.cp.near = std::max(1, sc.nwin / 64);
        side.n_windows = sc.nwin;
        const size_t ncnt = (size_t)kSchedCats * sc.nwin;
        a.hdr[i] = reinterpret_cast<SchedHeader*>(report) + i;
        a.counts[i] = reinterpret_cast<uint32_t*>(report) + kReportHead + (size_t)i * 2 * ncnt;
        a.offs[i] = a.counts[i] + ncnt;
        sc.cap_long = cap_long_rows(N, E);
        sc.cap_block = cap_block_items(N, E);
        TGT_HIP_CHECK(dev_alloc((void**)&side.items, sizeof(Item) * (size_t)(N + 1), st));
        TGT_HIP_CHECK(dev_alloc((void**)&side.block_items, sizeof(Item) * (size_t)sc.cap_block, st));
        TGT_HIP_CHECK(dev_alloc((void**)&side.split_row, sizeof(int32_t) * (size_t)(sc.cap_long + 1), st));
        TGT_HIP_CHECK(dev_alloc((void**)&side.split_off, sizeof(int32_t) * (size_t)(sc.cap_long + 1), st));
        TGT_HIP_CHECK(dev_alloc((void**)&side.split_grp, sizeof(int32_t) * (size_t)(sc.cap_long + 1), st));
        TGT_HIP_CHECK(dev_alloc((void**)&side.part2split, sizeof(int32_t) * (size_t)(sc.cap_block + 1), st));
        TGT_HIP_CHECK(sc.rows.alloc(sizeof(int32_t) * (6 * (size_t)sc.cap_long + 1), st));
        a.rowptr[i] = side.rowptr; a.col[i] = side.col; a.items[i] = side.items; a.block_items[i] = side.block_items;
        a.long_rows[i] = sc.rows.as<int32_t>();
        a.row_split_idx[i] = a.long_rows[i] + 3 * sc.cap_long; a.row_part_off[i] = a.row_split_idx[i] + sc.cap_long; a.row_item_off[i] = a.row_part_off[i] + sc.cap_long;
        a.split_row[i] = side.split_row; a.split_off[i] = side.split_off; a.split_grp[i] = side.split_grp; a.part2split[i] = side.part2split;
        a.meta[i] = metas + i * sc.cap_block;
    }
    const SideScratch& sc = scr[0];      // (sizes and parameters are the same)
    hipLaunchKernelGGL(k_sched_count, dim3(sc.nwin, 2), dim3(sc.W), 0, st, a, N, sc.wave_row_max, skip_empty);
    hipLaunchKernelGGL(k_sched_scan, dim3(1, 2), dim3(1024), 0, st, a, sc.nwin);
    hipLaunchKernelGGL(k_sched_fill, dim3(sc.nwin, 2), dim3(sc.W), 0, st, a, N, sc.wave_row_max, skip_empty, sc.cap_long);
    hipLaunchKernelGGL(k_cut_rows, dim3(1, 2), dim3(1024), 0, st, a, sc.cp);
    hipLaunchKernelGGL(k_emit_items, dim3((unsigned)((sc.cap_block + 255) / 256), 2), dim3(256), 0, st, a, sc.cp);
    TGT_HIP_CHECK(hipGetLastError());
    return TGT_OK;
}

// The counts are on the host: sizes of the view's schedule and the per-window tables the placement reads.
static void schedule_counts(Side& side, const SideScratch& sc, const int32_t* report, int side_idx) {
    const SchedHeader& h = reinterpret_cast<const SchedHeader*>(report)[side_idx];
    const size_t ncnt = (size_t)kSchedCats * sc.nwin;
    const uint32_t* counts = reinterpret_cast<const uint32_t*>(report) + kReportHead + (size_t)side_idx * 2 * ncnt;
    side.win_class_cnt.assign(counts, counts + ncnt);
    side.win_class_off.assign(counts + ncnt, counts + 2 * ncnt);
    side.n_block_items = h.n_block;
    side.n_items = h.n_block + h.n_wave;
    side.n_split = h.n_split;
    side.n_parts = h.n_parts;
    side.n_groups = h.n_groups;
}

// ---------------------------------------------------------------------------
// launch descriptors
// ---------------------------------------------------------------------------
// Workgroups reach the 8 XCDs round-robin (workgroup id mod 8) and every XCD has its own L2.  The
// windows are cut into 8 contiguous ranges of about equal work, XCD x walks range x in window order,
// and inside a window the workgroup items homed there come first, then the waves of its rows, longest
// class first - for the backward both views of the window side by side.  What the rows of a window
// load (their own q/k/v/dout rows, the rows of their self-loops, the window's share of a global node's
// segment) then meets in one L2 at about the same time.
namespace {
// Waves of n rows of a class (rows per wave are powers of two)
struct WaveShift {
    int sh[8] = {};      // by kind
    explicit WaveShift(int lpe) {
        for (int c = 0; c < 8; ++c)
            while (desc_is_rows(c) && (1 << sh[c]) < rows_per_wave(lpe, c)) ++sh[c];
    }
    int32_t waves(int c, int64_t n) const { return (int32_t)((n + (1 << sh[c]) - 1) >> sh[c]); }
};
// One XCD's list as runs of waves.
struct XcdList {
    std::vector<Run> runs;
    int32_t waves = 0;
    const WaveShift* ws = nullptr;
    uint32_t where = 0;      // the list's bits of a run's code
    bool grouped = false;    // classes 1 to 3 go out together as kind 6
    void add(uint32_t code, int32_t first, int32_t n) {
        if (n <= 0) return;
        runs.push_back(Run{waves, first, n, code | where});
        const uint32_t kind = code & 7u;
        waves += kind == kDescBlock ? 4 : (kind == kDescNone ? n : ws->waves((int)kind, n));
    }
    void pad4() { if (waves % 4) add(kDescNone, 0, 4 - waves % 4); }
};

// Workgroup items homed at window w_items and the waves of window w of one view (either may be -1: none), appended
// to the list.  part 0: the heavy share (segments of ordinary long rows and the rows of the longest class, which
// run for many steps and whose edges have no tie to the window), part 1: the rest (segments of a row that
// spans the graph, which gather exactly the window's rows, and the short rows).
void append_side(XcdList& xl, const Side& s, int w, int w_items, bool src_side, int part) {
    if (w_items >= 0) {
        for (int32_t q = s.homed_off[w_items]; q < s.homed_off[w_items + 1]; ++q) {
            const int32_t it = s.homed_idx[q];
            if ((s.block_spread[it] != 0) != (part == 1)) continue;
            xl.pad4();      // close a partly filled workgroup first: a workgroup item takes all four waves
            xl.add(desc_code(kDescBlock, src_side, 0), it, 1);
        }
    }
    if (w < 0) return;
    for (int c = (part == 0 ? 0 : 1); c < (part == 0 ? 1 : kNumClass); ++c) {
        uint32_t n = s.win_class_cnt[(size_t)w * (kNumClass + 1) + c], kind = (uint32_t)c;
        if (xl.grouped && c >= 1 && c <= 3) {      // (the classes of a window lie behind each other)
            if (c != 1) continue;
            kind = kDescGroup;
            n += s.win_class_cnt[(size_t)w * (kNumClass + 1) + 2] + s.win_class_cnt[(size_t)w * (kNumClass + 1) + 3];
        }
        xl.add(desc_code(kind, src_side, 0), (int32_t)s.win_class_off[(size_t)w * (kNumClass + 1) + c], (int32_t)n);
    }
}

// runs of all windows -> block order.  XCD x gets a contiguous range of windows; it first walks the
// heavy share of all its windows (long work first keeps the end of the launch short), then window by window.
// Appends one launch's runs to `all_runs`.
void place(const std::vector<const Side*>& sides, int lpe, int list, int32_t* n_blocks, std::vector<Run>& all_runs) {
    const bool grouped = list == LIST_BWD_GROUPED;
    const int nwin = sides[0]->n_windows;
    const bool heavy_first = env_int("TGT_HEAVY_FIRST", 1) == 1;
    const WaveShift shift(lpe);
    // 8 contiguous window ranges with about equal numbers of edges and rows
    int bound[9];
    bound[0] = 0;
    {
        std::vector<double> cost(nwin + 1, 0.0);
        for (int w = 0; w < nwin; ++w) {
            double c = 0.0;
            for (size_t k = 0; k < sides.size(); ++k) {
                const Side* sd = sides[k];
                for (int32_t q = sd->homed_off[w]; q < sd->homed_off[w + 1]; ++q) c += 1.0 + sd->block_len[sd->homed_idx[q]] / 128.0;
                for (int kk = 0; kk < kNumClass; ++kk)
                    c += (kk == 0 ? 0.75 : 0.25) * shift.waves(kk, sd->win_class_cnt[(size_t)w * (kNumClass + 1) + kk]);      // (of grouped rows, too)
            }
            cost[w + 1] = cost[w] + c;
        }
        int x = 1;
        for (int w = 0; w < nwin && x < 8; ++w)
            while (x < 8 && cost[w + 1] * 8 >= cost[nwin] * x) bound[x++] = w + 1;
        while (x <= 8) bound[x++] = nwin;
    }
    // Per XCD and part: runs of whole workgroups.  Part 0 (heavy share) of all windows of the range first.  In
    // part 1 the segments homed at a window run `lead` windows ahead of the window's rows: close enough in
    // time for the rows to meet in the L2, and the last windows of a range end with short rows only - the
    // chain of a split row (partial slot, arrival, sums of the group and of the row) is not left for the end.
    const int lead = env_int("TGT_SEGMENT_LEAD", 3), early_share = env_int("TGT_EARLY_SHARE", 2);
    XcdList xl[8];
    for (int x = 0; x < 8; ++x) {
        XcdList& wv = xl[x];
        wv.ws = &shift;
        wv.grouped = grouped;
        wv.where = ((uint32_t)x << 8) | ((uint32_t)list << 11);
        wv.runs.reserve((size_t)(bound[x + 1] - bound[x] + 8) * 8 * sides.size());
        const int w0 = bound[x], w1 = bound[x + 1];
        if (heavy_first) {
            // one view after the other: the long rows of the destination view gather k and v rows, those of the source
            // view q, dout and the per-node scalars; side by side the two sets compete for the L2 (870 K nodes with
            // 50 edges per row: 3 % faster one after the other; no difference where long rows are few)
            for (size_t k = 0; k < sides.size(); ++k)
                for (int w = w0; w < w1; ++w) append_side(wv, *sides[k], w, w, k == 1, 0);
            wv.pad4();
        }
        // the segments of the last half of the range go first: when the launch ends no split row is still
        // being added up (those windows give up meeting their segment in the L2)
        const int w_early = w1 - (w1 - w0) / early_share;
        for (int w = w_early; w < w1; ++w)
            for (size_t k = 0; k < sides.size(); ++k) append_side(wv, *sides[k], -1, w, k == 1, 1);
        for (int w = w0 - lead; w < w1; ++w) {
            const int wi = w + lead < w_early ? w + lead : -1;        // segments of the window `lead` ahead
            for (size_t k = 0; k < sides.size(); ++k) {
                if (!heavy_first) append_side(wv, *sides[k], w >= w0 ? w : -1, w >= w0 ? w : -1, k == 1, 0);
                append_side(wv, *sides[k], w >= w0 ? w : -1, wi >= w0 ? wi : -1, k == 1, 1);
            }
            if (!grouped) wv.pad4();
        }
    }
    int32_t per = 0;
    for (int x = 0; x < 8; ++x) per = std::max(per, (xl[x].waves + 3) / 4);
    *n_blocks = per * 8;
    for (int x = 0; x < 8; ++x) {
        xl[x].add(kDescNone, 0, per * 4 - xl[x].waves);       // behind the end of the list: records that say "nothing"
        all_runs.insert(all_runs.end(), xl[x].runs.begin(), xl[x].runs.end());
    }
}

// The records of all lists.  `runs` feeds an asynchronous copy: it lives until the stream has been synchronised.
int build_records(const tgt_plan* plan, int lpe, Schedule& sc, std::vector<Run>& runs, DevBuf& runs_d, hipStream_t st) {
    Schedule::List* const lists[LIST_COUNT] = {&sc.fwd, &sc.bwd, &sc.bwd_grouped};
    place({&plan->dst}, lpe, LIST_FWD, &sc.fwd.blocks, runs);
    place({&plan->dst, &plan->src}, lpe, LIST_BWD, &sc.bwd.blocks, runs);
    if (has_grouped_list(plan, lpe)) place({&plan->dst, &plan->src}, lpe, LIST_BWD_GROUPED, &sc.bwd_grouped.blocks, runs);
    const WaveRecLayout L(lpe);
    const size_t rec = (size_t)L.stride * sizeof(int32_t) * 4;
    if (runs.empty()) return TGT_OK;
    TGT_HIP_CHECK(runs_d.alloc(sizeof(Run) * runs.size(), st));
    TGT_HIP_CHECK(hipMemcpyAsync(runs_d.p, runs.data(), sizeof(Run) * runs.size(), hipMemcpyHostToDevice, st));
    RecordLists out{};
    for (int l = 0; l < LIST_COUNT; ++l) {
        if (lists[l]->blocks) TGT_HIP_CHECK(dev_alloc(&lists[l]->recs, rec * lists[l]->blocks, st));
        out.recs[l] = static_cast<int32_t*>(lists[l]->recs);
    }
    const Side &d = plan->dst, &s = plan->src;
    hipLaunchKernelGGL(k_build_records, dim3((unsigned)runs.size()), dim3(64 * kRecordWaves), 0, st, runs_d.as<Run>(), d.items, s.items, d.block_items, s.block_items, d.col,
                       d.eid, s.col, s.eid, L, lpe, out);
    TGT_HIP_CHECK(hipGetLastError());
    return TGT_OK;
}
}  // namespace

const Schedule* plan_schedule_if_ready(const tgt_plan* plan_c, int lpe) {
    tgt_plan* plan = const_cast<tgt_plan*>(plan_c);
    std::lock_guard<std::mutex> lock(plan->sched_mutex);
    for (int idx = 0; idx < kNumLpe; ++idx)
        if ((1 << idx) == lpe) return plan->sched[idx].ready ? &plan->sched[idx] : nullptr;
    return nullptr;
}

const Schedule* plan_schedule(const tgt_plan* plan_c, int lpe, hipStream_t st) {
    int idx = 0;
    while (idx < kNumLpe && (1 << idx) != lpe) ++idx;
    if (idx == kNumLpe) { set_error("no schedule for %d lanes per edge", lpe); return nullptr; }
    tgt_plan* plan = const_cast<tgt_plan*>(plan_c);
    Schedule& sc = plan->sched[idx];
    // the descriptors of a shape are made once, whichever thread or stream asks first
    std::lock_guard<std::mutex> lock(plan->sched_mutex);
    if (sc.ready) return &sc;
    std::vector<Run> runs;
    DevBuf runs_d;
    int rc = build_records(plan, lpe, sc, runs, runs_d, st);
    // the host vector feeds an asynchronous copy: it may go once the stream is idle
    if (hipStreamSynchronize(st) != hipSuccess && rc == TGT_OK) { set_error("hipStreamSynchronize failed"); rc = TGT_ERR_HIP; }
    if (rc != TGT_OK) {
        for (Schedule::List* l : {&sc.fwd, &sc.bwd, &sc.bwd_grouped}) dev_free(l->recs);
        sc = Schedule();
        return nullptr;
    }
    sc.ready = true;
    return &sc;
}

// inv[eid[c]] = c, then pos[p] = inv[eid_src[p]]: where each edge of the source-sorted order sits in the
// destination-sorted order
__global__ void k_invert_perm(const int32_t* __restrict__ eid, int64_t E, int32_t* __restrict__ inv) {
    const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c < E) inv[eid[c]] = (int32_t)c;
}
__global__ void k_compose_perm(const int32_t* __restrict__ eid, const int32_t* __restrict__ inv, int64_t E,
                               int32_t* __restrict__ pos) {
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p < E) pos[p] = inv[eid[p]];
}

__global__ void k_widen(const int32_t* __restrict__ in, int64_t n, int64_t* __restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = in[i];
}

// rows of nv vectors: out[i] = in[eid[i]] (inverse: out[eid[i]] = in[i])
template <typename V>
__global__ void k_permute_rows(const V* __restrict__ in, const int32_t* __restrict__ eid, int64_t E, int nv,
                               V* __restrict__ out, bool inverse) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= E * nv) return;
    const int64_t i = t / nv;
    const int v = (int)(t % nv);
    const int64_t j = eid[i];
    if (!inverse) out[i * nv + v] = in[j * nv + v];
    else out[j * nv + v] = in[i * nv + v];
}

static void free_side(Side& s) {
    dev_free(s.rowptr); dev_free(s.col); dev_free(s.eid); dev_free(s.pos);
    dev_free(s.items); dev_free(s.block_items);
    dev_free(s.split_row); dev_free(s.split_off); dev_free(s.part2split); dev_free(s.split_grp);
    s = Side();
}

static void free_schedules(tgt_plan* plan) {
    for (Schedule& sc : plan->sched) {
        for (Schedule::List* l : {&sc.fwd, &sc.bwd, &sc.bwd_grouped}) dev_free(l->recs);
        sc = Schedule();
    }
}

static int create_impl(const int64_t* d_src, const int64_t* d_dst, int64_t E, int64_t N, hipStream_t st,
                       tgt_plan* plan) {
    plan->N = N;
    plan->E = E;
    TGT_HIP_CHECK(hipGetDevice(&plan->device));
    for (Side* s : {&plan->dst, &plan->src}) {
        TGT_HIP_CHECK(dev_alloc((void**)&s->rowptr, sizeof(int32_t) * (N + 1), st));
        TGT_HIP_CHECK(dev_alloc((void**)&s->col, sizeof(int32_t) * (E ? E : 1), st));
        TGT_HIP_CHECK(dev_alloc((void**)&s->eid, sizeof(int32_t) * (E ? E : 1), st));
    }
    DevBuf s32, d32, report_d;
    RadixSorter sorter;
    const size_t eb = sizeof(uint32_t) * (size_t)(E ? E : 1);
    TGT_HIP_CHECK(s32.alloc(eb, st));
    TGT_HIP_CHECK(d32.alloc(eb, st));
    {
        int rc0 = sorter.init(E, st, 2);
        if (rc0) return rc0;
    }
    // what comes back to the host, in one copy: the two schedule headers, the range-check flag, per view the
    // per-window row counts and their offsets, and where the workgroup items go if there is room for few of them (else that
    // is a second copy, of the items there are)
    const auto report_of = [&](int W) { return kReportHead + 4 * (size_t)kSchedCats * (size_t)((N + W - 1) / W); };      // ints
    const size_t cap_meta = (size_t)cap_block_items(N, E), meta_bytes = 2 * sizeof(BlockMeta) * cap_meta;
    const bool one_copy = meta_bytes <= kOneCopyBytes;
    TGT_HIP_CHECK(report_d.alloc(sizeof(int32_t) * report_of(window_rows(false)) + meta_bytes, st));
    TGT_HIP_CHECK(hipMemsetAsync(report_d.p, 0, sizeof(int32_t) * kReportHead, st));
    int32_t* report = report_d.as<int32_t>();
    if (E > 0) {
        const RadixSorter::Counts c = sorter.counts(E, 2);
        hipLaunchKernelGGL(c.items == RadixSorter::kFewItems ? &k_convert_validate<RadixSorter::kFewItems> : &k_convert_validate<RadixSorter::kManyItems>, dim3(c.blocks),
                           dim3(RadixSorter::kThreads), 0, st, d_src, d_dst, E, N, s32.as<uint32_t>(), d32.as<uint32_t>(), report + kReportFlag, c);
        TGT_HIP_CHECK(hipGetLastError());
    }
    // out-of-range endpoints were replaced by node 0 (and flagged): everything below runs on valid ids
    int rc = build_sides(d32.as<uint32_t>(), s32.as<uint32_t>(), E, N, sorter, plan->dst, plan->src, st);
    if (rc) return rc;
    SideScratch scr[2];
    Side* const views[2] = {&plan->dst, &plan->src};
    bool twice = N >= kManyRows && E < kDenseRows * N;
    if (may_group(N, E) && !plan->rows_with_edges_only) {
        SideArrays a{};
        for (int i = 0; i < 2; ++i) { a.rowptr[i] = views[i]->rowptr; a.col[i] = views[i]->col; }
        constexpr int per = kNearWindows * kWindowRows;
        hipLaunchKernelGGL(k_look_near, dim3((unsigned)((N + per - 1) / per), 2), dim3(kWindowRows), 0, st, a, reinterpret_cast<SchedHeader*>(report), N);
        TGT_HIP_CHECK(hipGetLastError());
        if (N >= kManyRows && !twice) {      // the windows' size follows from it: it comes to the host first
            SchedHeader h[2];
            TGT_HIP_CHECK(hipMemcpyAsync(h, report, sizeof(h), hipMemcpyDeviceToHost, st));
            TGT_HIP_CHECK(hipStreamSynchronize(st));
            twice = mostly_near(h[0]) && mostly_near(h[1]);
        }
    }
    const int W = window_rows(twice);
    const size_t report_ints = report_of(W);
    BlockMeta* const metas = reinterpret_cast<BlockMeta*>(report + report_ints);
    rc = schedule_device(N, E, views, scr, report, metas, plan->rows_with_edges_only, W, st);
    if (rc) return rc;
    std::vector<int32_t> h_report(report_ints + (one_copy ? meta_bytes / 4 : 0));
    TGT_HIP_CHECK(hipMemcpyAsync(h_report.data(), report, sizeof(int32_t) * h_report.size(), hipMemcpyDeviceToHost, st));
    TGT_HIP_CHECK(hipStreamSynchronize(st));
    if (h_report[kReportFlag]) {
        set_error("edge_index holds a node id outside [0, %lld)", (long long)N);
        return TGT_ERR_INDEX_RANGE;
    }
    schedule_counts(plan->dst, scr[0], h_report.data(), 0);
    schedule_counts(plan->src, scr[1], h_report.data(), 1);
    const SchedHeader* hdr = reinterpret_cast<const SchedHeader*>(h_report.data());
    plan->grouped = mostly_near(hdr[0]) && mostly_near(hdr[1]);
    // graphs with rows longer than a wave row: where their workgroup items go
    std::vector<BlockMeta> meta[2];
    for (int i = 0; i < 2; ++i) {
        meta[i].resize(views[i]->n_block_items);
        if (meta[i].empty()) continue;
        if (one_copy) memcpy(meta[i].data(), reinterpret_cast<const BlockMeta*>(h_report.data() + report_ints) + i * cap_meta, sizeof(BlockMeta) * meta[i].size());
        else TGT_HIP_CHECK(hipMemcpyAsync(meta[i].data(), metas + i * cap_meta, sizeof(BlockMeta) * meta[i].size(), hipMemcpyDeviceToHost, st));
    }
    if (!one_copy && !(meta[0].empty() && meta[1].empty())) TGT_HIP_CHECK(hipStreamSynchronize(st));
    for (auto sm : {std::make_pair(&plan->dst, &meta[0]), std::make_pair(&plan->src, &meta[1])}) {
        Side& sd = *sm.first;
        const std::vector<BlockMeta>& m = *sm.second;
        sd.block_home.resize(m.size()); sd.block_len.resize(m.size()); sd.block_spread.resize(m.size());
        for (size_t i = 0; i < m.size(); ++i) {
            sd.block_home[i] = m[i].home; sd.block_len[i] = m[i].len; sd.block_spread[i] = (uint8_t)m[i].spread;
        }
        // workgroup items by the window they are scheduled with (counting sort: item order is kept inside a window)
        const int nw = sd.n_windows > 0 ? sd.n_windows : 1;
        sd.homed_off.assign((size_t)nw + 1, 0);
        for (int32_t& h : sd.block_home) { h = h < 0 ? 0 : (h >= nw ? nw - 1 : h); sd.homed_off[(size_t)h + 1]++; }
        for (int w = 0; w < nw; ++w) sd.homed_off[(size_t)w + 1] += sd.homed_off[w];
        sd.homed_idx.resize(m.size());
        std::vector<int32_t> at(sd.homed_off.begin(), sd.homed_off.end() - 1);
        for (size_t i = 0; i < m.size(); ++i) sd.homed_idx[at[sd.block_home[i]]++] = (int32_t)i;
    }
    // the shape of the reference's node-level models (hidden 64: 8 heads of 8, or 4 of 16); other shapes on first use
    return plan_schedule(plan, 8, st) ? TGT_OK : TGT_ERR_HIP;
}

// ---------------------------------------------------------------------------
// content key of an edge list
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint64_t mix64(uint64_t x) {
    x ^= x >> 33; x *= 0xff51afd7ed558ccdull;
    x ^= x >> 33; x *= 0xc4ceb9fe1a85ec53ull;
    x ^= x >> 33;
    return x;
}
constexpr int kHashBlocks = 1024;
// Two 64-bit sums over all 2E endpoints of mixed (value, position) pairs: a sum does not depend on the order
// of the additions, so the key is the same whatever the grid does, and a value that moves or changes moves it.
__global__ __launch_bounds__(256) void k_hash_partial(const int64_t* __restrict__ src, const int64_t* __restrict__ dst,
                                                      int64_t E, uint64_t* __restrict__ partial) {
    __shared__ uint64_t sh[2][4];
    uint64_t a = 0, b = 0;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < 2 * E; i += (int64_t)gridDim.x * blockDim.x) {
        const uint64_t v = (uint64_t)(i < E ? src[i] : dst[i - E]);
        a += mix64(v * 0x9e3779b97f4a7c15ull + (uint64_t)i * 0xd6e8feb86659fd93ull + 0x2545f4914f6cdd1dull);
        b += mix64((v + (uint64_t)i * 0xa0761d6478bd642full) ^ 0xe7037ed1a0b428dbull);
    }
    for (int off = 32; off > 0; off >>= 1) { a += __shfl_xor(a, off); b += __shfl_xor(b, off); }
    if ((threadIdx.x & 63) == 0) { sh[0][threadIdx.x >> 6] = a; sh[1][threadIdx.x >> 6] = b; }
    __syncthreads();
    if (threadIdx.x == 0) {
        partial[2 * blockIdx.x] = sh[0][0] + sh[0][1] + sh[0][2] + sh[0][3];
        partial[2 * blockIdx.x + 1] = sh[1][0] + sh[1][1] + sh[1][2] + sh[1][3];
    }
}
__global__ __launch_bounds__(64) void k_hash_final(const uint64_t* __restrict__ partial, int n, int64_t E,
                                                   uint64_t* __restrict__ out) {
    uint64_t a = 0, b = 0;
    for (int i = threadIdx.x; i < n; i += 64) { a += partial[2 * i]; b += partial[2 * i + 1]; }
    for (int off = 32; off > 0; off >>= 1) { a += __shfl_xor(a, off); b += __shfl_xor(b, off); }
    if (threadIdx.x == 0) { out[0] = mix64(a ^ (uint64_t)E); out[1] = mix64(b + (uint64_t)E); }
}

}  // namespace tgt

// ---------------------------------------------------------------------------
// C ABI
// ---------------------------------------------------------------------------
extern "C" {

int tgt_version(void) { return 1; }

int tgt_plan_enable_bias_order(tgt_plan_t* plan, void* stream) {
    if (!plan) { tgt::set_error("tgt_plan_enable_bias_order: null plan"); return TGT_ERR_INVALID_ARG; }
    if (plan->src.pos) return TGT_OK;
    const int64_t E = plan->E;
    hipStream_t st = (hipStream_t)stream;
    TGT_HIP_CHECK(tgt::dev_alloc((void**)&plan->src.pos, sizeof(int32_t) * (size_t)(E ? E : 1), st));
    if (E == 0) return TGT_OK;
    tgt::DevBuf inv;
    TGT_HIP_CHECK(inv.alloc(sizeof(int32_t) * (size_t)E, st));
    const unsigned grid = (unsigned)((E + 255) / 256);
    hipLaunchKernelGGL(tgt::k_invert_perm, dim3(grid), dim3(256), 0, st, plan->dst.eid, E, inv.as<int32_t>());
    hipLaunchKernelGGL(tgt::k_compose_perm, dim3(grid), dim3(256), 0, st, plan->src.eid, inv.as<int32_t>(), E,
                       plan->src.pos);
    TGT_HIP_CHECK(hipGetLastError());
    return TGT_OK;      // the scratch buffer goes back to its allocator behind the kernels that read it
}

const char* tgt_error_string(int code) {
    switch (code) {
        case TGT_OK: return "ok";
        case TGT_ERR_INVALID_ARG: return "invalid argument";
        case TGT_ERR_INDEX_RANGE: return "edge endpoint out of range";
        case TGT_ERR_UNSUPPORTED: return "unsupported (H, d, dtype) combination";
        case TGT_ERR_HIP: return "HIP runtime error";
        case TGT_ERR_WORKSPACE: return "workspace too small or misaligned";
        default: return "unknown error";
    }
}

const char* tgt_last_error(void) { return tgt::last_error(); }

int tgt_edge_index_hash(const int64_t* d_src, const int64_t* d_dst, int64_t E, void* stream, uint64_t h_key[2]) {
    if (!h_key || E < 0 || (E > 0 && (!d_src || !d_dst))) {
        tgt::set_error("tgt_edge_index_hash: null pointer or E < 0");
        return TGT_ERR_INVALID_ARG;
    }
    hipStream_t st = (hipStream_t)stream;
    const int nb = (int)std::min<int64_t>(tgt::kHashBlocks, std::max<int64_t>(1, (2 * E + 1023) / 1024));
    tgt::DevBuf buf;
    TGT_HIP_CHECK(buf.alloc(sizeof(uint64_t) * (2 * (size_t)nb + 2), st));
    uint64_t* partial = buf.as<uint64_t>();
    hipLaunchKernelGGL(tgt::k_hash_partial, dim3(nb), dim3(256), 0, st, d_src, d_dst, E, partial);
    hipLaunchKernelGGL(tgt::k_hash_final, dim3(1), dim3(64), 0, st, partial, nb, E, partial + 2 * nb);
    TGT_HIP_CHECK(hipGetLastError());
    TGT_HIP_CHECK(hipMemcpyAsync(h_key, partial + 2 * nb, 2 * sizeof(uint64_t), hipMemcpyDeviceToHost, st));
    TGT_HIP_CHECK(hipStreamSynchronize(st));
    return TGT_OK;
}

static int plan_create_checked(const int64_t* d_src, const int64_t* d_dst, int64_t E, int64_t N, void* stream,
                               bool rows_with_edges_only, tgt_plan_t** out_plan) {
    if (!out_plan || E < 0 || N < 1 || (E > 0 && (!d_src || !d_dst))) {
        tgt::set_error("tgt_plan_create: null pointer, E < 0 or N < 1");
        return TGT_ERR_INVALID_ARG;
    }
    if (E > 0x7fff0000LL || N > 0x7fff0000LL) {
        tgt::set_error("tgt_plan_create: E and N must fit 31 bits");
        return TGT_ERR_INVALID_ARG;
    }
    tgt_plan* plan = new (std::nothrow) tgt_plan();
    if (!plan) return TGT_ERR_INVALID_ARG;
    plan->rows_with_edges_only = rows_with_edges_only;
    int rc = tgt::create_impl(d_src, d_dst, E, N, (hipStream_t)stream, plan);
    if (rc != TGT_OK) {
        tgt::free_side(plan->dst);
        tgt::free_side(plan->src);
        tgt::free_schedules(plan);
        delete plan;
        return rc;
    }
    *out_plan = plan;
    return TGT_OK;
}

int tgt_plan_create(const int64_t* d_src, const int64_t* d_dst, int64_t E, int64_t N, void* stream,
                    tgt_plan_t** out_plan) {
    return plan_create_checked(d_src, d_dst, E, N, stream, false, out_plan);
}

int tgt_plan_create_remaining(const int64_t* d_src, const int64_t* d_dst, int64_t E, int64_t N, void* stream,
                              tgt_plan_t** out_plan) {
    return plan_create_checked(d_src, d_dst, E, N, stream, true, out_plan);
}

int tgt_plan_destroy(tgt_plan_t* plan) {
    if (!plan) return TGT_OK;
    tgt::free_side(plan->dst);
    tgt::free_side(plan->src);
    tgt::free_schedules(plan);
    delete plan;
    return TGT_OK;
}

int tgt_plan_info(const tgt_plan_t* plan, int64_t info[16]) {
    if (!plan || !info) return TGT_ERR_INVALID_ARG;
    for (int i = 0; i < 16; ++i) info[i] = 0;
    info[0] = plan->N;
    info[1] = plan->E;
    info[2] = plan->dst.n_items;
    info[3] = plan->dst.n_split;
    info[4] = plan->dst.n_parts;
    info[5] = plan->src.n_items;
    info[6] = plan->src.n_split;
    info[7] = plan->src.n_parts;
    info[8] = tgt::kBlockSeg;
    info[9] = tgt::kWaveRowMax;
    info[10] = plan->dst.n_block_items;
    info[11] = plan->src.n_block_items;
    info[12] = plan->grouped;
    return TGT_OK;
}

int64_t tgt_plan_array_len(const tgt_plan_t* plan, int which) {
    if (!plan) return -1;
    switch (which) {
        case TGT_PLAN_ROWPTR_DST: case TGT_PLAN_ROWPTR_SRC: return plan->N + 1;
        case TGT_PLAN_COL_DST: case TGT_PLAN_EID_DST:
        case TGT_PLAN_COL_SRC: case TGT_PLAN_EID_SRC: return plan->E;
        case TGT_PLAN_POS_SRC: return plan->src.pos ? plan->E : 0;
        case TGT_PLAN_ITEMS_DST: return 4 * (int64_t)plan->dst.n_items;
        case TGT_PLAN_ITEMS_SRC: return 4 * (int64_t)plan->src.n_items;
        default: return -1;
    }
}

int tgt_plan_export(const tgt_plan_t* plan, int which, int32_t* h_out, int64_t capacity) {
    const int64_t n = tgt_plan_array_len(plan, which);
    if (n < 0 || !h_out || capacity < n) {
        tgt::set_error("tgt_plan_export: bad array id or capacity");
        return TGT_ERR_INVALID_ARG;
    }
    if (n == 0) return TGT_OK;
    if (which == TGT_PLAN_ITEMS_DST || which == TGT_PLAN_ITEMS_SRC) {   // workgroup items, then wave items
        const tgt::Side& s = which == TGT_PLAN_ITEMS_DST ? plan->dst : plan->src;
        const int64_t nb = 4 * (int64_t)s.n_block_items;
        if (nb > 0) TGT_HIP_CHECK(hipMemcpy(h_out, s.block_items, sizeof(int32_t) * nb, hipMemcpyDeviceToHost));
        if (n > nb) TGT_HIP_CHECK(hipMemcpy(h_out + nb, s.items, sizeof(int32_t) * (n - nb), hipMemcpyDeviceToHost));
        return TGT_OK;
    }
    const void* p = nullptr;
    switch (which) {
        case TGT_PLAN_ROWPTR_DST: p = plan->dst.rowptr; break;
        case TGT_PLAN_COL_DST: p = plan->dst.col; break;
        case TGT_PLAN_EID_DST: p = plan->dst.eid; break;
        case TGT_PLAN_ROWPTR_SRC: p = plan->src.rowptr; break;
        case TGT_PLAN_COL_SRC: p = plan->src.col; break;
        case TGT_PLAN_EID_SRC: p = plan->src.eid; break;
        case TGT_PLAN_POS_SRC: p = plan->src.pos; break;
    }
    TGT_HIP_CHECK(hipMemcpy(h_out, p, sizeof(int32_t) * n, hipMemcpyDeviceToHost));
    return TGT_OK;
}

int tgt_plan_sort_rows(const tgt_plan_t* plan, const void* d_in, int row_bytes, void* d_out, int direction, void* stream) {
    if (!plan || row_bytes < 1 || direction < 0 || direction > 2 || (plan->E > 0 && (!d_in || !d_out))) {
        tgt::set_error("tgt_plan_sort_rows: null pointer or bad row size");
        return TGT_ERR_INVALID_ARG;
    }
    if (plan->E == 0) return TGT_OK;
    hipStream_t st = (hipStream_t)stream;
    const int64_t E = plan->E;
    const int32_t* eid = direction == 2 ? plan->src.eid : plan->dst.eid;
    const bool inv = direction == 1;
#define TGT_LAUNCH_PERMUTE(V)                                                                                  \
    do {                                                                                                       \
        const int nv = row_bytes / (int)sizeof(V);                                                             \
        const int64_t total = E * nv;                                                                          \
        hipLaunchKernelGGL((tgt::k_permute_rows<V>), dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st,  \
                           (const V*)d_in, eid, E, nv, (V*)d_out, inv);                                        \
    } while (0)
    const uintptr_t al = (uintptr_t)d_in | (uintptr_t)d_out | (uintptr_t)row_bytes;
    if (al % 16 == 0) TGT_LAUNCH_PERMUTE(uint4);
    else if (al % 8 == 0) TGT_LAUNCH_PERMUTE(uint2);
    else if (al % 4 == 0) TGT_LAUNCH_PERMUTE(uint32_t);
    else if (al % 2 == 0) TGT_LAUNCH_PERMUTE(uint16_t);
    else TGT_LAUNCH_PERMUTE(uint8_t);
#undef TGT_LAUNCH_PERMUTE
    TGT_HIP_CHECK(hipGetLastError());
    return TGT_OK;
}

int tgt_plan_edge_order_src(const tgt_plan_t* plan, int64_t* d_out, void* stream) {
    if (!plan || (plan->E > 0 && !d_out)) { tgt::set_error("tgt_plan_edge_order_src: null pointer"); return TGT_ERR_INVALID_ARG; }
    if (plan->E == 0) return TGT_OK;
    hipLaunchKernelGGL(tgt::k_widen, dim3((unsigned)((plan->E + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                       plan->src.eid, plan->E, d_out);
    TGT_HIP_CHECK(hipGetLastError());
    return TGT_OK;
}

int tgt_plan_edge_order(const tgt_plan_t* plan, int64_t* d_out, void* stream) {
    if (!plan || (plan->E > 0 && !d_out)) { tgt::set_error("tgt_plan_edge_order: null pointer"); return TGT_ERR_INVALID_ARG; }
    if (plan->E == 0) return TGT_OK;
    hipLaunchKernelGGL(tgt::k_widen, dim3((unsigned)((plan->E + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                       plan->dst.eid, plan->E, d_out);
    TGT_HIP_CHECK(hipGetLastError());
    return TGT_OK;
}

}  // extern "C"
