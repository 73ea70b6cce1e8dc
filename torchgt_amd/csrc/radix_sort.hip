// Stable LSD radix sort of (uint32 key, uint32 value) pairs, 8-bit digits.
//
// The ranking is position-based (ballots and prefix counts), so the output is
// the stable order - what numpy's argsort(kind='stable') gives - and is
// bit-reproducible: integer LDS counters only count, they never decide an order.
// Used for the CSR/CSC build (keys = destination / source node) and for the
// graph reordering (keys = partition id, new source id).
#include "common.h"
#include <mutex>
#include <unordered_map>
#include <utility>

namespace tgt {

constexpr int RS_THREADS = RadixSorter::kThreads;
// Keys per thread (a workgroup's tile is 256 times as many; a wave takes a quarter of it, consecutive keys): 4 as long as every tile of a launch has
// a place of its own (eight workgroups per CU), 16 with more.  Few keys are bound by the chain of one tile, sixteen rounds of ballots and
// an LDS counter: 0.53 M keys of two sorts 8.6 us a pass with 4, 12 with 8, 14.5 with 16; 0.2 M of one 6.1, 8.1, 13.9.  Many pay for the
// digits' counts of every tile: a plan of 2 M edges 584 us and 537 with 16, of 44 M 6.9 ms and 5.5.
constexpr int kFewItems = RadixSorter::kFewItems, kManyItems = RadixSorter::kManyItems;
static int rs_items(int64_t n, int sorts) { return n * sorts <= (int64_t)8 * num_cus() * RS_THREADS * kFewItems ? kFewItems : kManyItems; }

// One or two sorts of the same size in a launch (blockIdx.y): the two views of a plan are sorted side by side - at half a
// million keys one of them is a hundred workgroups.
struct RsArgs {
    const uint32_t *keys_in[2], *vals_in[2];
    uint32_t *keys_out[2], *vals_out[2], *hist[2], *totals[2];
};

// Per-workgroup digit histogram, stored digit-major: hist[digit * nblocks + block].
template <int RS_ITEMS>
__global__ __launch_bounds__(RS_THREADS) void k_rs_hist(const RsArgs a, int64_t n, int shift, int nblocks) {
    const uint32_t* __restrict__ keys = a.keys_in[blockIdx.y];
    uint32_t* __restrict__ hist = a.hist[blockIdx.y];
    __shared__ uint32_t h[256];
    const int tid = threadIdx.x;
    h[tid] = 0;
    __syncthreads();
    const int64_t base = (int64_t)blockIdx.x * RS_THREADS * RS_ITEMS;
    uint32_t key[RS_ITEMS];
#pragma unroll
    for (int i = 0; i < RS_ITEMS; ++i) key[i] = keys[min(base + i * RS_THREADS + tid, n - 1)];
#pragma unroll
    for (int i = 0; i < RS_ITEMS; ++i)
        if (base + i * RS_THREADS + tid < n) atomicAdd(&h[(key[i] >> shift) & 255u], 1u);   // integer count: order-free
    __syncthreads();
    hist[(int64_t)tid * nblocks + blockIdx.x] = h[tid];
}

// Workgroup `digit` turns its row of per-block counts into exclusive offsets and
// records the row total.
__global__ __launch_bounds__(256) void k_rs_scan_rows(const RsArgs a, int nblocks) {
    uint32_t *__restrict__ hist = a.hist[blockIdx.y], *__restrict__ totals = a.totals[blockIdx.y];
    __shared__ uint32_t part[256];
    const int tid = threadIdx.x;
    uint32_t* row = hist + (int64_t)blockIdx.x * nblocks;
    const int chunk = (nblocks + 255) / 256;
    const int b = tid * chunk;
    const int e = min(b + chunk, nblocks);
    uint32_t s = 0;
    for (int i = b; i < e; ++i) s += row[i];
    part[tid] = s;
    __syncthreads();
    for (int off = 1; off < 256; off <<= 1) {
        uint32_t x = tid >= off ? part[tid - off] : 0u;
        __syncthreads();
        part[tid] += x;
        __syncthreads();
    }
    uint32_t run = tid ? part[tid - 1] : 0u;
    for (int i = b; i < e; ++i) {
        uint32_t x = row[i];
        row[i] = run;
        run += x;
    }
    if (tid == 255) totals[blockIdx.x] = part[255];
}

// Stable scatter of one radix pass.  Each wave owns a quarter of the tile, consecutive keys, and ranks them in rounds of 64; the rank of a key among equal digits is
// (count in earlier rounds) + (number of lower lanes with the same digit).  The tile
// is then put in digit order in LDS (stable), so that the writes to global memory go
// out as runs of consecutive addresses, one run per digit, instead of one scattered
// 4-byte store per key.  A wave asks for all its keys and values before it ranks the first (past the end: the last key's); loads inside
// the branch that uses them went out one after the other (16.5 us for 0.53 M keys, 14.5 without).
template <int RS_ITEMS>
__global__ __launch_bounds__(RS_THREADS) void k_rs_scatter(const RsArgs a, int64_t n, int shift, int nblocks) {
    constexpr int RS_TILE = RS_THREADS * RS_ITEMS;
    const uint32_t *__restrict__ keys_in = a.keys_in[blockIdx.y], *__restrict__ vals_in = a.vals_in[blockIdx.y];
    uint32_t *__restrict__ keys_out = a.keys_out[blockIdx.y], *__restrict__ vals_out = a.vals_out[blockIdx.y];
    const uint32_t *__restrict__ hist = a.hist[blockIdx.y], *__restrict__ totals = a.totals[blockIdx.y];
    __shared__ uint32_t cnt[4][256];
    __shared__ uint32_t base[256];        // first output position of this tile's keys of a digit
    __shared__ uint32_t scan[256];        // scan of the global digit totals
    __shared__ uint32_t tstart[256];      // scan of the tile's digit counts: first LDS slot of a digit
    __shared__ uint32_t lkey[RS_TILE];
    __shared__ uint32_t lval[RS_TILE];
    const int tid = threadIdx.x;
    const int wave = tid >> 6;
    const int lane = tid & 63;
    for (int i = tid; i < 4 * 256; i += RS_THREADS) (&cnt[0][0])[i] = 0;
    scan[tid] = totals[tid];
    __syncthreads();

    volatile uint32_t* wcnt = &cnt[wave][0];
    uint32_t key[RS_ITEMS], val[RS_ITEMS], rank[RS_ITEMS];
    const int64_t tbase = (int64_t)blockIdx.x * RS_TILE;
    const int64_t wbase = tbase + (int64_t)wave * kWave * RS_ITEMS;
    const uint64_t lower_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
#pragma unroll
    for (int r = 0; r < RS_ITEMS; ++r) key[r] = keys_in[min(wbase + r * kWave + lane, n - 1)];
#pragma unroll
    for (int r = 0; r < RS_ITEMS; ++r) val[r] = vals_in ? vals_in[min(wbase + r * kWave + lane, n - 1)] : (uint32_t)(wbase + r * kWave + lane);
#pragma unroll
    for (int r = 0; r < RS_ITEMS; ++r) {
        const bool valid = wbase + r * kWave + lane < n;
        const uint32_t dg = (key[r] >> shift) & 255u;
        uint64_t same = __ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const bool bit = (dg >> b) & 1u;
            const uint64_t bal = __ballot(bit);
            same &= bit ? bal : ~bal;
        }
        uint32_t prior = 0;
        if (valid) prior = wcnt[dg];
        const uint32_t lower = (uint32_t)__popcll(same & lower_mask);
        rank[r] = prior + lower;
        if (valid && lower == 0) wcnt[dg] = prior + (uint32_t)__popcll(same);
    }
    __syncthreads();
    // exclusive prefix over the 4 waves (thread = digit); the tile's count of the digit
    {
        const uint32_t c0 = cnt[0][tid], c1 = cnt[1][tid], c2 = cnt[2][tid], c3 = cnt[3][tid];
        cnt[0][tid] = 0;
        cnt[1][tid] = c0;
        cnt[2][tid] = c0 + c1;
        cnt[3][tid] = c0 + c1 + c2;
        tstart[tid] = c0 + c1 + c2 + c3;
    }
    __syncthreads();
    // inclusive scans over the 256 digits: global totals and tile counts
    for (int off = 1; off < 256; off <<= 1) {
        const uint32_t x = tid >= off ? scan[tid - off] : 0u;
        const uint32_t y = tid >= off ? tstart[tid - off] : 0u;
        __syncthreads();
        scan[tid] += x;
        tstart[tid] += y;
        __syncthreads();
    }
    const uint32_t my_tstart = tid ? tstart[tid - 1] : 0u;
    base[tid] = (tid ? scan[tid - 1] : 0u) + hist[(int64_t)tid * nblocks + blockIdx.x];
    __syncthreads();
    tstart[tid] = my_tstart;              // now exclusive
    __syncthreads();
    // the tile in digit order (stable) in LDS
#pragma unroll
    for (int r = 0; r < RS_ITEMS; ++r) {
        const int64_t idx = wbase + r * kWave + lane;
        if (idx < n) {
            const uint32_t dg = (key[r] >> shift) & 255u;
            const uint32_t slot = tstart[dg] + cnt[wave][dg] + rank[r];
            lkey[slot] = key[r];
            lval[slot] = val[r];
        }
    }
    __syncthreads();
    const int tile_n = (int)min((int64_t)RS_TILE, n - tbase);
    for (int i = tid; i < tile_n; i += RS_THREADS) {
        const uint32_t kk = lkey[i];
        const uint32_t dg = (kk >> shift) & 255u;
        const uint32_t pos = base[dg] + ((uint32_t)i - tstart[dg]);
        keys_out[pos] = kk;
        vals_out[pos] = lval[i];
    }
}


// allocator hooks (tgt_set_allocator); read on every call, set before the first plan is made
static tgt_alloc_fn g_alloc = nullptr;
static tgt_free_fn g_free = nullptr;
static void* g_alloc_user = nullptr;
// what the hook handed out and has not taken back: memory goes back to where it came from even if the
// hooks were set or cleared in between
static std::mutex g_hooked_mutex;
static std::unordered_map<void*, std::pair<tgt_free_fn, void*>> g_hooked;

hipError_t dev_alloc(void** p, size_t bytes, hipStream_t st) {
    if (bytes == 0) bytes = 4;
    const tgt_alloc_fn alloc = g_alloc;
    if (alloc) {
        *p = alloc(bytes, (void*)st, g_alloc_user);
        if (!*p) return hipErrorOutOfMemory;
        std::lock_guard<std::mutex> lock(g_hooked_mutex);
        g_hooked[*p] = std::make_pair(g_free, g_alloc_user);
        return hipSuccess;
    }
    return hipMalloc(p, bytes);
}
void dev_free(void* p) {
    if (!p) return;
    std::pair<tgt_free_fn, void*> how(nullptr, nullptr);
    {
        std::lock_guard<std::mutex> lock(g_hooked_mutex);
        auto it = g_hooked.find(p);
        if (it != g_hooked.end()) { how = it->second; g_hooked.erase(it); }
    }
    if (how.first) how.first(p, how.second);
    else (void)hipFree(p);
}

hipError_t DevBuf::alloc(size_t bytes, hipStream_t st) {
    if (p) { dev_free(p); p = nullptr; }
    return dev_alloc(&p, bytes, st);
}
DevBuf::~DevBuf() { dev_free(p); }

int bits_for(int64_t n) {
    int bits = 1;
    while (bits < 32 && ((int64_t)1 << bits) < n) ++bits;
    return bits;
}

int RadixSorter::init(int64_t n, hipStream_t st, int sorts) {
    cap_ = n > 0 ? n : 1;
    const int tile = RS_THREADS * rs_items(cap_, sorts);
    nblocks_ = (int)((cap_ + tile - 1) / tile);
    sorts_ = sorts;
    TGT_HIP_CHECK(buf_.alloc(sizeof(uint32_t) * sorts * (4 * (size_t)cap_ + 256 * (size_t)nblocks_ + 256), st));
    return TGT_OK;
}

RadixSorter::Counts RadixSorter::counts(int64_t n, int sorts) const {
    Counts c{};
    // items of the capacity: a smaller sort never has more workgroups than there is room for
    c.items = rs_items(cap_, sorts_);
    c.blocks = (int)((n + RS_THREADS * c.items - 1) / (RS_THREADS * c.items));
    for (int i = 0; i < sorts; ++i) c.hist[i] = buf_.as<uint32_t>() + i * (4 * (size_t)cap_ + 256 * (size_t)nblocks_ + 256) + 4 * (size_t)cap_;
    return c;
}

int RadixSorter::sort(const uint32_t* const* keys_in, const uint32_t* const* vals_in, int sorts, int64_t n, int bits, hipStream_t st,
                      const uint32_t** keys_out, const uint32_t** vals_out, bool counted) {
    if (n > cap_ || sorts > sorts_) { set_error("RadixSorter: n exceeds capacity"); return TGT_ERR_INVALID_ARG; }
    const int passes = (bits + 7) / 8 > 0 ? (bits + 7) / 8 : 1;
    const Counts c = counts(n, sorts);
    const int items = c.items, nblocks = c.blocks;
    RsArgs a{};
    uint32_t *key[2][2], *val[2][2];      // [sort][ping, pong]
    for (int i = 0; i < sorts; ++i) {
        uint32_t* at = c.hist[i] - 4 * (size_t)cap_;
        for (int j = 0; j < 2; ++j) { key[i][j] = at; val[i][j] = at + cap_; at += 2 * cap_; }
        a.hist[i] = c.hist[i]; a.totals[i] = c.hist[i] + 256 * (size_t)nblocks_;
        a.keys_in[i] = keys_in[i];
        a.vals_in[i] = vals_in ? vals_in[i] : nullptr;
    }
    for (int p = 0; p < passes && n > 0; ++p) {
        const int shift = 8 * p;
        for (int i = 0; i < sorts; ++i) { a.keys_out[i] = key[i][p & 1]; a.vals_out[i] = val[i][p & 1]; }
        if (p > 0 || !counted)
            hipLaunchKernelGGL(items == kFewItems ? &k_rs_hist<kFewItems> : &k_rs_hist<kManyItems>, dim3(nblocks, sorts), dim3(RS_THREADS), 0, st, a, n, shift, nblocks);
        hipLaunchKernelGGL(k_rs_scan_rows, dim3(256, sorts), dim3(256), 0, st, a, nblocks);
        hipLaunchKernelGGL(items == kFewItems ? &k_rs_scatter<kFewItems> : &k_rs_scatter<kManyItems>, dim3(nblocks, sorts), dim3(RS_THREADS), 0, st, a, n, shift, nblocks);
        for (int i = 0; i < sorts; ++i) { a.keys_in[i] = a.keys_out[i]; a.vals_in[i] = a.vals_out[i]; }
    }
    TGT_HIP_CHECK(hipGetLastError());
    for (int i = 0; i < sorts; ++i) { keys_out[i] = a.keys_in[i]; vals_out[i] = a.vals_in[i]; }
    return TGT_OK;
}

}  // namespace tgt

extern "C" int tgt_set_allocator(tgt_alloc_fn alloc, tgt_free_fn free_fn, void* user) {
    if ((alloc == nullptr) != (free_fn == nullptr)) {
        tgt::set_error("tgt_set_allocator: give both functions or neither");
        return TGT_ERR_INVALID_ARG;
    }
    tgt::g_alloc = alloc;
    tgt::g_free = free_fn;
    tgt::g_alloc_user = user;
    return TGT_OK;
}
