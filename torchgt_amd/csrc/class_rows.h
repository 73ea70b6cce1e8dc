// Rows of class values (log-probabilities, logits and their gradients) on their way between memory and a wave's tile: the last step
// of the node-level models (node_layer.hip, readout.hip).
#pragma once
#include "node_tile.h"

namespace tgt {
namespace {

// Rows of class values.  A wave's R rows are R C consecutive elements of the [N - tokens, C] array and travel through its
// row image, in words: for bf16 the image starts one element late where the rows begin in the middle of a word.
template <typename T, int R> struct ClassRows {
    static constexpr int kPerWord = 4 / (int)sizeof(T);
    T* img;
    int C, lo, hi;            // elements of the wave's rows that exist: [lo, hi)
    int64_t first, total;     // element of the array the rows start at (negative: token rows), elements of the array
    int shift;
    __device__ __forceinline__ ClassRows(vec16* stage, int64_t row0, int64_t N, int tokens, int classes) {
        C = classes;
        const int64_t r = row0 - tokens, left = N - row0;
        first = r * C; total = (N - tokens) * C;
        lo = r < 0 ? (int)(-r < R ? -r : R) * C : 0;
        hi = (int)(left < 0 ? 0 : (left < R ? left : R)) * C;
        shift = kPerWord == 2 ? (int)(first & 1) : 0;
        img = reinterpret_cast<T*>(stage) + shift;
    }
    __device__ __forceinline__ int words() const { return (hi + shift + kPerWord - 1) / kPerWord; }
    // array -> image, in two steps: every load is issued before the first is waited for
    struct Words { uint32_t v[R]; };
    __device__ __forceinline__ void ask(const T* __restrict__ src, Words& words_, int lane) const {
        uint32_t (&v)[R] = words_.v;
        const int n = words();
        const int64_t w0 = (first - shift) / kPerWord, last = total / kPerWord - 1;
        const uint32_t* p = reinterpret_cast<const uint32_t*>(src);
        TGT_EACH(i)
            if (i * 64 < n && last >= 0) {
                int64_t w = w0 + i * 64 + lane;
                w = w < 0 ? 0 : (w > last ? last : w);
                v[i] = p[w];
            }
    }
    __device__ __forceinline__ void land(const T* __restrict__ src, const Words& words_, int lane) const {
        const uint32_t (&v)[R] = words_.v;
        const int n = words();
        const int64_t last = total / kPerWord - 1;
        wave_sync();
        uint32_t* d = reinterpret_cast<uint32_t*>(img - shift);
        TGT_EACH(i)
            if (i * 64 < n && last >= 0 && i * 64 + lane < n) d[i * 64 + lane] = v[i];
        wave_sync();
        if (kPerWord == 2 && (total & 1) && first + hi == total && hi > lo && lane == 0) img[hi - 1] = src[total - 1];      // half a word at the end
        wave_sync();
    }
    __device__ __forceinline__ void store(T* __restrict__ dst, int lane) const {
        const uint32_t* d = reinterpret_cast<const uint32_t*>(img - shift);
        T* out = dst + first;
        const int n = words();
        for (int w = lane; w < n; w += 64) {
            const int e = w * kPerWord - shift;
            if (e >= lo && e + kPerWord <= hi) *reinterpret_cast<uint32_t*>(out + e) = d[w];
            else {
#pragma unroll
                for (int k = 0; k < kPerWord; ++k)
                    if (e + k >= lo && e + k < hi) out[e + k] = img[e + k];
            }
        }
    }
};
template <typename T> __device__ __forceinline__ T to_elem(float v);
template <> __device__ __forceinline__ float to_elem<float>(float v) { return v; }
template <> __device__ __forceinline__ nbf16 to_elem<nbf16>(float v) { return nbf16{__builtin_bit_cast(uint16_t, static_cast<__bf16>(v))}; }

// log_softmax (linear: the rows themselves) over the first C features of a wave's R rows, without the token rows, to `dst`
// NEAR: y - top - log1p(sum - 1), of which neither the sum (the 1 of the largest class comes off exactly) nor top + log sum is rounded to its own size.  rms error
// against 64 bits for 3, 16, 40 and 64 logits of size 1: 4.2e-8, 3.8e-8, 3.9e-8, 3.9e-8, by logf 5.1e-8, 4.7e-8, 4.9e-8, 5.2e-8, torch's log_softmax 4.9e-8, 4.4e-8, 4.5e-8, 4.9e-8.  1 us of
// 18 for 64 K rows, so the GT readout has it, in whose place torch's was.
template <typename T, bool NEAR, int R> __device__ __forceinline__ void put_classes(T* __restrict__ dst, TileOf<R>& y, bool linear, int C, int tokens, int64_t row0, int64_t N, vec16* stage, int lane) {
    const int g = lane / R;
    float lse = 0.f;
    if (!linear) {
        float top = -INFINITY, sum = 0.f;
        TGT_EACH(i) {      // rounded first: log_softmax reads the logits as a T tensor would hold them
            y.set(i, stored(y.get(i), (const T*)nullptr));
            if (R * g + i < C) top = fmaxf(top, y.get(i));
        }
#pragma unroll
        for (int off = R; off < 64; off <<= 1) top = fmaxf(top, __shfl_xor(top, off, 64));
        if constexpr (NEAR) TGT_EACH(i) y.set(i, y.get(i) - top);
        TGT_EACH(i) if (R * g + i < C) sum += expf(NEAR ? y.get(i) : y.get(i) - top);
        sum = node_sum<R>(sum);
        lse = NEAR ? log1pf(sum - 1.f) : top + logf(sum);
    }
    const ClassRows<T, R> out(stage, row0, N, tokens, C);
    wave_sync();
    TGT_EACH(i) if (R * g + i < C) out.img[(lane % R) * C + R * g + i] = to_elem<T>(y.get(i) - lse);
    wave_sync();
    out.store(dst, lane);
}

// Class gradients of a wave's R rows: d logits = d logp - softmax * sum(d logp) (linear: d logits as they come); zero for tokens and past the end.
// bfloat16 asks for both arrays where the object is made, float32 has no registers for that (k_readout_bwd would put 75 to scratch, k_node_bwd_pre 16).
template <typename T, int R> struct ClassGrads {
    static constexpr bool kEarly = sizeof(T) == 2;
    using Words = typename ClassRows<T, R>::Words;
    struct None {};
    ClassRows<T, R> rows;
    std::conditional_t<kEarly, Words, None> dlogp, logp;
    const T *from_d, *from_p;
    int C, lane;
    bool linear;
    __device__ __forceinline__ ClassGrads(const T* __restrict__ dlogp_, const T* __restrict__ logp_, bool linear_, int classes, int tokens, int64_t row0, int64_t N, vec16* stage, int lane_)
        : rows(stage, row0, N, tokens, classes), from_d(dlogp_), from_p(logp_), C(classes), lane(lane_), linear(linear_) {
        if constexpr (kEarly) {
            rows.ask(from_d, dlogp, lane);
            if (!linear) rows.ask(from_p, logp, lane);
        }
    }
    __device__ __forceinline__ void arrive(const T* __restrict__ src, const Words& early) { rows.land(src, early, lane); }
    __device__ __forceinline__ void arrive(const T* __restrict__ src, None) {
        Words w;
        rows.ask(src, w, lane);
        rows.land(src, w, lane);
    }
    __device__ __forceinline__ void settle(TileOf<R>& d) {
        const int n = lane % R, g = lane / R;
        const bool in = n * C >= rows.lo && n * C < rows.hi;
        const T* mine = rows.img + (in ? n * C + R * g : 0);
        arrive(from_d, dlogp);
        float sum = 0.f;
        TGT_EACH(i) {
            d.set(i, in && R * g + i < C ? as_float(mine[i]) : 0.f);
            sum += d.get(i);
        }
        if (linear) return;
        sum = node_sum<R>(sum);
        arrive(from_p, logp);
        TGT_EACH(i) if (in && R * g + i < C) d.set(i, d.get(i) - expf(as_float(mine[i])) * sum);
    }
};

}  // namespace
}  // namespace tgt
