// Whole node-level models as one operator and one autograd node each, over the kernels that take one step of a layer each
// (linears, LayerNorms, activations, attention): the models whose widths the fused per-node kernels do not have.  The numbers
// are those of the modules step by step; what goes away is the host's time between the launches - a step of four layers
// passes through some forty operators and autograd nodes otherwise, 1.3 ms of host time whatever the graph's size.
//
//   torchgt::layered_graphormer(x, params[7 + 16 L], plan holder, workspace, heads, tokens, classes, eps[2 L + 1]) -> log-probabilities
//   torchgt::layered_gt(x, params[8 + 16 L], plan holder, workspace, heads, classes, eps[2 L]) -> log-probabilities
//
// classes: output columns that count (the last weight may be padded to a width the linears read in 16-byte pieces).
#include "torch_common.h"

namespace {

using namespace tgt_torch;

// Runs a pass, or only counts the bytes it takes, or only says where its parts are: the same code lays out a pass and
// performs it.
struct Tape {
    char* base = nullptr;
    bool launch = false;
    int64_t used = 0;
    bool dry() const { return !launch; }
    void* take(int64_t bytes) {
        void* p = base + used;
        used += (bytes + 255) & ~int64_t(255);
        return p;
    }
};
// f(tape) with memory for all that it takes
template <typename F> Tensor record(const at::TensorOptions& opt, const F& f) {
    Tape count;
    f(count);
    Tensor mem = at::empty({count.used + 256}, opt.dtype(at::kByte));
    Tape tape;
    tape.base = static_cast<char*>(mem.data_ptr());
    tape.launch = true;
    f(tape);
    return mem;
}

struct Dims {
    int64_t n, N, F, L, H, tokens, C, W, ff, Cp, M1 = 0, M2 = 0;      // C: width, W: heads' width, ff: feed-forward, Cp: classes of the last weight
    int code, size;
    void* stream;
};

struct Norm { void* s; float *mean, *rstd; };
struct Linear { const void *W, *b; };

// ---- steps ------------------------------------------------------------------------------------------------------------
void linear(Tape& t, const Dims& D, const void* x, std::initializer_list<Linear> w, std::initializer_list<void*> y, int64_t rows, int64_t in, int64_t out) {
    if (t.dry()) return;
    const void *W[3], *B[3];
    void* Y[3];
    int j = 0;
    for (const Linear& l : w) { W[j] = l.W; B[j++] = l.b; }
    j = 0;
    for (void* p : y) Y[j++] = p;
    check(tgt_linear_fwd(x, W, B, Y, j, rows, (int)in, (int)out, D.code, D.stream), "tgt_linear_fwd");
}
void copy(Tape& t, const Dims& D, void* dst, const void* src, int64_t bytes) {
    if (!t.dry()) TORCH_CHECK(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, (hipStream_t)D.stream) == hipSuccess, "hipMemcpyAsync failed");
}
void add_norm(Tape& t, const Dims& D, const void* x, const void* r, const void* gamma, const void* beta, double eps, const Norm& keep, void* y) {
    if (t.dry()) return;
    check(tgt_add_layer_norm_fwd(x, r, gamma, beta, D.N, (int)D.C, (float)eps, D.code, r ? keep.s : nullptr, y, keep.mean, keep.rstd, D.stream), "tgt_add_layer_norm_fwd");
}
void add(Tape& t, const Dims& D, const void* x, const void* r, void* sum, int64_t rows, int64_t width) {
    if (t.dry()) return;
    check(tgt_add_layer_norm_fwd(x, r, nullptr, nullptr, rows, (int)width, 0.f, D.code, sum, nullptr, nullptr, nullptr, D.stream), "tgt_add_layer_norm_fwd");
}
void linear_act(Tape& t, const Dims& D, const void* x, const Linear& w, int act, void* u, void* h, int64_t rows, int64_t in, int64_t out) {
    if (t.dry()) return;
    check(tgt_linear_act_fwd(x, w.W, w.b, rows, (int)in, (int)out, D.code, act, u, h, D.stream), "tgt_linear_act_fwd");
}
// sums over partials, gathered until the workspaces are wanted again
struct Sums {
    std::vector<tgt_reduce_desc> d;
    void run(Tape& t, const Dims& D) {
        if (!t.dry())
            for (size_t i = 0; i < d.size(); i += 8) check(tgt_reduce_partials(d.data() + i, (int)std::min<size_t>(8, d.size() - i), D.code, D.stream), "tgt_reduce_partials");
        d.clear();
    }
};
void linear_back(Tape& t, const Dims& D, const void* x, std::initializer_list<const void*> W_, std::initializer_list<const void*> dy, void* dx,
                 std::initializer_list<void*> dW, std::initializer_list<void*> db, int64_t rows, int64_t in, int64_t out, Sums& sums) {
    const int n = (int)W_.size();
    const int64_t bytes = tgt_linear_bwd_workspace_bytes(n, (int)in, (int)out);
    void* ws = t.take(bytes);
    if (t.dry()) return;
    const void *W[3], *DY[3];
    void *DW[3], *DB[3];
    for (int j = 0; j < n; ++j) { W[j] = W_.begin()[j]; DY[j] = dy.begin()[j]; DW[j] = dW.begin()[j]; DB[j] = db.begin()[j]; }
    sums.d.emplace_back();
    check(tgt_linear_bwd_deferred(x, W, DY, n, rows, (int)in, (int)out, D.code, dx, DW, DB, ws, bytes, D.stream, &sums.d.back()), "tgt_linear_bwd_deferred");
}
void linear_act_back(Tape& t, const Dims& D, const void* h, const void* W, const void* dy, const void* u, int act, void* du, void* dW, void* db, int64_t rows,
                     int64_t in, int64_t out, Sums& sums) {
    const int64_t bytes = tgt_linear_bwd_workspace_bytes(1, (int)in, (int)out);
    void* ws = t.take(bytes);
    if (t.dry()) return;
    sums.d.emplace_back();
    check(tgt_linear_act_bwd(h, W, dy, u, rows, (int)in, (int)out, D.code, act, du, dW, db, ws, bytes, D.stream, &sums.d.back()), "tgt_linear_act_bwd");
}
void norm_back(Tape& t, const Dims& D, const Norm& k, const void* gamma, const void* dy, const void* extra, void* ds, void* dgamma, void* dbeta, Sums& sums) {
    const int64_t bytes = tgt_layer_norm_bwd_workspace_bytes((int)D.C);
    void* ws = t.take(bytes);
    if (t.dry()) return;
    sums.d.emplace_back();
    check(tgt_layer_norm_bwd_deferred(k.s, gamma, k.mean, k.rstd, dy, extra, D.N, (int)D.C, D.code, ds, dgamma, dbeta, ws, bytes, D.stream, &sums.d.back()),
          "tgt_layer_norm_bwd_deferred");
}

// What a layer keeps for its backward.
struct Layer {
    void *x, *y1, *q, *k, *v, *o, *y, *u, *h;
    float* Z;
    Norm n1, n2;
};
struct Saved {
    void *rows_in, *out, *m1, *r1, *m2, *r2, *logits;      // readout: graphormer: out = rows of the final norm; gt: out = last layer's rows
    Norm last;
    std::vector<Layer> l;
};

Norm take_norm(Tape& t, const Dims& D, bool with_sum) { return {with_sum ? t.take(D.N * D.C * D.size) : nullptr, (float*)t.take(4 * D.N), (float*)t.take(4 * D.N)}; }
void attention(Tape& t, const Dims& D, const Layer& l, const tgt_plan_t* plan, const Tensor& ws) {
    if (t.dry()) return;
    check(tgt_sparse_attn_fwd(plan, l.q, l.k, l.v, nullptr, TGT_BIAS_NONE, (int)D.H, (int)(D.W / D.H), D.code, l.o, l.Z, ws.data_ptr(), ws.numel(), D.stream), "tgt_sparse_attn_fwd");
}
void attention_back(Tape& t, const Dims& D, const Layer& l, const tgt_plan_t* plan, const Tensor& ws, const void* d_o, void* dq, void* dk, void* dv) {
    if (t.dry()) return;
    check(tgt_sparse_attn_bwd(plan, l.q, l.k, l.v, nullptr, TGT_BIAS_NONE, (int)D.H, (int)(D.W / D.H), D.code, l.o, l.Z, d_o, dq, dk, dv, nullptr, ws.data_ptr(), ws.numel(),
                              D.stream),
          "tgt_sparse_attn_bwd");
}

// ---- node-level Graphormer (models/graphormer_dist_node_level.py:316-392) -------------------------------------------------
// params: Wn, bn, token table; per layer gamma1, beta1, Wq, bq, Wk, bk, Wv, bv, Wo, bo, gamma2, beta2, W1, b1, W2, b2; gamma, beta, Wh, bh
struct GraphormerModel {
    static constexpr int kHead = 3, kTail = 4;
    static constexpr int kQuery = 2, kFfn = 12;
    static void check_shapes(const char* name, const Dims& D, at::TensorList P) {
        auto is = [&](int64_t i, int64_t out, int64_t in) { TORCH_CHECK(P[i].dim() == 2 && P[i].size(0) == out && P[i].size(1) == in && P[i + 1].numel() == out, name, ": parameter ", i); };
        is(0, D.C, D.F);
        TORCH_CHECK(P[2].dim() == 2 && P[2].size(0) == D.tokens && P[2].size(1) == D.C, name, ": token table");
        for (int64_t l = 0; l < D.L; ++l) {
            const int64_t b = kHead + 16 * l;
            for (int i : {0, 1, 10, 11}) TORCH_CHECK(P[b + i].numel() == D.C, name, ": norms of layer ", l);
            for (int i : {2, 4, 6}) is(b + i, D.W, D.C);
            is(b + 8, D.C, D.W); is(b + 12, D.ff, D.C); is(b + 14, D.C, D.ff);
        }
        const int64_t e = kHead + 16 * D.L;
        TORCH_CHECK(P[e].numel() == D.C && P[e + 1].numel() == D.C, name, ": final norm");
        is(e + 2, D.Cp, D.C);
    }
    static void forward(Tape& t, const Dims& D, const std::vector<Tensor>& p, const void* x, const tgt_plan_t* plan, const Tensor& ws, const std::vector<double>& eps, bool keep,
                        Saved& s) {
        const int64_t row = D.N * D.C * D.size;
        auto P = [&](int64_t i) { return p[i].data_ptr(); };
        s.l.assign(D.L, Layer{});
        s.rows_in = t.take(row);
        if (D.tokens) copy(t, D, s.rows_in, P(2), D.tokens * D.C * D.size);
        linear(t, D, x, {{P(0), P(1)}}, {(char*)s.rows_in + D.tokens * D.C * D.size}, D.n, D.F, D.C);
        void *a = t.take(row), *f = t.take(row), *y1 = keep ? nullptr : t.take(row);
        const void *in = s.rows_in, *pending = nullptr;
        for (int64_t i = 0; i < D.L; ++i) {
            Layer& l = s.l[i];
            const int64_t b = kHead + 16 * i;
            if (i > 0 && !keep) l = s.l[0];
            else {
                l.n1 = take_norm(t, D, i > 0); l.n2 = take_norm(t, D, true);
                l.y1 = keep ? t.take(row) : y1; l.y = t.take(row);
                l.q = t.take(D.N * D.W * D.size); l.k = t.take(D.N * D.W * D.size); l.v = t.take(D.N * D.W * D.size); l.o = t.take(D.N * D.W * D.size);
                l.Z = (float*)t.take(4 * D.N * D.H);
                l.u = t.take(D.N * D.ff * D.size); l.h = t.take(D.N * D.ff * D.size);
            }
            if (!pending) l.n1.s = const_cast<void*>(in);
            add_norm(t, D, in, pending, P(b), P(b + 1), eps[2 * i], l.n1, l.y1);
            linear(t, D, l.y1, {{P(b + 2), P(b + 3)}, {P(b + 4), P(b + 5)}, {P(b + 6), P(b + 7)}}, {l.q, l.k, l.v}, D.N, D.C, D.W);
            attention(t, D, l, plan, ws);
            linear(t, D, l.o, {{P(b + 8), P(b + 9)}}, {a}, D.N, D.W, D.C);
            add_norm(t, D, l.n1.s, a, P(b + 10), P(b + 11), eps[2 * i + 1], l.n2, l.y);
            linear_act(t, D, l.y, {P(b + 12), P(b + 13)}, TGT_ACT_GELU, l.u, l.h, D.N, D.C, D.ff);
            linear(t, D, l.h, {{P(b + 14), P(b + 15)}}, {f}, D.N, D.ff, D.C);
            in = l.n2.s; pending = f;
        }
        const int64_t b = kHead + 16 * D.L;
        s.last = take_norm(t, D, true);
        s.out = t.take(row);
        s.logits = t.take(D.n * D.Cp * D.size);
        add_norm(t, D, in, pending, P(b), P(b + 1), eps[2 * D.L], s.last, s.out);
        linear(t, D, (char*)s.out + D.tokens * D.C * D.size, {{P(b + 2), P(b + 3)}}, {s.logits}, D.n, D.C, D.Cp);
    }
    static void backward(Tape& t, const Dims& D, const std::vector<const void*>& P, const std::vector<void*>& G, const void* x, void* dx, const void* dlogits,
                         const tgt_plan_t* plan, const Tensor& ws, const Saved& s) {
        const int64_t row = D.N * D.C * D.size, heads = D.N * D.W * D.size;
        void *g = t.take(row), *d2 = t.take(row), *dy = t.take(row), *d_o = t.take(heads), *dq = t.take(heads), *dk = t.take(heads), *dv = t.take(heads), *du = t.take(D.N * D.ff * D.size);
        Sums sums;
        const int64_t mark = t.used, e = kHead + 16 * D.L;
        int64_t high = mark;
        auto done = [&] { sums.run(t, D); high = std::max(high, t.used); t.used = mark; };
        if (D.tokens && !t.dry()) at::from_blob(dy, {D.tokens * D.C * D.size}, ws.options()).zero_();      // the classes are not read from the tokens
        linear_back(t, D, (char*)s.out + D.tokens * D.C * D.size, {P[e + 2]}, {dlogits}, (char*)dy + D.tokens * D.C * D.size, {G[e + 2]}, {G[e + 3]}, D.n, D.C, D.Cp, sums);
        norm_back(t, D, s.last, P[e], dy, nullptr, g, G[e], G[e + 1], sums);
        done();
        for (int64_t i = D.L - 1; i >= 0; --i) {
            const Layer& l = s.l[i];
            const int64_t b = kHead + 16 * i;      // g: gradient of the layer's output, of its feed-forward branch and of the stream alike
            linear_act_back(t, D, l.h, P[b + 14], g, l.u, TGT_ACT_GELU, du, G[b + 14], G[b + 15], D.N, D.ff, D.C, sums);
            linear_back(t, D, l.y, {P[b + 12]}, {du}, dy, {G[b + 12]}, {G[b + 13]}, D.N, D.C, D.ff, sums);
            norm_back(t, D, l.n2, P[b + 10], dy, g, d2, G[b + 10], G[b + 11], sums);
            linear_back(t, D, l.o, {P[b + 8]}, {d2}, d_o, {G[b + 8]}, {G[b + 9]}, D.N, D.W, D.C, sums);
            attention_back(t, D, l, plan, ws, d_o, dq, dk, dv);
            linear_back(t, D, l.y1, {P[b + 2], P[b + 4], P[b + 6]}, {dq, dk, dv}, dy, {G[b + 2], G[b + 4], G[b + 6]}, {G[b + 3], G[b + 5], G[b + 7]}, D.N, D.C, D.W, sums);
            norm_back(t, D, l.n1, P[b], dy, d2, g, G[b], G[b + 1], sums);
            done();
        }
        if (D.tokens) copy(t, D, G[2], g, D.tokens * D.C * D.size);
        linear_back(t, D, x, {P[0]}, {(char*)g + D.tokens * D.C * D.size}, dx, {G[0]}, {G[1]}, D.n, D.F, D.C, sums);
        done();
        t.used = high;
    }
};

// ---- node-level GT (models/gt_dist_node_level.py:218-341) -----------------------------------------------------------------
// params: Wn, bn; per layer Wq, bq, Wk, bk, Wv, bv, O, bo, gamma1, beta1, W1, b1, W2, b2, gamma2, beta2; readout W, b three times
struct GtModel {
    static constexpr int kHead = 2, kTail = 6;
    static constexpr int kQuery = 0, kFfn = 10;
    static void check_shapes(const char* name, const Dims& D, at::TensorList P) {
        auto is = [&](int64_t i, int64_t out, int64_t in) { TORCH_CHECK(P[i].dim() == 2 && P[i].size(0) == out && P[i].size(1) == in && P[i + 1].numel() == out, name, ": parameter ", i); };
        is(0, D.C, D.F);
        for (int64_t l = 0; l < D.L; ++l) {
            const int64_t b = kHead + 16 * l;
            for (int i : {0, 2, 4}) is(b + i, D.W, D.C);
            is(b + 6, D.C, D.W);
            for (int i : {8, 9, 14, 15}) TORCH_CHECK(P[b + i].numel() == D.C, name, ": norms of layer ", l);
            is(b + 10, D.ff, D.C); is(b + 12, D.C, D.ff);
        }
        const int64_t e = kHead + 16 * D.L;
        is(e, D.M1, D.C); is(e + 2, D.M2, D.M1); is(e + 4, D.Cp, D.M2);
    }
    static void forward(Tape& t, const Dims& D, const std::vector<Tensor>& p, const void* x, const tgt_plan_t* plan, const Tensor& ws, const std::vector<double>& eps, bool keep,
                        Saved& s) {
        const int64_t row = D.N * D.C * D.size;
        auto P = [&](int64_t i) { return p[i].data_ptr(); };
        s.l.assign(D.L, Layer{});
        s.rows_in = t.take(row);
        linear(t, D, x, {{P(0), P(1)}}, {s.rows_in}, D.n, D.F, D.C);
        void *x1 = t.take(row), *f = t.take(row), *in = s.rows_in;
        for (int64_t i = 0; i < D.L; ++i) {
            Layer& l = s.l[i];
            const int64_t b = kHead + 16 * i;
            if (i > 0 && !keep) l = s.l[0];
            else {
                l.n1 = take_norm(t, D, true); l.n2 = take_norm(t, D, true);
                l.y = t.take(row); l.y1 = t.take(row);
                l.q = t.take(D.N * D.W * D.size); l.k = t.take(D.N * D.W * D.size); l.v = t.take(D.N * D.W * D.size); l.o = t.take(D.N * D.W * D.size);
                l.Z = (float*)t.take(4 * D.N * D.H);
                l.u = t.take(D.N * D.ff * D.size); l.h = t.take(D.N * D.ff * D.size);
            }
            l.x = in;
            linear(t, D, in, {{P(b), P(b + 1)}, {P(b + 2), P(b + 3)}, {P(b + 4), P(b + 5)}}, {l.q, l.k, l.v}, D.N, D.C, D.W);
            attention(t, D, l, plan, ws);
            linear(t, D, l.o, {{P(b + 6), P(b + 7)}}, {l.y}, D.N, D.W, D.C);
            add_norm(t, D, in, l.y, P(b + 8), P(b + 9), eps[2 * i], l.n1, x1);
            linear_act(t, D, l.y, {P(b + 10), P(b + 11)}, TGT_ACT_RELU, l.u, l.h, D.N, D.C, D.ff);
            linear(t, D, l.h, {{P(b + 12), P(b + 13)}}, {f}, D.N, D.ff, D.C);
            add_norm(t, D, x1, f, P(b + 14), P(b + 15), eps[2 * i + 1], l.n2, l.y1);      // y1: the layer's output
            in = l.y1;
        }
        const int64_t b = kHead + 16 * D.L;
        s.out = in;
        s.m1 = t.take(D.N * D.M1 * D.size); s.r1 = t.take(D.N * D.M1 * D.size); s.m2 = t.take(D.N * D.M2 * D.size); s.r2 = t.take(D.N * D.M2 * D.size);
        s.logits = t.take(D.n * D.Cp * D.size);
        linear_act(t, D, in, {P(b), P(b + 1)}, TGT_ACT_RELU, s.m1, s.r1, D.N, D.C, D.M1);
        linear_act(t, D, s.r1, {P(b + 2), P(b + 3)}, TGT_ACT_RELU, s.m2, s.r2, D.N, D.M1, D.M2);
        linear(t, D, s.r2, {{P(b + 4), P(b + 5)}}, {s.logits}, D.n, D.M2, D.Cp);
    }
    static void backward(Tape& t, const Dims& D, const std::vector<const void*>& P, const std::vector<void*>& G, const void* x, void* dx, const void* dlogits,
                         const tgt_plan_t* plan, const Tensor& ws, const Saved& s) {
        const int64_t row = D.N * D.C * D.size, heads = D.N * D.W * D.size;
        void *g = t.take(row), *d2 = t.take(row), *d1 = t.take(row), *dy = t.take(row), *d_o = t.take(heads), *dq = t.take(heads), *dk = t.take(heads), *dv = t.take(heads),
             *du = t.take(D.N * std::max(D.ff, D.M1) * D.size), *dm = t.take(D.N * D.M2 * D.size);
        Sums sums;
        const int64_t mark = t.used, e = kHead + 16 * D.L;
        int64_t high = mark;
        auto done = [&] { sums.run(t, D); high = std::max(high, t.used); t.used = mark; };
        linear_act_back(t, D, s.r2, P[e + 4], dlogits, s.m2, TGT_ACT_RELU, dm, G[e + 4], G[e + 5], D.n, D.M2, D.Cp, sums);
        linear_act_back(t, D, s.r1, P[e + 2], dm, s.m1, TGT_ACT_RELU, du, G[e + 2], G[e + 3], D.N, D.M1, D.M2, sums);
        linear_back(t, D, s.out, {P[e]}, {du}, g, {G[e]}, {G[e + 1]}, D.N, D.C, D.M1, sums);
        done();
        for (int64_t i = D.L - 1; i >= 0; --i) {
            const Layer& l = s.l[i];
            const int64_t b = kHead + 16 * i;
            norm_back(t, D, l.n2, P[b + 14], g, nullptr, d2, G[b + 14], G[b + 15], sums);      // of x1 and of the feed-forward branch
            linear_act_back(t, D, l.h, P[b + 12], d2, l.u, TGT_ACT_RELU, du, G[b + 12], G[b + 13], D.N, D.ff, D.C, sums);
            linear_back(t, D, l.y, {P[b + 10]}, {du}, dy, {G[b + 10]}, {G[b + 11]}, D.N, D.C, D.ff, sums);
            norm_back(t, D, l.n1, P[b + 8], d2, nullptr, d1, G[b + 8], G[b + 9], sums);        // of the layer's input and of y
            add(t, D, dy, d1, dy, D.N, D.C);
            linear_back(t, D, l.o, {P[b + 6]}, {dy}, d_o, {G[b + 6]}, {G[b + 7]}, D.N, D.W, D.C, sums);
            attention_back(t, D, l, plan, ws, d_o, dq, dk, dv);
            linear_back(t, D, l.x, {P[b], P[b + 2], P[b + 4]}, {dq, dk, dv}, g, {G[b], G[b + 2], G[b + 4]}, {G[b + 1], G[b + 3], G[b + 5]}, D.N, D.C, D.W, sums);
            add(t, D, g, d1, g, D.N, D.C);
            done();
        }
        linear_back(t, D, x, {P[0]}, {g}, dx, {G[0]}, {G[1]}, D.n, D.F, D.C, sums);
        done();
        t.used = high;
    }
};

template <typename M>
Dims dims_of(const Tensor& x, at::TensorList P, int64_t H, int64_t tokens, int64_t L) {
    Dims D{};
    D.n = x.size(0); D.tokens = tokens; D.N = D.n + tokens; D.F = x.size(1); D.L = L; D.H = H;
    D.C = P[0].size(0); D.W = P[M::kHead + M::kQuery].size(0); D.ff = P[M::kHead + M::kFfn].size(0);
    const int64_t e = M::kHead + 16 * L;
    if (M::kTail == 6) { D.M1 = P[e].size(0); D.M2 = P[e + 2].size(0); }
    D.Cp = P[P.size() - 2].size(0);
    D.code = dtype_code(x); D.size = (int)x.element_size(); D.stream = stream_of(x);
    return D;
}
Tensor log_probabilities(const Saved& s, const Dims& D, int64_t classes, const at::TensorOptions& opt) {
    return at::log_softmax(at::from_blob(s.logits, {D.n, D.Cp}, opt).narrow(1, 0, classes), 1);
}

template <typename M>
struct LayeredFn : public torch::autograd::Function<LayeredFn<M>> {
    static Tensor forward(AutogradContext* ctx, Tensor x, at::TensorList P, c10::intrusive_ptr<PlanHolder> holder, Tensor ws, int64_t H, int64_t tokens, int64_t classes,
                          std::vector<double> eps) {
        c10::DeviceGuard guard(x.device());
        const Dims D = dims_of<M>(x, P, H, tokens, (int64_t)(P.size() - M::kHead - M::kTail) / 16);
        std::vector<Tensor> save;
        save.reserve(P.size() + 4);
        for (const Tensor& t : P) save.push_back(t.contiguous());
        Saved s;
        const auto* plan = reinterpret_cast<const tgt_plan_t*>(holder->h);
        Tensor mem = record(x.options(), [&](Tape& t) { M::forward(t, D, save, x.data_ptr(), plan, ws, eps, true, s); });
        Tensor logp = log_probabilities(s, D, classes, x.options());
        for (const Tensor& t : {x, mem, logp, ws}) save.push_back(t);
        ctx->save_for_backward(save);
        ctx->saved_data["plan"] = holder;
        ctx->saved_data["dims"] = std::vector<int64_t>{H, tokens, classes};
        ctx->saved_data["eps"] = eps;
        return logp;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        std::vector<Tensor> sv = ctx->get_saved_variables();
        const size_t np = sv.size() - 4;
        const Tensor x = sv[np], mem = sv[np + 1], logp = sv[np + 2], ws = sv[np + 3];
        sv.resize(np);
        c10::DeviceGuard guard(x.device());
        const auto dv = ctx->saved_data["dims"].toIntVector();
        const auto eps = ctx->saved_data["eps"].toDoubleVector();
        const auto holder = ctx->saved_data["plan"].toCustomClass<PlanHolder>();
        const auto* plan = reinterpret_cast<const tgt_plan_t*>(holder->h);
        const Dims D = dims_of<M>(x, sv, dv[0], dv[1], (int64_t)(np - M::kHead - M::kTail) / 16);
        const int64_t classes = dv[2];
        Saved s;
        Tape where;
        where.base = static_cast<char*>(mem.data_ptr());
        M::forward(where, D, sv, x.data_ptr(), plan, ws, eps, true, s);
        Tensor dlogits = at::_log_softmax_backward_data(grads[0], logp, 1, logp.scalar_type());
        if (D.Cp != classes) dlogits = at::constant_pad_nd(dlogits, {0, D.Cp - classes});
        dlogits = dlogits.contiguous();
        std::vector<std::vector<int64_t>> shapes;
        std::vector<const void*> W;
        for (const Tensor& t : sv) { shapes.push_back(t.sizes().vec()); W.push_back(t.data_ptr()); }
        FlatGrads grad(shapes, x.options());
        std::vector<void*> G;
        for (const Tensor& t : grad.t) G.push_back(t.data_ptr());
        Tensor dx;
        if (ctx->needs_input_grad(0)) dx = at::empty_like(x);
        record(x.options(), [&](Tape& t) { M::backward(t, D, W, G, x.data_ptr(), dx.defined() ? dx.data_ptr() : nullptr, dlogits.data_ptr(), plan, ws, s); });
        variable_list out;
        out.reserve(np + 7);
        out.push_back(dx);
        for (Tensor& t : grad.t) out.push_back(std::move(t));
        for (int i = 0; i < 6; ++i) out.push_back(Tensor());
        return out;
    }
};

template <typename M>
Tensor layered(const char* name, const Tensor& x, at::TensorList P, const c10::intrusive_ptr<PlanHolder>& holder, const Tensor& ws, int64_t H, int64_t tokens, int64_t classes,
               at::ArrayRef<double> eps) {
    on_gpu(x, name);
    TORCH_CHECK(x.dim() == 2 && x.is_contiguous(), name, ": x must be a contiguous [n, features]");
    const int64_t per = (int64_t)P.size() - M::kHead - M::kTail, L = per / 16;
    TORCH_CHECK(L >= 1 && per % 16 == 0 && (int64_t)eps.size() == 2 * L + (M::kTail == 4 ? 1 : 0), name, ": 16 parameters and two eps per layer");
    bool train = x.requires_grad();
    for (const Tensor& t : P) {
        TORCH_CHECK(t.defined() && t.is_cuda() && t.scalar_type() == x.scalar_type(), name, ": parameters must be GPU tensors of x's dtype");
        train = train || t.requires_grad();
    }
    const Dims D = dims_of<M>(x, P, H, tokens, L);
    M::check_shapes(name, D, P);
    TORCH_CHECK(classes >= 1 && classes <= D.Cp && D.W % H == 0, name, ": classes or heads");
    rows_match_plan(holder, D.N, name);
    std::vector<double> e(eps.begin(), eps.end());
    if (train && at::GradMode::is_enabled()) return LayeredFn<M>::apply(x, P, holder, ws, H, tokens, classes, e);
    c10::DeviceGuard guard(x.device());
    std::vector<Tensor> p;
    for (const Tensor& t : P) p.push_back(t.contiguous());
    Saved s;
    Tensor mem = record(x.options(), [&](Tape& t) { M::forward(t, D, p, x.data_ptr(), reinterpret_cast<const tgt_plan_t*>(holder->h), ws, e, false, s); });
    return log_probabilities(s, D, classes, x.options());
}
Tensor layered_graphormer(const Tensor& x, at::TensorList P, const c10::intrusive_ptr<PlanHolder>& holder, const Tensor& ws, int64_t H, int64_t tokens, int64_t classes,
                          at::ArrayRef<double> eps) {
    return layered<GraphormerModel>("layered_graphormer", x, P, holder, ws, H, tokens, classes, eps);
}
Tensor layered_gt(const Tensor& x, at::TensorList P, const c10::intrusive_ptr<PlanHolder>& holder, const Tensor& ws, int64_t H, int64_t classes, at::ArrayRef<double> eps) {
    return layered<GtModel>("layered_gt", x, P, holder, ws, H, 0, classes, eps);
}

}  // namespace

TORCH_LIBRARY_FRAGMENT(torchgt, m) {
    m.def("layered_graphormer(Tensor x, Tensor[] params, __torch__.torch.classes.torchgt.PlanHolder plan, Tensor workspace, int heads, int tokens, int classes, "
          "float[] eps) -> Tensor");
    m.def("layered_gt(Tensor x, Tensor[] params, __torch__.torch.classes.torchgt.PlanHolder plan, Tensor workspace, int heads, int classes, float[] eps) -> Tensor");
}
TORCH_LIBRARY_IMPL(torchgt, CompositeImplicitAutograd, m) {
    m.impl("layered_graphormer", layered_graphormer);
    m.impl("layered_gt", layered_gt);
}
