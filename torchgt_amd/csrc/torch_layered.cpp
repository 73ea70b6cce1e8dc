// Whole node-level models as one operator and one autograd node each, over the kernels that take one step of a layer each
// (linears, LayerNorms, activations, attention): the models whose widths the fused per-node kernels do not have.  The numbers
// are those of the modules step by step; what goes away is the host's time between the launches - a step of four layers
// passes through some forty operators and autograd nodes otherwise, 1.3 ms of host time whatever the graph's size.
// GT of hidden size 64 runs its layers on the fused kernels of gt_layer.hip instead.
//
//   torchgt::layered_graphormer(x, params[7 + 16 L], plan holder, workspace, heads, tokens, classes, eps[2 L + 1]) -> log-probabilities
//   torchgt::node_gt(x, params[8 + 16 L], plan holder, workspace, heads, classes, eps[2 L]) -> log-probabilities
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
    void *packed, *rows_in, *out, *m1, *r1, *m2, *r2, *logits;      // readout: graphormer: out = rows of the final norm; gt: out = last layer's rows
    Norm last;
    std::vector<Layer> l;
    const std::vector<double>* eps;
    void* logp = nullptr;      // fused readout: the log-probabilities [n, classes]
    int64_t classes = 0;
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
    static bool fused_readout(const Dims&) { return false; }
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
    static bool fused_readout(const Dims&) { return false; }
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
    // models/gt_dist_node_level.py:270-286
    static void readout(Tape& t, const Dims& D, const std::vector<Tensor>& p, void* in, Saved& s) {
        auto P = [&](int64_t i) { return p[i].data_ptr(); };
        const int64_t b = kHead + 16 * D.L;
        s.out = in;
        s.m1 = t.take(D.N * D.M1 * D.size); s.r1 = t.take(D.N * D.M1 * D.size); s.m2 = t.take(D.N * D.M2 * D.size); s.r2 = t.take(D.N * D.M2 * D.size);
        s.logits = t.take(D.n * D.Cp * D.size);
        linear_act(t, D, in, {P(b), P(b + 1)}, TGT_ACT_RELU, s.m1, s.r1, D.N, D.C, D.M1);
        linear_act(t, D, s.r1, {P(b + 2), P(b + 3)}, TGT_ACT_RELU, s.m2, s.r2, D.N, D.M1, D.M2);
        linear(t, D, s.r2, {{P(b + 4), P(b + 5)}}, {s.logits}, D.n, D.M2, D.Cp);
    }
    static void readout_back(Tape& t, const Dims& D, const std::vector<const void*>& P, const std::vector<void*>& G, const void* dlogits, void* dm, void* du, void* g,
                             const Saved& s, Sums& sums) {
        const int64_t e = kHead + 16 * D.L;
        linear_act_back(t, D, s.r2, P[e + 4], dlogits, s.m2, TGT_ACT_RELU, dm, G[e + 4], G[e + 5], D.n, D.M2, D.Cp, sums);
        linear_act_back(t, D, s.r1, P[e + 2], dm, s.m1, TGT_ACT_RELU, du, G[e + 2], G[e + 3], D.N, D.M1, D.M2, sums);
        linear_back(t, D, s.out, {P[e]}, {du}, g, {G[e]}, {G[e + 1]}, D.N, D.C, D.M1, sums);
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
        readout(t, D, p, in, s);
    }
    static void backward(Tape& t, const Dims& D, const std::vector<const void*>& P, const std::vector<void*>& G, const void* x, void* dx, const void* dlogits,
                         const tgt_plan_t* plan, const Tensor& ws, const Saved& s) {
        const int64_t row = D.N * D.C * D.size, heads = D.N * D.W * D.size;
        void *g = t.take(row), *d2 = t.take(row), *d1 = t.take(row), *dy = t.take(row), *d_o = t.take(heads), *dq = t.take(heads), *dk = t.take(heads), *dv = t.take(heads),
             *du = t.take(D.N * std::max(D.ff, D.M1) * D.size), *dm = t.take(D.N * D.M2 * D.size);
        Sums sums;
        const int64_t mark = t.used;
        int64_t high = mark;
        auto done = [&] { sums.run(t, D); high = std::max(high, t.used); t.used = mark; };
        readout_back(t, D, P, G, dlogits, dm, du, g, s, sums);
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

// The same with hidden size 64 and 8, 4 or 2 heads, layers on gt_layer.hip.  Packed per layer: O, W1 (two halves of its rows), W2 (two
// halves of its columns), Wq, Wk, Wv and bo, gamma1, beta1, b1 (two), b2, gamma2, beta2, bq, bk, bv.
struct FusedGtModel : GtModel {
    static constexpr int kMats = 8, kVecs = 11, kOut = 3;      // kOut: weights (and biases) of the readout behind the layers'
    static constexpr int64_t kPre = 3 * 4096 + 5 * 64, kPostA = kPre, kPostB = 2 * 4096 + 4 * 64;      // floats of a worker's partials
    static bool covers(const Dims& D) { return D.C == 64 && D.W == 64 && D.ff == 128 && (D.H == 8 || D.H == 4 || D.H == 2); }
    static int64_t unit(const Dims& D) { return tgt_node_frag_bytes(1, D.code) / 2; }
    static bool fused_readout(const Dims& D) { return D.M1 <= 64 && D.M2 <= 64 && D.Cp <= 64; }
    static int64_t mats(const Dims& D) { return kMats * D.L + kOut; }
    static char* weight(const Dims& D, const Saved& s, int64_t l, int i) { return (char*)s.packed + (kMats * l + i) * unit(D); }
    static char* transposed(const Dims& D, const Saved& s, int64_t l, int i) { return weight(D, s, l, i) + mats(D) * unit(D); }
    static float* vec(const Dims& D, const Saved& s, int64_t l, int i) { return (float*)((char*)s.packed + 2 * mats(D) * unit(D)) + (kVecs * l + i) * 64; }
    // the packed parameters and the first linear's rows
    static void begin(Tape& t, const Dims& D, const std::vector<Tensor>& p, const void* x, Saved& s) {
        s.packed = t.take(2 * mats(D) * unit(D) + (kVecs * D.L + kOut) * 64 * 4);
        s.rows_in = t.take(D.N * 64 * D.size);
        if (t.dry()) return;
        std::vector<const void*> m, v;
        std::vector<int> ld, rows(kMats * D.L, 64), cols(kMats * D.L, 64), len(kVecs * D.L, 64);
        for (int64_t l = 0; l < D.L; ++l) {
            const Tensor* w = &p[kHead + 16 * l];
            auto part = [&](int i, int64_t elements) { return static_cast<char*>(w[i].data_ptr()) + elements * D.size; };
            for (const void* q : {part(6, 0), part(10, 0), part(10, 64 * 64), part(12, 0), part(12, 64), part(0, 0), part(2, 0), part(4, 0)}) m.push_back(q);
            for (int i : {64, 64, 64, 128, 128, 64, 64, 64}) ld.push_back(i);
            for (const void* q : {part(7, 0), part(8, 0), part(9, 0), part(11, 0), part(11, 64), part(13, 0), part(14, 0), part(15, 0), part(1, 0), part(3, 0), part(5, 0)}) v.push_back(q);
        }
        // the readout's; where it has kernels of its own widths, the first layer's query weight and bias in its place (not read)
        const Tensor* out = &p[kHead + 16 * D.L];
        for (int i = 0; i < kOut; ++i) {
            const Tensor &W = fused_readout(D) ? out[2 * i] : p[kHead], &b = fused_readout(D) ? out[2 * i + 1] : p[kHead + 1];
            m.push_back(W.data_ptr()); ld.push_back((int)W.size(1)); rows.push_back((int)W.size(0)); cols.push_back((int)W.size(1));
            v.push_back(b.data_ptr()); len.push_back((int)b.numel());
        }
        const tgt_node_pack_args a{m.data(), ld.data(), rows.data(), cols.data(), (int)m.size(), v.data(), len.data(), (int)v.size(), s.packed, vec(D, s, 0, 0)};
        check(tgt_linear_fwd_and_pack(x, p[0].data_ptr(), p[1].data_ptr(), s.rows_in, D.n, (int)D.F, 64, &a, D.code, D.stream), "tgt_linear_fwd_and_pack");
    }
    static void forward(Tape& t, const Dims& D, const std::vector<Tensor>& p, const void* x, const tgt_plan_t* plan, const Tensor& ws, const std::vector<double>& eps, bool keep,
                        Saved& s) {
        const int64_t row = D.N * 64 * D.size;
        auto P = [&](int64_t i) { return p[i].data_ptr(); };
        s.l.assign(D.L, Layer{});
        begin(t, D, p, x, s);
        for (int64_t i = 0; i < D.L; ++i) {
            Layer& l = s.l[i];
            if (i > 0 && !keep) l = s.l[0];
            else {
                l.q = t.take(row); l.k = t.take(row); l.v = t.take(row); l.o = t.take(row);
                l.Z = (float*)t.take(4 * D.N * D.H);
                if (keep) { l.n2.s = t.take(row); l.y1 = t.take(row); }
            }
            l.x = i == 0 || !keep ? s.rows_in : s.l[i - 1].y1;      // (without a backward the stream is rewritten in place)
            if (!keep) l.y1 = l.x;
        }
        const int64_t b = kHead;
        linear(t, D, s.rows_in, {{P(b), P(b + 1)}, {P(b + 2), P(b + 3)}, {P(b + 4), P(b + 5)}}, {s.l[0].q, s.l[0].k, s.l[0].v}, D.N, 64, 64);
        for (int64_t i = 0; i < D.L; ++i) {
            const Layer& l = s.l[i];
            attention(t, D, l, plan, ws);
            tgt_gt_fwd_args a{};
            a.rows = D.N; a.dtype = D.code; a.eps1 = (float)eps[2 * i]; a.eps2 = (float)eps[2 * i + 1];
            a.attn = l.o; a.x = l.x; a.s2 = keep ? l.n2.s : nullptr; a.x_out = l.y1; a.w = weight(D, s, i, 0); a.vec = vec(D, s, i, 0);
            if (i + 1 < D.L) {
                const Layer& n = s.l[i + 1];
                a.q = n.q; a.k = n.k; a.v = n.v; a.w_next = weight(D, s, i + 1, 5); a.v_next = vec(D, s, i + 1, 8);
            }
            if (!t.dry()) check(tgt_gt_fwd(&a, D.stream), "tgt_gt_fwd");
        }
        if (!fused_readout(D)) return readout(t, D, p, s.l[D.L - 1].y1, s);
        s.out = s.l[D.L - 1].y1;
        tgt_readout_fwd_args a{};
        a.rows = D.N; a.dtype = D.code; a.m1 = (int)D.M1; a.m2 = (int)D.M2; a.out = (int)D.Cp; a.classes = (int)s.classes;
        a.x = s.out; a.w = weight(D, s, D.L, 0); a.v = vec(D, s, D.L, 0); a.logp = s.logp;
        if (!t.dry()) check(tgt_readout_fwd(&a, D.stream), "tgt_readout_fwd");
    }
    // dlogits: of the log-probabilities where the readout is one kernel
    static void backward(Tape& t, const Dims& D, const std::vector<const void*>& P, const std::vector<void*>& G, const void* x, void* dx, const void* dlogits,
                         const tgt_plan_t* plan, const Tensor& ws, const Saved& s) {
        const int64_t row = D.N * 64 * D.size;
        void *g = t.take(row), *d1 = t.take(row), *d_o = t.take(row), *dq = t.take(row), *dk = t.take(row), *dv = t.take(row), *du = t.take(D.N * D.M1 * D.size),
             *dm = t.take(D.N * D.M2 * D.size);
        const int workers = tgt_node_bwd_workers(D.N);
        float* partial = (float*)t.take(4 * workers * D.L * (kPre + kPostA + kPostB));
        Sums sums;
        if (fused_readout(D)) {
            tgt_readout_bwd_args a{};
            a.rows = D.N; a.dtype = D.code; a.m1 = (int)D.M1; a.m2 = (int)D.M2; a.out = (int)D.Cp; a.classes = (int)s.classes;
            a.x = s.out; a.dlogp = dlogits; a.logp = s.logp; a.w = weight(D, s, D.L, 0); a.w_back = transposed(D, s, D.L, 0); a.v = vec(D, s, D.L, 0); a.dx = g;
            const int order[6] = {0, 2, 4, 1, 3, 5};
            for (int i = 0; i < 6; ++i) a.grads[i] = G.empty() ? nullptr : G[kHead + 16 * D.L + order[i]];
            a.partial = (float*)t.take(4 * tgt_readout_partial_floats(D.N, (int)D.M1, (int)D.M2, (int)D.Cp));
            if (!t.dry()) check(tgt_readout_bwd(&a, D.stream), "tgt_readout_bwd");
        } else readout_back(t, D, P, G, dlogits, dm, du, g, s, sums);
        std::vector<tgt_node_sum> later;
        auto partial_of = [&](int mats, int ld, std::initializer_list<void*> out) {
            tgt_node_sum d{};
            d.partial = partial; d.workers = workers; d.mats = mats; d.rows = 64; d.ld = ld;
            int i = 0;
            for (void* o : out) d.out[i++] = o;
            later.push_back(d);
            partial += (int64_t)workers * (mats * 4096 + (mats + 2) * 64);
            return const_cast<float*>(d.partial);
        };
        for (int64_t i = D.L - 1; i >= 0; --i) {
            const Layer& l = s.l[i];
            void* const* w = &G[kHead + 16 * i];
            auto part = [&](int k, int64_t elements) { return static_cast<char*>(w[k]) + elements * D.size; };
            tgt_gt_bwd_args a{};
            a.rows = D.N; a.dtype = D.code; a.heads = (int)D.H; a.eps1 = (float)(*s.eps)[2 * i]; a.eps2 = (float)(*s.eps)[2 * i + 1];
            a.g_in = g; a.x = l.x; a.attn = l.o; a.s2 = l.n2.s; a.w = weight(D, s, i, 0); a.w_back = transposed(D, s, i, 0); a.vec = vec(D, s, i, 0); a.Z = l.Z;
            a.g_out = d1; a.d_attn = d_o; a.nd = static_cast<float*>(ws.data_ptr());
            tgt_node_bwd_pre_args b{};
            b.rows = D.N; b.dtype = D.code; b.dq = dq; b.dk = dk; b.dv = dv; b.g_in = d1; b.s = l.x; b.w_back = transposed(D, s, i, 5); b.g_out = g;
            if (t.dry()) continue;
            a.partial_a = partial_of(3, 64, {w[6], w[10], part(10, 64 * 64), w[7], w[11], part(11, 64), w[8], w[9]});
            a.partial_b = partial_of(2, 128, {w[12], part(12, 64), w[13], nullptr, w[14], w[15]});
            b.partial = partial_of(3, 64, {w[0], w[2], w[4], w[1], w[3], w[5], nullptr, nullptr});
            check(tgt_gt_bwd(&a, D.stream), "tgt_gt_bwd");
            check(tgt_sparse_attn_bwd_from_nd(plan, l.q, l.k, l.v, (int)D.H, (int)(64 / D.H), D.code, d_o, dq, dk, dv, ws.data_ptr(), ws.numel(), D.stream),
                  "tgt_sparse_attn_bwd_from_nd");
            check(tgt_node_bwd_pre(&b, D.stream), "tgt_node_bwd_pre");
        }
        linear_back(t, D, x, {P[0]}, {g}, dx, {G[0]}, {G[1]}, D.n, D.F, 64, sums);
        if (!t.dry()) {
            check(tgt_node_sums_and_reduce(later.data(), (int)later.size(), &sums.d.back(), D.code, D.stream), "tgt_node_sums_and_reduce");
            sums.d.pop_back();
        }
        sums.run(t, D);
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
// In the dtype of x also under autocast: the kernels of the backward are told that its gradient has that dtype.
Tensor log_probabilities(const Saved& s, const Dims& D, int64_t classes, const at::TensorOptions& opt) {
    c10::impl::ExcludeDispatchKeyGuard no_autocast(c10::autocast_dispatch_keyset);
    return at::log_softmax(at::from_blob(s.logits, {D.n, D.Cp}, opt).narrow(1, 0, classes), 1);
}

// The tensor that a model with a readout of its own writes them to
template <typename M> Tensor own_log_probabilities(Saved& s, const Dims& D, int64_t classes, const at::TensorOptions& opt) {
    if (!M::fused_readout(D)) return Tensor();
    Tensor logp = at::empty({D.n, classes}, opt);
    s.logp = logp.data_ptr();
    s.classes = classes;
    return logp;
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
        Saved s{};
        const auto* plan = reinterpret_cast<const tgt_plan_t*>(holder->h);
        Tensor logp = own_log_probabilities<M>(s, D, classes, x.options());
        Tensor mem = record(x.options(), [&](Tape& t) { M::forward(t, D, save, x.data_ptr(), plan, ws, eps, true, s); });
        if (!s.logp) logp = log_probabilities(s, D, classes, x.options());
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
        Saved s{};
        s.eps = &eps;
        Tape where;
        where.base = static_cast<char*>(mem.data_ptr());
        M::forward(where, D, sv, x.data_ptr(), plan, ws, eps, true, s);
        Tensor dlogits = grads[0];
        if (M::fused_readout(D)) {
            s.logp = logp.data_ptr();
            s.classes = classes;
        } else {
            dlogits = at::_log_softmax_backward_data(grads[0], logp, 1, logp.scalar_type());
            if (D.Cp != classes) dlogits = at::constant_pad_nd(dlogits, {0, D.Cp - classes});
        }
        TORCH_CHECK(dlogits.scalar_type() == x.scalar_type(), "gradient of the logits in another dtype than x");
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
    Wanted wanted;
    wanted.look(x);
    for (const Tensor& t : P) {
        same_gpu(t, x, name, "every parameter");
        TORCH_CHECK(t.scalar_type() == x.scalar_type(), name, ": parameters must be GPU tensors of x's dtype");
        wanted.look(t);
    }
    same_gpu(ws, x, name, "the plan");
    const Dims D = dims_of<M>(x, P, H, tokens, L);
    M::check_shapes(name, D, P);
    TORCH_CHECK(classes >= 1 && classes <= D.Cp && D.W % H == 0, name, ": classes or heads");
    rows_match_plan(holder, D.N, name);
    std::vector<double> e(eps.begin(), eps.end());
    if (wanted.node()) return LayeredFn<M>::apply(x, P, holder, ws, H, tokens, classes, e);
    c10::DeviceGuard guard(x.device());
    std::vector<Tensor> p;
    for (const Tensor& t : P) p.push_back(t.contiguous());
    Saved s{};
    Tensor logp = own_log_probabilities<M>(s, D, classes, x.options());
    Tensor mem = record(x.options(), [&](Tape& t) { M::forward(t, D, p, x.data_ptr(), reinterpret_cast<const tgt_plan_t*>(holder->h), ws, e, false, s); });
    return s.logp ? logp : log_probabilities(s, D, classes, x.options());
}
Tensor layered_graphormer(const Tensor& x, at::TensorList P, const c10::intrusive_ptr<PlanHolder>& holder, const Tensor& ws, int64_t H, int64_t tokens, int64_t classes,
                          at::ArrayRef<double> eps) {
    TORCH_CHECK(tokens == 1, "layered_graphormer: one global token (its rows are the nodes', the model's are 1 .. of the sequence)");
    return layered<GraphormerModel>("layered_graphormer", x, P, holder, ws, H, tokens, classes, eps);
}
Tensor node_gt(const Tensor& x, at::TensorList P, const c10::intrusive_ptr<PlanHolder>& holder, const Tensor& ws, int64_t H, int64_t classes, at::ArrayRef<double> eps) {
    const bool fused = P.size() >= 24 && FusedGtModel::covers(dims_of<GtModel>(x, P, H, 0, (int64_t)(P.size() - 8) / 16));
    return fused ? layered<FusedGtModel>("node_gt", x, P, holder, ws, H, 0, classes, eps) : layered<GtModel>("node_gt", x, P, holder, ws, H, 0, classes, eps);
}

}  // namespace

TORCH_LIBRARY_FRAGMENT(torchgt, m) {
    m.def("layered_graphormer(Tensor x, Tensor[] params, __torch__.torch.classes.torchgt.PlanHolder plan, Tensor workspace, int heads, int tokens, int classes, "
          "float[] eps) -> Tensor");
    m.def("node_gt(Tensor x, Tensor[] params, __torch__.torch.classes.torchgt.PlanHolder plan, Tensor workspace, int heads, int classes, float[] eps) -> Tensor");
}
TORCH_LIBRARY_IMPL(torchgt, CompositeImplicitAutograd, m) {
    m.impl("layered_graphormer", layered_graphormer);
    m.impl("node_gt", node_gt);
}
