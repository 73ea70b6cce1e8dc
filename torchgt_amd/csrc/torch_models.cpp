// Whole models as one operator and one autograd node each, over the fused per-node kernels (node_layer.hip) and the
// attention: between Python and the kernels of a step there is one call forward and one backward.
//
//   torchgt::node_graphormer(x, params[7 + 16 L], plan holder, workspace, heads, tokens, eps[2 L + 1]) -> log-probabilities
//   torchgt::graph_graphormer(x, in_degree, out_degree, attn_bias, spatial_pos, edge_ids, params[11 (12) + 16 L], multi_hop, max_dist,
//                             heads, eps[2 L + 1], p_drop, seeds[L]) -> predictions
//
// A step's intermediate rows live in one allocation, its parameter gradients in another: with some seventy parameters the
// host's time for tensors of their own would be longer than the kernels of a small graph take.  So every parameter's gradient is a
// part of one storage (a kept one keeps them all, 0.5 MB for the slim models; clone() it to keep one), and all of them are ready when the
// node ends.  Where somebody waits for single gradients (gradients_watched) the model runs layer by layer instead.
//
//   torchgt::gradients_watched(params[]) -> bool
#include "torch_common.h"

namespace {

using namespace tgt_torch;

constexpr int64_t kWidth = 64;

char* at_row(const Tensor& buf, int64_t row) { return static_cast<char*>(buf.data_ptr()) + row * kWidth * buf.element_size(); }
// Packed parameters of the layers: fragments of six weights per layer (Wo, W1, W2, Wq, Wk, Wv), then the classes'; vectors
// per layer (bo, gamma2, beta2, b1, b2; gamma1, beta1, bq, bk, bv), then (gamma, beta, bh) of the classes.
// Order of a layer's parameters: gamma1, beta1, Wq, bq, Wk, bk, Wv, bv, Wo, bo, gamma2, beta2, W1, b1, W2, b2.
struct Packed {
    Tensor frags, vecs;
    int64_t unit = 0;
    int mats = 0;
    Packed() = default;
    // the linear in front of the layers, which one launch does together with the packing
    struct First { const void *x, *W, *b; void* y; int64_t rows, features; };
    // layers: first of their 16 L parameters; classes: gamma, beta, Wh, bh or nullptr
    Packed(const Tensor* layers, int64_t L, const Tensor* classes, int code, const at::TensorOptions& opt, void* stream, const First* first = nullptr) {
        std::vector<const void*> m, v;
        std::vector<int> ld, rows, len;
        static const int wi[6] = {8, 12, 14, 2, 4, 6}, vi[10] = {9, 10, 11, 13, 15, 0, 1, 3, 5, 7};
        for (int64_t l = 0; l < L; ++l) {
            const Tensor* p = layers + 16 * l;
            for (int i : wi) { m.push_back(p[i].data_ptr()); ld.push_back(kWidth); rows.push_back(kWidth); }
            for (int i : vi) { v.push_back(p[i].data_ptr()); len.push_back(kWidth); }
        }
        if (classes) {
            m.push_back(classes[2].data_ptr()); ld.push_back(kWidth); rows.push_back((int)classes[2].size(0));
            v.push_back(classes[0].data_ptr()); len.push_back(kWidth);
            v.push_back(classes[1].data_ptr()); len.push_back(kWidth);
            v.push_back(classes[3].data_ptr()); len.push_back((int)classes[2].size(0));
        }
        mats = (int)m.size();
        const int64_t bytes = tgt_node_frag_bytes(mats, code), vec_bytes = (int64_t)v.size() * kWidth * 4;
        unit = bytes / (2 * mats);
        frags = at::empty({bytes + vec_bytes}, opt.dtype(at::kByte));
        const tgt_node_pack_args a{m.data(), ld.data(), rows.data(), nullptr, mats, v.data(), len.data(), (int)v.size(), frags.data_ptr(),
                                   reinterpret_cast<float*>(static_cast<char*>(frags.data_ptr()) + bytes)};
        if (first)
            check(tgt_linear_fwd_and_pack(first->x, first->W, first->b, first->y, first->rows, (int)first->features, (int)kWidth, &a, code, stream), "tgt_linear_fwd_and_pack");
        else check(tgt_node_pack(a.mats, a.ld, a.rows, a.n_mats, a.vecs, a.lens, a.n_vecs, code, a.d_frags, a.d_vecs, stream), "tgt_node_pack");
    }
    // for the backward: the buffer and what it was made from
    Packed(const Tensor& buf, int n_mats, int code) : frags(buf), unit(tgt_node_frag_bytes(n_mats, code) / (2 * n_mats)), mats(n_mats) {}
    const void* weight(int64_t i) const { return static_cast<char*>(frags.data_ptr()) + i * unit; }
    const void* transposed(int64_t i) const { return static_cast<char*>(frags.data_ptr()) + (mats + i) * unit; }
    const float* vec(int64_t i) const { return reinterpret_cast<const float*>(static_cast<char*>(frags.data_ptr()) + 2 * mats * unit) + i * kWidth; }
};

constexpr int64_t kLayerPartial = 3 * 4096 + 5 * 64, kClassPartial = 4096 + 3 * 64;

// ---------------------------------------------------------------------------------------------------------------
// node-level Graphormer (models/graphormer_dist_node_level.py:316-392), sparse attention without bias, no dropout at work
// ---------------------------------------------------------------------------------------------------------------
struct GraphormerDims { int64_t n, N, F, L, H, tokens, C; };

// params: Wn, bn (node encoder), token table, 16 per layer, gamma, beta (final norm), Wh, bh (classes)
struct GraphormerState {
    Tensor rows, Z, x, logp;      // rows: s_0 .. s_L, then q, k, v, a of every layer
    Packed packed;
};

void graphormer_forward(GraphormerState& st, const GraphormerDims& D, const std::vector<Tensor>& p, const tgt_plan_t* plan, const Tensor& ws,
                        const std::vector<double>& eps, bool keep) {
    const Tensor& x = st.x;
    const int code = dtype_code(x);
    void* stream = stream_of(x);
    const int64_t N = D.N, L = D.L;
    const auto opt = x.options();
    // without a backward the stream is rewritten in place and one set of q, k, v, a serves all layers
    const int64_t ns = keep ? L + 1 : 1, na = keep ? 4 * L : 4;
    st.rows = at::empty({(ns + na) * N, kWidth}, opt);
    st.Z = at::empty({keep ? L * N * D.H : N * D.H}, opt.dtype(at::kFloat));
    st.logp = at::empty({D.n, D.C}, opt);
    const Packed::First encoder{x.data_ptr(), p[0].data_ptr(), p[1].data_ptr(), at_row(st.rows, D.tokens), D.n, x.size(1)};
    st.packed = Packed(p.data() + 3, L, p.data() + 3 + 16 * L, code, opt, stream, &encoder);
    auto s_row = [&](int64_t l) { return at_row(st.rows, keep ? l * N : 0); };
    auto a_row = [&](int64_t l, int i) { return at_row(st.rows, (ns + (keep ? 4 * l : 0) + i) * N); };
    for (int64_t l = 0; l <= L; ++l) {
        tgt_node_fwd_args a{};
        a.rows = N; a.dtype = code; a.tokens = (int)D.tokens;
        if (l == 0) {
            a.s_in = a.s_out = s_row(0);
            a.token = D.tokens ? p[2].data_ptr() : nullptr;
        } else {
            a.attn = a_row(l - 1, 3);
            a.s_in = s_row(l - 1); a.s_out = s_row(l);
            a.w_post = st.packed.weight(6 * (l - 1)); a.v_post = st.packed.vec(10 * (l - 1)); a.eps_post = (float)eps[2 * (l - 1) + 1];
        }
        if (l < L) {
            a.q = a_row(l, 0); a.k = a_row(l, 1); a.v = a_row(l, 2);
            a.w_next = st.packed.weight(6 * l + 3); a.v_next = st.packed.vec(10 * l + 5); a.eps_next = (float)eps[2 * l];
        } else {
            a.logp = st.logp.data_ptr(); a.classes = (int)D.C;
            a.w_next = st.packed.weight(6 * L); a.v_next = st.packed.vec(10 * L); a.eps_next = (float)eps[2 * L];
        }
        check(tgt_node_fwd(&a, stream), "tgt_node_fwd");
        if (l < L)
            check(tgt_sparse_attn_fwd(plan, a.q, a.k, a.v, nullptr, TGT_BIAS_NONE, (int)D.H, (int)(kWidth / D.H), code, a_row(l, 3),
                                      st.Z.data_ptr<float>() + (keep ? l * N * D.H : 0), ws.data_ptr(), ws.numel(), stream),
                  "tgt_sparse_attn_fwd");
    }
}

struct NodeGraphormerFn : public torch::autograd::Function<NodeGraphormerFn> {
    static Tensor forward(AutogradContext* ctx, Tensor x, at::TensorList P, c10::intrusive_ptr<PlanHolder> holder, Tensor ws, GraphormerDims D,
                          std::vector<double> eps) {
        GraphormerState st;
        std::vector<Tensor> p;
        p.reserve(P.size());
        for (const Tensor& t : P) p.push_back(t.contiguous());
        st.x = x;
        c10::DeviceGuard guard(x.device());
        graphormer_forward(st, D, p, reinterpret_cast<const tgt_plan_t*>(holder->h), ws, eps, true);
        ctx->save_for_backward({x, st.rows, st.Z, st.packed.frags, st.logp, ws, p[0]});
        ctx->saved_data["plan"] = holder;
        ctx->saved_data["dims"] = std::vector<int64_t>{D.n, D.N, D.F, D.L, D.H, D.tokens, D.C};
        ctx->saved_data["eps"] = eps;
        ctx->saved_data["token_rows"] = p[2].size(0);
        return st.logp;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        auto sv = ctx->get_saved_variables();
        const Tensor &x = sv[0], &rows = sv[1], &Z = sv[2], &logp = sv[4], &ws = sv[5], &Wn = sv[6];
        const auto dv = ctx->saved_data["dims"].toIntVector();
        const GraphormerDims D{dv[0], dv[1], dv[2], dv[3], dv[4], dv[5], dv[6]};
        const auto eps = ctx->saved_data["eps"].toDoubleVector();
        const int64_t N = D.N, L = D.L, H = D.H;
        const int code = dtype_code(x);
        c10::DeviceGuard guard(x.device());
        void* stream = stream_of(x);
        const auto plan_holder = ctx->saved_data["plan"].toCustomClass<PlanHolder>();
        const tgt_plan_t* plan = reinterpret_cast<const tgt_plan_t*>(plan_holder->h);
        const Packed packed(sv[3], (int)(6 * L + 1), code);
        const Tensor dlogp = grads[0].contiguous();
        std::vector<std::vector<int64_t>> shapes{{kWidth, x.size(1)}, {kWidth}, {ctx->saved_data["token_rows"].toInt(), kWidth}};
        for (int64_t l = 0; l < L; ++l)
            for (int i = 0; i < 16; ++i) {
                if (i >= 2 && i % 2 == 0 && i != 10) shapes.push_back({kWidth, kWidth});
                else shapes.push_back({kWidth});
            }
        for (int i = 0; i < 2; ++i) shapes.push_back({kWidth});
        shapes.push_back({D.C, kWidth});
        shapes.push_back({D.C});
        FlatGrads G(shapes, x.options());
        const int workers = tgt_node_bwd_workers(N);
        Tensor work = at::empty({6 * N, kWidth}, x.options());
        Tensor partial = at::empty({workers * (2 * L * kLayerPartial + kClassPartial)}, x.options().dtype(at::kFloat));
        char *g[2] = {at_row(work, 0), at_row(work, N)}, *da = at_row(work, 2 * N), *dq = at_row(work, 3 * N), *dk = at_row(work, 4 * N), *dvr = at_row(work, 5 * N);
        float* next_partial = partial.data_ptr<float>();
        std::vector<tgt_node_sum> sums;
        auto new_sum = [&](int mats, int n_rows) -> tgt_node_sum& {
            sums.push_back(tgt_node_sum{});
            tgt_node_sum& s = sums.back();
            s.partial = next_partial; s.workers = workers; s.mats = mats; s.rows = n_rows;
            next_partial += (int64_t)workers * (mats * 4096 + (mats + 2) * 64);
            return s;
        };
        // the part in front of an attention (or the classes) waits for the part behind the attention before it: one launch for both
        tgt_node_bwd_pre_args a{};
        {
            a.rows = N; a.dtype = code; a.tokens = (int)D.tokens; a.classes = (int)D.C; a.eps = (float)eps[2 * L];
            a.s = at_row(rows, L * N); a.dlogp = dlogp.data_ptr(); a.logp = logp.data_ptr();
            a.w_back = packed.transposed(6 * L); a.v_next = packed.vec(10 * L); a.g_out = g[0]; a.partial = next_partial;
            tgt_node_sum& s = new_sum(1, (int)D.C);
            const Tensor* c = &G.t[3 + 16 * L];
            s.out[0] = c[2].data_ptr(); s.out[1] = c[3].data_ptr(); s.out[2] = c[0].data_ptr(); s.out[3] = c[1].data_ptr();
        }
        for (int64_t l = L - 1; l >= 0; --l) {
            const Tensor* w = &G.t[3 + 16 * l];
            const char *q = at_row(rows, (L + 1 + 4 * l) * N), *k = q + N * kWidth * x.element_size(), *v = k + N * kWidth * x.element_size(),
                       *at = v + N * kWidth * x.element_size();
            tgt_node_bwd_post_args b{};
            b.rows = N; b.dtype = code; b.heads = (int)H; b.eps = (float)eps[2 * l + 1];
            b.g_in = g[0]; b.s = at_row(rows, l * N); b.attn = at; b.w_post = packed.weight(6 * l); b.w_back = packed.transposed(6 * l);
            b.v_post = packed.vec(10 * l); b.Z = Z.data_ptr<float>() + l * N * H; b.g_out = g[1]; b.d_attn = da;
            b.nd = static_cast<float*>(ws.data_ptr()); b.partial = next_partial;
            tgt_node_sum& s = new_sum(3, (int)kWidth);
            static const int post[8] = {8, 12, 14, 9, 13, 15, 10, 11}, pre[8] = {2, 4, 6, 3, 5, 7, 0, 1};
            for (int i = 0; i < 8; ++i) s.out[i] = w[post[i]].data_ptr();
            check(tgt_node_bwd_both(&a, &b, stream), "tgt_node_bwd_both");
            check(tgt_sparse_attn_bwd_from_nd(plan, q, k, v, (int)H, (int)(kWidth / H), code, da, dq, dk, dvr, ws.data_ptr(), ws.numel(), stream),
                  "tgt_sparse_attn_bwd_from_nd");
            a = tgt_node_bwd_pre_args{};
            a.rows = N; a.dtype = code; a.tokens = (int)D.tokens; a.eps = (float)eps[2 * l];
            a.dq = dq; a.dk = dk; a.dv = dvr; a.g_in = g[1]; a.s = at_row(rows, l * N);
            a.w_back = packed.transposed(6 * l + 3); a.v_next = packed.vec(10 * l + 5); a.g_out = g[0]; a.partial = next_partial;
            a.d_token = l == 0 && D.tokens ? G.t[2].data_ptr() : nullptr;
            tgt_node_sum& s2 = new_sum(3, (int)kWidth);
            for (int i = 0; i < 8; ++i) s2.out[i] = w[pre[i]].data_ptr();
        }
        check(tgt_node_bwd_pre(&a, stream), "tgt_node_bwd_pre");
        Tensor dx;
        {      // the encoder's weight gradient, whose partials are added up beside the layers'
            if (ctx->needs_input_grad(0)) dx = at::empty_like(x);
            const void *W[1] = {Wn.data_ptr()}, *DY[1] = {g[0] + D.tokens * kWidth * x.element_size()};
            void *DW[1] = {G.t[0].data_ptr()}, *DB[1] = {G.t[1].data_ptr()};
            const int64_t bytes = tgt_linear_bwd_workspace_bytes(1, (int)x.size(1), (int)kWidth);
            Tensor lws = at::empty({bytes}, x.options().dtype(at::kByte));
            tgt_reduce_desc sum;
            check(tgt_linear_bwd_deferred(x.data_ptr(), W, DY, 1, D.n, (int)x.size(1), (int)kWidth, code, dx.defined() ? dx.data_ptr() : nullptr, DW, DB,
                                          lws.data_ptr(), bytes, stream, &sum),
                  "tgt_linear_bwd_deferred");
            check(tgt_node_sums_and_reduce(sums.data(), (int)sums.size(), &sum, code, stream), "tgt_node_sums_and_reduce");
        }
        variable_list out;
        out.reserve(G.t.size() + 5);
        out.push_back(dx);
        for (Tensor& t : G.t) out.push_back(std::move(t));
        for (int i = 0; i < 4; ++i) out.push_back(Tensor());
        return out;
    }
};

Tensor node_graphormer(const Tensor& x, at::TensorList P, const c10::intrusive_ptr<PlanHolder>& holder, const Tensor& ws, int64_t H, int64_t tokens,
                       at::ArrayRef<double> eps) {
    on_gpu(x, "node_graphormer");
    TORCH_CHECK(x.dim() == 2 && x.is_contiguous(), "node_graphormer: x must be a contiguous [n, features]");
    TORCH_CHECK(P.size() >= 7 && (P.size() - 7) % 16 == 0, "node_graphormer takes 7 + 16 L parameter tensors");
    TORCH_CHECK(tokens == 1, "node_graphormer: one global token (its rows are the nodes', the model's are 1 .. of the sequence)");
    GraphormerDims D{};
    D.L = (int64_t)(P.size() - 7) / 16; D.n = x.size(0); D.tokens = tokens; D.N = D.n + tokens; D.F = x.size(1); D.H = H;
    TORCH_CHECK((int64_t)eps.size() == 2 * D.L + 1, "node_graphormer: 2 L + 1 values of eps");
    Wanted wanted;
    for (const Tensor& t : P) {
        same_gpu(t, x, "node_graphormer", "every parameter");
        TORCH_CHECK(t.scalar_type() == x.scalar_type(), "parameters must be GPU tensors of x's dtype");
        wanted.look(t);
    }
    same_gpu(ws, x, "node_graphormer", "the plan");
    const Tensor* q = P.data() + 3;
    TORCH_CHECK(P[0].dim() == 2 && P[0].size(0) == kWidth && P[0].size(1) == D.F && P[1].numel() == kWidth && P[2].dim() == 2 && P[2].size(0) == tokens &&
                    P[2].size(1) == kWidth, "node_graphormer: encoder shapes");
    for (int64_t i = 0; i < 16 * D.L; ++i) {
        const int64_t k = i % 16;
        TORCH_CHECK(q[i].numel() == (k >= 2 && k % 2 == 0 && k != 10 ? kWidth * kWidth : kWidth), "node_graphormer: layers are 64 wide");
    }
    q += 16 * D.L;
    D.C = q[2].size(0);
    TORCH_CHECK(q[0].numel() == kWidth && q[1].numel() == kWidth && q[2].dim() == 2 && q[2].size(1) == kWidth && D.C >= 1 && D.C <= 64 && q[3].numel() == D.C,
                "node_graphormer: 1 to 64 classes on 64 features");
    TORCH_CHECK(H == 8 || H == 4 || H == 2, "node_graphormer: 8, 4 or 2 heads");
    rows_match_plan(holder, D.N, "node_graphormer");
    wanted.look(x);
    std::vector<double> e(eps.begin(), eps.end());
    if (wanted.node()) return NodeGraphormerFn::apply(x, P, holder, ws, D, e);
    GraphormerState st;
    std::vector<Tensor> p;
    p.reserve(P.size());
    for (const Tensor& t : P) p.push_back(t.contiguous());
    st.x = x;
    c10::DeviceGuard guard(x.device());
    graphormer_forward(st, D, p, reinterpret_cast<const tgt_plan_t*>(holder->h), ws, e, false);
    return st.logp;
}

// ---------------------------------------------------------------------------------------------------------------
// graph-level Graphormer (models/graphormer_graph_level.py:309-389): node features, attention bias, layers around the dense
// attention, head; attention dropout inside the kernels, no other dropout at work
// ---------------------------------------------------------------------------------------------------------------
// params: atom, in-degree, out-degree tables, graph token; spatial table, edge table, virtual distance (, hop matrices);
// 16 per layer; gamma, beta (final norm), Wh, bh
struct GraphCall {
    bool multi_hop = false;
    int64_t max_dist = 0, H = 0;
    double p_drop = 0;
    std::vector<double> eps;
    std::vector<int64_t> seeds;
};

struct GraphBatch { Tensor x, in_degree, out_degree, spatial, edges; };      // int64, contiguous

// Bytes of bias gradients that may wait to be folded together.  Adding one to a running sum reads two, writes one and rounds (28.6 us of
// GPU time for 68 MB in bf16, the batch of 256 graphs of 129 rows, whose step waits for its host: 864 us with a running sum, 867 with
// all three kept); kept, it is read once, by the fold, and takes its memory until then.
constexpr int64_t kSideBySide = int64_t(256) << 20;

struct GraphGraphormerFn : public torch::autograd::Function<GraphGraphormerFn> {
    static constexpr int kFixed = 7;
    // rows of the buffer: s_0 .. s_{L-1}, then q, k, v, a of every layer but the last, then q, k, v of the last, whose attention
    // and everything behind it is needed at one row per graph only: a, s and s' of those rows follow
    struct Layout {
        int64_t N, b, L, ns;
        bool keep;
        Layout(int64_t N_, int64_t b_, int64_t L_, bool k) : N(N_), b(b_), L(L_), ns(k ? L_ : 1), keep(k) {}
        int64_t s(int64_t l) const { return keep ? l * N : 0; }
        int64_t a(int64_t l, int i) const { return (ns + (keep ? 4 * l : 0) + i) * N; }
        int64_t thin(int i) const { return (ns + (keep ? 4 * L - 1 : 4)) * N + i * b; }      // 0: a, 1: s, 2: s'
        int64_t rows() const { return thin(3); }
    };
    static Tensor compute(const GraphBatch& in, const Tensor& attn_bias, const std::vector<Tensor>& p, const GraphCall& c, bool keep, Tensor& rows, Tensor& lse, Tensor& bias,
                          Packed& packed) {
        const int code = dtype_code(p[0]), H = (int)c.H, d = (int)(kWidth / c.H), tables = kFixed + (c.multi_hop ? 1 : 0);
        const int64_t L = (int64_t)(p.size() - tables - 4) / 16, b = in.x.size(0), s = in.x.size(1), S = s + 1, N = b * S;
        const auto opt = p[0].options();
        void* stream = stream_of(p[0]);
        const Layout at(N, b, L, keep);
        rows = at::empty({at.rows(), kWidth}, opt);
        lse = at::empty({(keep ? (L - 1) * b * H * S : b * H * S) + b * H}, opt.dtype(at::kFloat));
        float* thin_lse = lse.data_ptr<float>() + lse.numel() - b * H;
        bias = at::empty({b, H, S, S}, opt);
        const Tensor* head = p.data() + tables + 16 * L;
        packed = Packed(p.data() + tables, L, head, code, opt, stream);
        check(tgt_graph_node_feature_fwd(in.x.data_ptr<int64_t>(), in.in_degree.data_ptr<int64_t>(), in.out_degree.data_ptr<int64_t>(), (int)in.x.size(2), p[0].data_ptr(),
                                         (int)p[0].size(0), p[1].data_ptr(), (int)p[1].size(0), p[2].data_ptr(), (int)p[2].size(0), p[3].data_ptr(), (int)b, (int)s,
                                         (int)kWidth, code, at_row(rows, 0), stream),
              "tgt_graph_node_feature_fwd");
        if (c.multi_hop)
            check(tgt_graph_attn_bias_multi_hop_fwd(attn_bias.data_ptr(), in.spatial.data_ptr<int64_t>(), in.edges.data_ptr<int64_t>(), (int)in.edges.size(3),
                                                    (int)in.edges.size(4), p[4].data_ptr(), (int)p[4].size(0), p[5].data_ptr(), (int)p[5].size(0), p[7].data_ptr(),
                                                    (int)(p[7].numel() / (H * H)), p[6].data_ptr(), (int)c.max_dist, (int)b, (int)s, H, code, bias.data_ptr(), stream),
                  "tgt_graph_attn_bias_multi_hop_fwd");
        else
            check(tgt_graph_attn_bias_fwd(attn_bias.data_ptr(), in.spatial.data_ptr<int64_t>(), in.edges.data_ptr<int64_t>(), (int)in.edges.size(3), p[4].data_ptr(),
                                          (int)p[4].size(0), p[5].data_ptr(), (int)p[5].size(0), p[6].data_ptr(), (int)b, (int)s, H, code, bias.data_ptr(), stream),
                  "tgt_graph_attn_bias_fwd");
        for (int64_t l = 0; l < L; ++l) {
            tgt_node_fwd_args a{};
            a.rows = N; a.dtype = code; a.same_bits = code == TGT_DTYPE_BF16;
            a.s_in = at_row(rows, at.s(l ? l - 1 : 0)); a.s_out = at_row(rows, at.s(l));
            if (l > 0) {
                a.attn = at_row(rows, at.a(l - 1, 3));
                a.w_post = packed.weight(6 * (l - 1)); a.v_post = packed.vec(10 * (l - 1)); a.eps_post = (float)c.eps[2 * (l - 1) + 1];
            }
            a.q = at_row(rows, at.a(l, 0)); a.k = at_row(rows, at.a(l, 1)); a.v = at_row(rows, at.a(l, 2));
            a.w_next = packed.weight(6 * l + 3); a.v_next = packed.vec(10 * l + 5); a.eps_next = (float)c.eps[2 * l];
            check(tgt_node_fwd(&a, stream), "tgt_node_fwd");
            if (l + 1 < L)
                check(tgt_dense_attn_dropout_fwd(a.q, a.k, a.v, bias.data_ptr(), (int)b, (int)S, H, d, code, (float)c.p_drop, (uint64_t)c.seeds[l], at_row(rows, at.a(l, 3)),
                                                 lse.data_ptr<float>() + (keep ? l * b * H * S : 0), stream),
                      "tgt_dense_attn_dropout_fwd");
            else
                check(tgt_dense_row0_fwd(a.q, a.k, a.v, bias.data_ptr(), a.s_out, (int)b, (int)S, H, d, code, (float)c.p_drop, (uint64_t)c.seeds[l], at_row(rows, at.thin(0)),
                                         at_row(rows, at.thin(1)), thin_lse, stream),
                      "tgt_dense_row0_fwd");
        }
        Tensor y = at::empty({b, head[2].size(0)}, opt);
        tgt_node_fwd_args a{};
        a.rows = b; a.dtype = code; a.classes = (int)head[2].size(0); a.linear = 1; a.same_bits = code == TGT_DTYPE_BF16;
        a.attn = at_row(rows, at.thin(0)); a.s_in = at_row(rows, at.thin(1)); a.s_out = at_row(rows, at.thin(2));
        a.w_post = packed.weight(6 * (L - 1)); a.v_post = packed.vec(10 * (L - 1)); a.eps_post = (float)c.eps[2 * L - 1];
        a.logp = y.data_ptr(); a.w_next = packed.weight(6 * L); a.v_next = packed.vec(10 * L); a.eps_next = (float)c.eps[2 * L];
        check(tgt_node_fwd(&a, stream), "tgt_node_fwd");
        return y;
    }
    static Tensor forward(AutogradContext* ctx, at::TensorList P, Tensor x, Tensor in_degree, Tensor out_degree, Tensor attn_bias, Tensor spatial, Tensor edges, GraphCall c) {
        std::vector<Tensor> p;
        p.reserve(P.size());
        for (const Tensor& t : P) p.push_back(t.contiguous());
        c10::DeviceGuard guard(p[0].device());
        Tensor rows, lse, bias;
        Packed packed;
        Tensor y = compute(GraphBatch{x, in_degree, out_degree, spatial, edges}, attn_bias, p, c, true, rows, lse, bias, packed);
        ctx->save_for_backward({x, in_degree, out_degree, spatial, edges, rows, lse, bias, packed.frags, p[0], p[1], p[2], p[4], p[5], c.multi_hop ? p[7] : Tensor(), p[3], p[6]});
        ctx->saved_data["multi_hop"] = c.multi_hop;
        ctx->saved_data["ints"] = std::vector<int64_t>{c.max_dist, c.H, (int64_t)p.size(), y.size(1)};
        ctx->saved_data["p"] = c.p_drop;
        ctx->saved_data["eps"] = c.eps;
        ctx->saved_data["seeds"] = c.seeds;
        return y;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        auto sv = ctx->get_saved_variables();
        const Tensor &x = sv[0], &ind = sv[1], &outd = sv[2], &spatial = sv[3], &edges = sv[4], &rows = sv[5], &lse = sv[6], &bias = sv[7], &atom = sv[9], &tin = sv[10],
                     &tout = sv[11], &sp = sv[12], &et = sv[13], &hops = sv[14], &token = sv[15], &vd = sv[16];
        const bool multi_hop = ctx->saved_data["multi_hop"].toBool();
        const auto ints = ctx->saved_data["ints"].toIntVector();
        const auto eps = ctx->saved_data["eps"].toDoubleVector();
        const auto seeds = ctx->saved_data["seeds"].toIntVector();
        const double p_drop = ctx->saved_data["p"].toDouble();
        const int tables = kFixed + (multi_hop ? 1 : 0), H = (int)ints[1], hd = (int)(kWidth / H);
        const int64_t L = (ints[2] - tables - 4) / 16, b = x.size(0), s = x.size(1), S = s + 1, N = b * S, O = ints[3];
        const int code = dtype_code(atom);
        const Layout lay(N, b, L, true);
        c10::DeviceGuard guard(atom.device());
        void* stream = stream_of(atom);
        const auto opt = atom.options(), bytes_opt = opt.dtype(at::kByte);
        const Packed packed(sv[8], (int)(6 * L + 1), code);
        std::vector<std::vector<int64_t>> shapes;
        for (const Tensor* t : {&atom, &tin, &tout, &token, &sp, &et, &vd}) shapes.push_back(t->sizes().vec());
        if (multi_hop) shapes.push_back(hops.sizes().vec());
        for (int64_t l = 0; l < L; ++l)
            for (int i = 0; i < 16; ++i) shapes.push_back(i >= 2 && i % 2 == 0 && i != 10 ? std::vector<int64_t>{kWidth, kWidth} : std::vector<int64_t>{kWidth});
        shapes.push_back({kWidth});
        shapes.push_back({kWidth});
        shapes.push_back({O, kWidth});
        shapes.push_back({O});
        FlatGrads G(shapes, opt);
        const Tensor dy = grads[0].contiguous();
        const int workers = tgt_node_bwd_workers(N), thin_workers = tgt_node_bwd_workers(b);
        Tensor work = at::empty({6 * N + 3 * b, kWidth}, opt);
        Tensor partial = at::empty({workers * (2 * L - 1) * kLayerPartial + thin_workers * (kLayerPartial + kClassPartial) + b * H}, opt.dtype(at::kFloat));
        char *g[2] = {at_row(work, 0), at_row(work, N)}, *da = at_row(work, 2 * N), *dq = at_row(work, 3 * N), *dk = at_row(work, 4 * N), *dv = at_row(work, 5 * N);
        char *thin_g = at_row(work, 6 * N), *thin_g2 = at_row(work, 6 * N + b), *thin_da = at_row(work, 6 * N + 2 * b);
        float *dvirt = partial.data_ptr<float>(), *next_partial = dvirt + b * H;
        std::vector<tgt_node_sum> sums;
        auto new_sum = [&](int n, int mats, int n_rows) -> tgt_node_sum& {
            sums.push_back(tgt_node_sum{});
            sums.back().partial = next_partial; sums.back().workers = n; sums.back().mats = mats; sums.back().rows = n_rows;
            next_partial += (int64_t)n * (mats * 4096 + (mats + 2) * 64);
            return sums.back();
        };
        {      // the head, one row per graph
            tgt_node_bwd_pre_args a{};
            a.rows = b; a.dtype = code; a.classes = (int)O; a.linear = 1; a.eps = (float)eps[2 * L];
            a.s = at_row(rows, lay.thin(2)); a.dlogp = dy.data_ptr(); a.w_back = packed.transposed(6 * L); a.v_next = packed.vec(10 * L);
            a.g_out = thin_g; a.partial = next_partial;
            tgt_node_sum& sm = new_sum(thin_workers, 1, (int)O);
            const Tensor* head = G.t.data() + tables + 16 * L;
            sm.out[0] = head[2].data_ptr(); sm.out[1] = head[3].data_ptr(); sm.out[2] = head[0].data_ptr(); sm.out[3] = head[1].data_ptr();
            check(tgt_node_bwd_pre(&a, stream), "tgt_node_bwd_pre");
        }
        // the layers share one bias: their gradients of it are added where they are folded into the tables, up to four at a time and
        // kSideBySide bytes in all; beyond that they go into a running sum as they come
        const int64_t together = multi_hop || H > 8 || edges.size(3) != 1 ? 1 : std::max<int64_t>(1, std::min<int64_t>(4, kSideBySide / (int64_t)bias.nbytes()));
        std::vector<Tensor> dbias;
        for (int64_t l = L - 1; l >= 0; --l) {
            const bool last = l == L - 1;
            const Tensor* w = G.t.data() + tables + 16 * l;
            const char *q = at_row(rows, lay.a(l, 0)), *k = at_row(rows, lay.a(l, 1)), *v = at_row(rows, lay.a(l, 2));
            tgt_node_bwd_post_args post{};
            post.rows = last ? b : N; post.dtype = code; post.same_bits = code == TGT_DTYPE_BF16; post.heads = H; post.eps = (float)eps[2 * l + 1];
            post.g_in = last ? thin_g : g[0]; post.s = at_row(rows, last ? lay.thin(1) : lay.s(l)); post.attn = at_row(rows, last ? lay.thin(0) : lay.a(l, 3));
            post.w_post = packed.weight(6 * l); post.w_back = packed.transposed(6 * l);
            post.v_post = packed.vec(10 * l); post.g_out = last ? thin_g2 : g[1]; post.d_attn = last ? thin_da : da; post.partial = next_partial;
            static const int to_post[8] = {8, 12, 14, 9, 13, 15, 10, 11}, to_pre[8] = {2, 4, 6, 3, 5, 7, 0, 1};
            tgt_node_sum& s1 = new_sum(last ? thin_workers : workers, 3, (int)kWidth);
            for (int i = 0; i < 8; ++i) s1.out[i] = w[to_post[i]].data_ptr();
            check(tgt_node_bwd_post(&post, stream), "tgt_node_bwd_post");
            if (last)
                check(tgt_dense_row0_bwd(q, k, v, bias.data_ptr(), (int)b, (int)S, H, hd, code, (float)p_drop, (uint64_t)seeds[l], post.attn,
                                         lse.data_ptr<float>() + lse.numel() - b * H, thin_da, thin_g2, dq, dk, dv, g[1], dvirt, stream),
                      "tgt_dense_row0_bwd");
            else {
                Tensor db = at::empty_like(bias);
                check(tgt_dense_attn_dropout_bwd(q, k, v, bias.data_ptr(), (int)b, (int)S, H, hd, code, (float)p_drop, (uint64_t)seeds[l], post.attn,
                                                 lse.data_ptr<float>() + l * b * H * S, da, dq, dk, dv, db.data_ptr(), stream),
                      "tgt_dense_attn_dropout_bwd");
                if ((int64_t)dbias.size() < together) dbias.push_back(db);
                else dbias.back().add_(db);
            }
            tgt_node_bwd_pre_args pre{};
            pre.rows = N; pre.dtype = code; pre.eps = (float)eps[2 * l];
            pre.dq = dq; pre.dk = dk; pre.dv = dv; pre.g_in = g[1]; pre.s = at_row(rows, lay.s(l));
            pre.w_back = packed.transposed(6 * l + 3); pre.v_next = packed.vec(10 * l + 5); pre.g_out = g[0]; pre.partial = next_partial;
            tgt_node_sum& s2 = new_sum(workers, 3, (int)kWidth);
            for (int i = 0; i < 8; ++i) s2.out[i] = w[to_pre[i]].data_ptr();
            check(tgt_node_bwd_pre(&pre, stream), "tgt_node_bwd_pre");
        }
        check(tgt_node_sums(sums.data(), (int)sums.size(), code, stream), "tgt_node_sums");
        if (dbias.empty())
            for (int i = 4; i < tables; ++i) G.t[i].zero_();      // one layer: only the virtual distance below
        else if (multi_hop) {
            const int D0 = (int)edges.size(3), md = (int)ints[0], D = md > 0 && md < D0 ? md : D0;
            const int64_t bytes = tgt_graph_attn_bias_multi_hop_bwd_workspace_bytes((int)sp.size(0), (int)et.size(0), H, D);
            Tensor ws = at::empty({bytes}, bytes_opt);
            check(tgt_graph_attn_bias_multi_hop_bwd(dbias[0].data_ptr(), spatial.data_ptr<int64_t>(), edges.data_ptr<int64_t>(), D0, (int)edges.size(4), et.data_ptr(),
                                                    (int)sp.size(0), (int)et.size(0), hops.data_ptr(), (int)(hops.numel() / (H * H)), md, (int)b, (int)s, H, code,
                                                    G.t[4].data_ptr(), G.t[5].data_ptr(), G.t[7].data_ptr(), G.t[6].data_ptr(), ws.data_ptr(), bytes, stream),
                  "tgt_graph_attn_bias_multi_hop_bwd");
        } else {
            const void* d[4] = {nullptr, nullptr, nullptr, nullptr};
            for (size_t i = 0; i < dbias.size(); ++i) d[i] = dbias[i].data_ptr();
            const int64_t bytes = tgt_graph_attn_bias_bwd_workspace_bytes((int)sp.size(0), (int)et.size(0), H);
            Tensor ws = at::empty({bytes}, bytes_opt);
            check(tgt_graph_attn_bias_bwd_sum(d, (int)dbias.size(), spatial.data_ptr<int64_t>(), edges.data_ptr<int64_t>(), (int)edges.size(3), (int)sp.size(0), (int)et.size(0),
                                              (int)b, (int)s, H, code, G.t[4].data_ptr(), G.t[5].data_ptr(), G.t[6].data_ptr(), ws.data_ptr(), bytes, stream),
                  "tgt_graph_attn_bias_bwd_sum");
        }
        check(tgt_dense_row0_virtual(dvirt, (int)b, H, code, G.t[6].data_ptr(), stream), "tgt_dense_row0_virtual");
        {
            const int64_t bytes = tgt_graph_node_feature_bwd_workspace_bytes((int)atom.size(0), (int)tin.size(0), (int)tout.size(0), (int)kWidth);
            Tensor ws = at::empty({bytes}, bytes_opt);
            check(tgt_graph_node_feature_bwd(g[0], x.data_ptr<int64_t>(), ind.data_ptr<int64_t>(), outd.data_ptr<int64_t>(), (int)x.size(2), (int)atom.size(0), (int)tin.size(0),
                                             (int)tout.size(0), (int)b, (int)s, (int)kWidth, code, G.t[0].data_ptr(), G.t[1].data_ptr(), G.t[2].data_ptr(), G.t[3].data_ptr(),
                                             ws.data_ptr(), bytes, stream),
                  "tgt_graph_node_feature_bwd");
        }
        variable_list out;
        out.reserve(G.t.size() + 7);
        for (Tensor& t : G.t) out.push_back(std::move(t));
        for (int i = 0; i < 7; ++i) out.push_back(Tensor());
        return out;
    }
};

Tensor graph_graphormer(const Tensor& x, const Tensor& in_degree, const Tensor& out_degree, const Tensor& attn_bias, const Tensor& spatial_pos, const Tensor& edge_ids,
                        at::TensorList P, bool multi_hop, int64_t max_dist, int64_t H, at::ArrayRef<double> eps, double p_drop, at::IntArrayRef seeds) {
    on_gpu(attn_bias, "graph_graphormer");
    const int64_t tables = GraphGraphormerFn::kFixed + (multi_hop ? 1 : 0);
    TORCH_CHECK((int64_t)P.size() >= tables + 4 && (P.size() - tables - 4) % 16 == 0, "graph_graphormer takes ", tables + 4, " + 16 L parameter tensors");
    const int64_t L = (int64_t)(P.size() - tables - 4) / 16;
    TORCH_CHECK((int64_t)eps.size() == 2 * L + 1 && (int64_t)seeds.size() == L, "graph_graphormer: 2 L + 1 values of eps, L seeds");
    TORCH_CHECK(H == 8 || H == 4 || H == 2, "graph_graphormer: 8, 4 or 2 heads");
    Wanted wanted;
    for (const Tensor& t : P) {
        same_gpu(t, attn_bias, "graph_graphormer", "every parameter");
        TORCH_CHECK(t.scalar_type() == P[0].scalar_type(), "graph_graphormer: parameters must be GPU tensors of one dtype");
        wanted.look(t);
    }
    same_gpu(x, attn_bias, "graph_graphormer", "x");
    same_gpu(in_degree, attn_bias, "graph_graphormer", "in_degree");
    same_gpu(out_degree, attn_bias, "graph_graphormer", "out_degree");
    same_gpu(spatial_pos, attn_bias, "graph_graphormer", "spatial_pos");
    same_gpu(edge_ids, attn_bias, "graph_graphormer", multi_hop ? "edge_input" : "attn_edge_type");
    for (int i : {0, 1, 2, 3}) TORCH_CHECK(P[i].dim() == 2 && P[i].size(1) == kWidth, "graph_graphormer: feature tables are [rows, 64]");
    for (int i : {4, 5, 6}) TORCH_CHECK(P[i].dim() == 2 && P[i].size(1) == H, "graph_graphormer: bias tables are [rows, heads]");
    TORCH_CHECK(!multi_hop || P[7].numel() % (H * H) == 0, "graph_graphormer: hop matrices");
    const Tensor* q = P.data() + tables;
    for (int64_t i = 0; i < 16 * L; ++i) {
        const int64_t k = i % 16;
        TORCH_CHECK(q[i].numel() == (k >= 2 && k % 2 == 0 && k != 10 ? kWidth * kWidth : kWidth), "graph_graphormer: layers are 64 wide");
    }
    q += 16 * L;
    TORCH_CHECK(q[0].numel() == kWidth && q[1].numel() == kWidth && q[2].dim() == 2 && q[2].size(1) == kWidth && q[2].size(0) >= 1 && q[2].size(0) <= 64 && q[3].numel() == q[2].size(0),
                "graph_graphormer: 1 to 64 outputs on 64 features");
    const int64_t b = x.size(0), s = x.size(1);
    TORCH_CHECK(x.dim() == 3 && in_degree.numel() == b * s && out_degree.numel() == b * s && attn_bias.dim() == 3 && attn_bias.size(0) == b && attn_bias.size(1) == s + 1 &&
                    attn_bias.size(2) == s + 1 && spatial_pos.dim() == 3 && spatial_pos.size(0) == b && spatial_pos.size(1) == s && spatial_pos.size(2) == s &&
                    edge_ids.dim() == (multi_hop ? 5 : 4) && edge_ids.size(0) == b && edge_ids.size(1) == s && edge_ids.size(2) == s,
                "graph_graphormer: x [b, s, F], degrees [b, s], attn_bias [b, s + 1, s + 1], spatial_pos [b, s, s], edge ids [b, s, s, ...]");
    GraphCall c;
    c.multi_hop = multi_hop; c.max_dist = max_dist; c.H = H; c.p_drop = p_drop;
    c.eps.assign(eps.begin(), eps.end());
    c.seeds.assign(seeds.begin(), seeds.end());
    const auto ids = [](const Tensor& t) { return t.to(at::kLong).contiguous(); };
    c10::DeviceGuard guard(P[0].device());
    const Tensor ab = attn_bias.to(P[0].scalar_type()).contiguous();
    if (wanted.node()) return GraphGraphormerFn::apply(P, ids(x), ids(in_degree), ids(out_degree), ab, ids(spatial_pos), ids(edge_ids), c);
    std::vector<Tensor> p;
    for (const Tensor& t : P) p.push_back(t.contiguous());
    Tensor rows, lse, bias;
    Packed packed;
    return GraphGraphormerFn::compute(GraphBatch{ids(x), ids(in_degree), ids(out_degree), ids(spatial_pos), ids(edge_ids)}, ab, p, c, false, rows, lse, bias, packed);
}

// Whether somebody waits for single gradients of these parameters: a data-parallel wrapper hooks every parameter's accumulation, to
// reduce gradients while the backward goes on.
bool gradients_watched(at::TensorList params) {
    for (const Tensor& t : params) {
        if (!t.defined() || !t.requires_grad()) continue;
        if (!torch::autograd::impl::hooks(t).empty() || torch::autograd::impl::post_acc_grad_hooks(t) != nullptr) return true;
        const auto node = torch::autograd::impl::try_get_grad_accumulator(t);
        if (node && (!node->post_hooks().empty() || !node->pre_hooks().empty())) return true;
    }
    return false;
}

}  // namespace

TORCH_LIBRARY_FRAGMENT(torchgt, m) {
    m.def("gradients_watched(Tensor[] params) -> bool");
    m.def("node_graphormer(Tensor x, Tensor[] params, __torch__.torch.classes.torchgt.PlanHolder plan, Tensor workspace, int heads, int tokens, "
          "float[] eps) -> Tensor");
    m.def("graph_graphormer(Tensor x, Tensor in_degree, Tensor out_degree, Tensor attn_bias, Tensor spatial_pos, Tensor edge_ids, Tensor[] params, "
          "bool multi_hop, int max_dist, int heads, float[] eps, float p_drop, int[] seeds) -> Tensor");
}
TORCH_LIBRARY_IMPL(torchgt, CompositeImplicitAutograd, m) {
    m.impl("gradients_watched", gradients_watched);
    m.impl("node_graphormer", node_graphormer);
    m.impl("graph_graphormer", graph_graphormer);
}
