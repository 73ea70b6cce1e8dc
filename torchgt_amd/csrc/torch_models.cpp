// Whole models as one operator and one autograd node each, over the fused per-node kernels (node_layer.hip) and the
// attention: between Python and the kernels of a step there is one call forward and one backward.
//
//   torchgt::node_graphormer(x, params[7 + 16 L], plan holder, workspace, heads, tokens, eps[2 L + 1]) -> log-probabilities
//
// A step's intermediate rows live in one allocation, its parameter gradients in another: with some seventy parameters the
// host's time for tensors of their own would be longer than the kernels of a small graph take.
#include "torch_common.h"

namespace {

using namespace tgt_torch;

constexpr int64_t kWidth = 64;

// A tensor of the given sizes on `base`'s memory from element `offset` (no dispatch, no autograd view: base is a plain
// buffer made here)
Tensor part_of(const Tensor& base, int64_t offset, at::IntArrayRef sizes) {
    auto impl = c10::make_intrusive<c10::TensorImpl>(c10::Storage(base.storage()), base.unsafeGetTensorImpl()->key_set(), base.dtype());
    impl->set_storage_offset(base.storage_offset() + offset);
    impl->set_sizes_contiguous(sizes);
    return Tensor(std::move(impl));
}
char* at_row(const Tensor& buf, int64_t row) { return static_cast<char*>(buf.data_ptr()) + row * kWidth * buf.element_size(); }
int64_t rounded(int64_t n) { return (n + 15) / 16 * 16; }      // parameter gradients start on their own 16 elements

// gradient buffers of a list of shapes in one allocation
struct FlatGrads {
    Tensor flat;
    std::vector<Tensor> t;
    FlatGrads(const std::vector<std::vector<int64_t>>& shapes, const at::TensorOptions& opt) {
        int64_t total = 0;
        std::vector<int64_t> off;
        for (const auto& s : shapes) {
            off.push_back(total);
            int64_t n = 1;
            for (int64_t d : s) n *= d;
            total += rounded(n);
        }
        flat = at::empty({total}, opt);
        t.reserve(shapes.size());
        for (size_t i = 0; i < shapes.size(); ++i) t.push_back(part_of(flat, off[i], shapes[i]));
    }
};

// Packed parameters of the layers: fragments of six weights per layer (Wo, W1, W2, Wq, Wk, Wv), then the classes'; vectors
// per layer (bo, gamma2, beta2, b1, b2; gamma1, beta1, bq, bk, bv), then (gamma, beta, bh) of the classes.
// Order of a layer's parameters: gamma1, beta1, Wq, bq, Wk, bk, Wv, bv, Wo, bo, gamma2, beta2, W1, b1, W2, b2.
struct Packed {
    Tensor frags, vecs;
    int64_t unit = 0;
    int mats = 0;
    Packed() = default;
    // layers: first of their 16 L parameters; classes: gamma, beta, Wh, bh or nullptr
    Packed(const Tensor* layers, int64_t L, const Tensor* classes, int code, const at::TensorOptions& opt, void* stream) {
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
        check(tgt_node_pack(m.data(), ld.data(), rows.data(), mats, v.data(), len.data(), (int)v.size(), code, frags.data_ptr(),
                            reinterpret_cast<float*>(static_cast<char*>(frags.data_ptr()) + bytes), stream),
              "tgt_node_pack");
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
    st.packed = Packed(p.data() + 3, L, p.data() + 3 + 16 * L, code, opt, stream);
    auto s_row = [&](int64_t l) { return at_row(st.rows, keep ? l * N : 0); };
    auto a_row = [&](int64_t l, int i) { return at_row(st.rows, (ns + (keep ? 4 * l : 0) + i) * N); };
    {
        const void *W[1] = {p[0].data_ptr()}, *B[1] = {p[1].data_ptr()};
        void* Y[1] = {at_row(st.rows, D.tokens)};
        check(tgt_linear_fwd(x.data_ptr(), W, B, Y, 1, D.n, (int)x.size(1), (int)kWidth, code, stream), "tgt_linear_fwd");
    }
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
        {
            tgt_node_bwd_pre_args a{};
            a.rows = N; a.dtype = code; a.tokens = (int)D.tokens; a.classes = (int)D.C; a.eps = (float)eps[2 * L];
            a.s = at_row(rows, L * N); a.dlogp = dlogp.data_ptr(); a.logp = logp.data_ptr();
            a.w_back = packed.transposed(6 * L); a.v_next = packed.vec(10 * L); a.g_out = g[0]; a.partial = next_partial;
            tgt_node_sum& s = new_sum(1, (int)D.C);
            const Tensor* c = &G.t[3 + 16 * L];
            s.out[0] = c[2].data_ptr(); s.out[1] = c[3].data_ptr(); s.out[2] = c[0].data_ptr(); s.out[3] = c[1].data_ptr();
            check(tgt_node_bwd_pre(&a, stream), "tgt_node_bwd_pre");
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
            check(tgt_node_bwd_post(&b, stream), "tgt_node_bwd_post");
            check(tgt_sparse_attn_bwd_from_nd(plan, q, k, v, (int)H, (int)(kWidth / H), code, da, dq, dk, dvr, ws.data_ptr(), ws.numel(), stream),
                  "tgt_sparse_attn_bwd_from_nd");
            tgt_node_bwd_pre_args a{};
            a.rows = N; a.dtype = code; a.tokens = (int)D.tokens; a.eps = (float)eps[2 * l];
            a.dq = dq; a.dk = dk; a.dv = dvr; a.g_in = g[1]; a.s = at_row(rows, l * N);
            a.w_back = packed.transposed(6 * l + 3); a.v_next = packed.vec(10 * l + 5); a.g_out = g[0]; a.partial = next_partial;
            a.d_token = l == 0 && D.tokens ? G.t[2].data_ptr() : nullptr;
            tgt_node_sum& s2 = new_sum(3, (int)kWidth);
            for (int i = 0; i < 8; ++i) s2.out[i] = w[pre[i]].data_ptr();
            check(tgt_node_bwd_pre(&a, stream), "tgt_node_bwd_pre");
        }
        check(tgt_node_sums(sums.data(), (int)sums.size(), code, stream), "tgt_node_sums");
        Tensor dx;
        {
            if (ctx->needs_input_grad(0)) dx = at::empty_like(x);
            const void *W[1] = {Wn.data_ptr()}, *DY[1] = {g[0] + D.tokens * kWidth * x.element_size()};
            void *DW[1] = {G.t[0].data_ptr()}, *DB[1] = {G.t[1].data_ptr()};
            const int64_t bytes = tgt_linear_bwd_workspace_bytes(1, (int)x.size(1), (int)kWidth);
            Tensor lws = at::empty({bytes}, x.options().dtype(at::kByte));
            check(tgt_linear_bwd(x.data_ptr(), W, DY, 1, D.n, (int)x.size(1), (int)kWidth, code, dx.defined() ? dx.data_ptr() : nullptr, DW, DB,
                                 lws.data_ptr(), bytes, stream),
                  "tgt_linear_bwd");
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
    GraphormerDims D{};
    D.L = (int64_t)(P.size() - 7) / 16; D.n = x.size(0); D.tokens = tokens; D.N = D.n + tokens; D.F = x.size(1); D.H = H;
    TORCH_CHECK((int64_t)eps.size() == 2 * D.L + 1, "node_graphormer: 2 L + 1 values of eps");
    bool train = false;
    for (const Tensor& t : P) {
        TORCH_CHECK(t.defined() && t.is_cuda() && t.scalar_type() == x.scalar_type(), "parameters must be GPU tensors of x's dtype");
        train = train || t.requires_grad();
    }
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
    train = at::GradMode::is_enabled() && (train || x.requires_grad());
    std::vector<double> e(eps.begin(), eps.end());
    if (train) return NodeGraphormerFn::apply(x, P, holder, ws, D, e);
    GraphormerState st;
    std::vector<Tensor> p;
    p.reserve(P.size());
    for (const Tensor& t : P) p.push_back(t.contiguous());
    st.x = x;
    c10::DeviceGuard guard(x.device());
    graphormer_forward(st, D, p, reinterpret_cast<const tgt_plan_t*>(holder->h), ws, e, false);
    return st.logp;
}

}  // namespace

TORCH_LIBRARY_FRAGMENT(torchgt, m) {
    m.def("node_graphormer(Tensor x, Tensor[] params, __torch__.torch.classes.torchgt.PlanHolder plan, Tensor workspace, int heads, int tokens, "
          "float[] eps) -> Tensor");
}
TORCH_LIBRARY_IMPL(torchgt, CompositeImplicitAutograd, m) { m.impl("node_graphormer", node_graphormer); }
