"""The whole-model operators against the same models run layer by layer (whose kernels are compared with the oracle in
test_gpu_encoder.py): output and every parameter gradient, at the sizes where the fused kernels can go wrong - row counts around
a wave's 32 rows and a workgroup's 128 and 256, class counts around the halves of a row, odd feature widths, all head shapes.

Bars: float32 1e-5 of the largest value of the tensor, bf16 6e-2 (the layer-by-layer path rounds every intermediate tensor)."""
import copy
import ctypes
import types

import pytest
import torch

from torchgt_amd import GT, GraphLevelGraphormer, Graphormer, GraphPlan, _ext, _lib, gt
from torchgt_amd.graph_prep import fix_edge_index

pytestmark = pytest.mark.gpu
TOL = {torch.float32: 1e-5, torch.bfloat16: 6e-2}


def random_edges(n, tokens, seed, device):
    g = torch.Generator().manual_seed(seed)
    e = torch.cat([torch.randint(0, n, (2, 5 * n), generator=g), torch.arange(n).repeat(2, 1)], 1).to(device)
    return fix_edge_index(e, n) if tokens else e


def scaled(model, seed, dtype, device):
    g = torch.Generator().manual_seed(seed)
    with torch.no_grad():
        for p in model.parameters():
            if p.dim() == 1:
                p.add_(torch.randn(p.shape, generator=g) * 0.1)
            else:
                p.copy_(torch.randn(p.shape, generator=g) / p.shape[-1] ** 0.5)
    return model.to(device, dtype)


def compare(cls, model, x, plan, seed):
    """(output, input gradient, parameter gradients) of both paths"""
    w = torch.randn(x.shape[0], 64, generator=torch.Generator().manual_seed(seed)).to(x.device)
    got = []
    for fused in (True, False):
        cls.one_operator = fused
        try:
            model.zero_grad(set_to_none=True)
            xr = x.clone().requires_grad_(True)
            out = model(xr, None, plan, attn_type="sparse")
            (out.float() * w[:, :out.shape[1]]).sum().backward()
            grads = {k: p.grad for k, p in model.named_parameters() if p.grad is not None}
            got.append((out.detach(), xr.grad, grads))
            with torch.no_grad():
                assert torch.equal(model(x, None, plan, attn_type="sparse"), out)
        finally:
            cls.one_operator = True
    tol = TOL[x.dtype]
    worst = max(float(g.float().abs().max()) for g in got[1][2].values())
    (o1, x1, g1), (o0, x0, g0) = got

    def close(name, a, b, floor=0.0):
        scale = max(float(b.float().abs().max()), floor)
        err = float((a.float() - b.float()).abs().max()) / (scale or 1.0)
        assert a.shape == b.shape and err <= tol, f"{name}: {err}"

    close("output", o1, o0)
    close("input gradient", x1, x0)
    assert g1.keys() == g0.keys()
    for k in g0:
        # (a key bias moves all scores of a query alike: its gradient is rounding noise and is held to the largest gradient)
        close(k, g1[k], g0[k], floor=worst * (1.0 if k.endswith("linear_k.bias") else 1e-2))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,features,classes,heads,layers", [(1, 32, 1, 8, 1), (30, 40, 5, 4, 2), (31, 100, 33, 8, 1), (32, 64, 32, 2, 2), (126, 72, 47, 8, 1),
                                                             (127, 128, 64, 8, 2), (128, 65, 31, 4, 1), (256, 128, 40, 8, 3), (1000, 500, 47, 8, 2),
                                                             (33333, 128, 40, 8, 2)])
def test_node_graphormer_as_one_operator(cuda, dtype, n, features, classes, heads, layers):
    print(f"node_graphormer case: n={n} features={features} classes={classes} heads={heads} layers={layers} {dtype}", flush=True)
    torch.manual_seed(n)
    model = scaled(Graphormer(layers, heads, features, 64, classes, 1, 0.0, 0.0, 0.0, 64, 1), n + 1, dtype, cuda)
    x = torch.randn(n, features).to(cuda, dtype)
    plan = GraphPlan(random_edges(n, 1, n + 2, cuda), n + 1)
    assert model._one_operator(x, None, plan, None, "sparse") is not None
    compare(Graphormer, model, x, plan, n + 3)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("b,s,outputs,heads,layers,edge_type,features,p_drop", [(1, 1, 1, 8, 1, "single_hop", 1, 0.0), (3, 31, 17, 8, 4, "single_hop", 1, 0.0),
                                                                              (17, 40, 64, 4, 5, "single_hop", 1, 0.3), (5, 70, 2, 2, 2, "single_hop", 3, 0.0),
                                                                              (33, 24, 1, 8, 3, "multi_hop", 1, 0.1)])
def test_graph_graphormer_as_one_operator(cuda, dtype, b, s, outputs, heads, layers, edge_type, features, p_drop):
    """The whole graph-level model against its layers one by one: one to five layers share the bias (up to four gradients of it
    are folded into the tables side by side, one edge feature or several), outputs around the sixteen of a pass."""
    print(f"graph_graphormer case: b={b} s={s} outputs={outputs} heads={heads} layers={layers} {edge_type} {dtype}", flush=True)
    torch.manual_seed(b)
    model = GraphLevelGraphormer(layers, heads, 64, 0.0, 0.0, 64, "ZINC", edge_type, 5, p_drop, outputs)
    model = scaled(model, b + 1, dtype, cuda)
    with torch.no_grad():      # queries of a size whose products mean something in bf16 (the layer multiplies them by sqrt(d))
        for layer in model.layers:
            layer.self_attention.linear_q.weight.mul_(0.2)
    g = torch.Generator().manual_seed(b + 2)
    ids = lambda hi, *shape: torch.randint(0, hi, shape, generator=g).to(cuda)
    batch = types.SimpleNamespace(x=ids(64, b, s, 1), in_degree=ids(64, b, s), out_degree=ids(64, b, s), attn_bias=torch.zeros(b, s + 1, s + 1, device=cuda, dtype=dtype),
                                  spatial_pos=ids(40, b, s, s), attn_edge_type=ids(64, b, s, s, features), edge_input=ids(64, b, s, s, 5, features))
    w = torch.randn(b, outputs, generator=g).to(cuda)
    got = []
    for fused in (True, False):
        model.one_operator = fused
        assert (model._one_operator(batch) is not None) == fused
        model.zero_grad(set_to_none=True)
        torch.manual_seed(7)
        out = model(batch)
        (out.float() * w).sum().backward()
        got.append((out.detach(), {k: p.grad for k, p in model.named_parameters() if p.grad is not None}))
    (o1, g1), (o0, g0) = got
    tol = (3 if dtype == torch.float32 else 2) * TOL[dtype]      # float32: the tables are summed with atomics; bf16: up to five layers of rounding on both sides
    assert float((o1.float() - o0.float()).abs().max()) <= tol * float(o0.float().abs().max())
    assert g1.keys() == g0.keys()
    worst = max(float(v.float().abs().max()) for v in g0.values())
    for k in g0:
        floor = worst * (1.0 if k.endswith("linear_k.bias") else 1e-2)
        err = float((g1[k].float() - g0[k].float()).abs().max()) / max(float(g0[k].float().abs().max()), floor)
        assert err <= tol, f"{k}: {err}"


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("kind,n,features,classes,heads,hidden,ffn,layers", [("gt", 1, 32, 3, 8, 128, 64, 1), ("gt", 999, 100, 47, 4, 32, 64, 3), ("gt", 3000, 51, 40, 8, 128, 128, 2),
                                                                          ("graphormer", 1, 32, 3, 8, 128, 128, 1), ("graphormer", 999, 100, 47, 8, 128, 128, 3),
                                                                          ("graphormer", 777, 64, 65, 4, 64, 64, 2), ("graphormer", 500, 51, 40, 4, 64, 96, 2)])
def test_other_widths_as_one_operator(cuda, dtype, kind, n, features, classes, heads, hidden, ffn, layers):
    """The models the fused kernels do not have: the same kernels in the same order as step by step, so the same bits."""
    print(f"layered case: {kind} n={n} features={features} classes={classes} heads={heads} hidden={hidden} ffn={ffn} {dtype}", flush=True)
    torch.manual_seed(n)
    cls, tokens = (GT, 0) if kind == "gt" else (Graphormer, 1)
    model = scaled(cls(layers, heads, features, hidden, classes, 1, 0.0, 0.0, 0.0, ffn, tokens), n + 1, dtype, cuda)
    x = torch.randn(n, features).to(cuda, dtype)
    plan = GraphPlan(random_edges(n, tokens, n + 2, cuda), n + tokens)
    w = torch.randn(n, classes, generator=torch.Generator().manual_seed(3)).to(cuda)
    got = []
    for one in (True, False):
        model.one_operator = one
        model.zero_grad(set_to_none=True)
        xr = x.clone().requires_grad_(True)
        out = model(xr, None, plan, attn_type="sparse")
        assert (type(out.grad_fn).__name__ == "LogSoftmaxBackward0") != one
        (out.float() * w).sum().backward()
        got.append([out.detach(), xr.grad] + [p.grad for p in model.parameters() if p.grad is not None])
        with torch.no_grad():
            assert torch.equal(model(x, None, plan, attn_type="sparse"), out)
    assert len(got[0]) == len(got[1])
    for i, (a, b) in enumerate(zip(*got)):
        assert torch.equal(a, b), (i, float((a.float() - b.float()).abs().max()))


@pytest.mark.parametrize("n,features,classes,heads,layers", [(1, 32, 3, 8, 1), (31, 64, 8, 4, 2), (32, 100, 47, 8, 1), (129, 51, 40, 2, 3), (256, 64, 16, 8, 2), (4097, 128, 40, 8, 4),
                                                             (40000, 64, 5, 8, 2)])
def test_gt_on_fused_layers(cuda, n, features, classes, heads, layers):
    """float32 against the kernels step by step; bf16, where a ReLU's input of nearly 0 may change its side, by how far both are from float32"""
    print(f"fused gt case: n={n} features={features} classes={classes} heads={heads} layers={layers}", flush=True)
    torch.manual_seed(n)
    model = scaled(GT(layers, heads, features, 64, classes, 1, 0.0, 0.0, 0.0, 64, 0), n + 1, torch.bfloat16, cuda)
    x, plan = torch.randn(n, features).to(cuda, torch.bfloat16), GraphPlan(random_edges(n, 0, n + 2, cuda), n)
    exact = copy.deepcopy(model).float()
    compare(GT, exact, x.float(), plan, n + 3)
    w = torch.randn(n, classes, generator=torch.Generator().manual_seed(n + 4)).to(cuda)
    got = []
    for m, fused in ((exact, False), (model, True), (model, False)):
        GT.one_operator = fused
        try:
            m.zero_grad(set_to_none=True)
            xr = x.to(next(m.parameters()).dtype).requires_grad_(True)
            out = m(xr, None, plan, attn_type="sparse")
            (out.float() * w).sum().backward()
            got.append([t.float() for t in (out.detach(), xr.grad, torch.cat([p.grad.flatten() for p in m.parameters() if p.grad is not None]))])
        finally:
            GT.one_operator = True
    for name, f32, one, steps in zip(("output", "input gradient", "parameter gradients"), *got):
        off, most = float((one - f32).norm() / f32.norm()), float((steps - f32).norm() / f32.norm())
        assert off <= 1.1 * most + 2e-3, f"{name}: {off}, step by step {most}"


@pytest.mark.parametrize("n,heads", [(15, 8), (16, 4), (17, 2), (64, 2), (65, 4), (16383, 8), (16384, 4), (32767, 2), (32768, 8), (40000, 4), (49152, 2), (49153, 8), (65535, 4), (65537, 2)])
def test_rows_beside_the_lines_between_variants(cuda, n, heads):
    """Sixteen or thirty-two rows per wave, 64 or 128 nodes per group (256 CUs: 16384, 32768, 49152 and 65536 rows), beside their edges"""
    for dtype in (torch.float32, torch.bfloat16):
        print(f"rows beside the lines: n={n} heads={heads} {dtype}", flush=True)
        model = scaled(Graphormer(1, heads, 32, 64, 5, 1, 0.0, 0.0, 0.0, 64, 1), n, dtype, cuda)
        x = torch.randn(n - 1, 32, generator=torch.Generator().manual_seed(n)).to(cuda, dtype)      # (one more row: the global token)
        compare(Graphormer, model, x, GraphPlan(random_edges(n - 1, 1, n + 2, cuda), n), n + 3)
    if n < 1000:
        return test_gt_on_fused_layers(cuda, n, 32, 5, heads, 1)
    # GT: among 128 n normal inputs of a ReLU those within rounding (1e-7) of 0 change their side between the two ways of summing, one for
    # 40 K nodes and as many in the readout; each moves one of 128 (32) features of one node, 1 / sqrt(128 n) (1 / sqrt(32 n)) of a
    # gradient's norm.  At 65 K nodes two of either kind, all in the same direction, are 0.5 / sqrt(n); the bar is 0.7 / sqrt(n), a
    # single row gone wrong would be 1 / sqrt(n).  The output is continuous.
    for dtype in (torch.float32, torch.bfloat16):
        model = scaled(GT(1, heads, 32, 64, 5, 1, 0.0, 0.0, 0.0, 64, 0), n, dtype, cuda)
        x, plan = torch.randn(n, 32, generator=torch.Generator().manual_seed(n)).to(cuda, dtype), GraphPlan(random_edges(n, 0, n + 2, cuda), n)
        w = torch.randn(n, 5, generator=torch.Generator().manual_seed(n + 4)).to(cuda)
        got = []
        for fused in (True, False):
            GT.one_operator = fused
            try:
                model.zero_grad(set_to_none=True)
                xr = x.clone().requires_grad_(True)
                out = model(xr, None, plan, attn_type="sparse")
                (out.float() * w).sum().backward()
                got.append([t.double() for t in [out.detach(), xr.grad] + [p.grad for p in model.parameters() if p.grad is not None]])
            finally:
                GT.one_operator = True
        off = [float((a - b).norm() / b.norm().clamp(min=1e-30)) for a, b in zip(*got)]
        names = ["output", "input gradient"] + [k for k, p in model.named_parameters() if p.grad is not None]
        for name, o in zip(names, off):
            if not name.endswith("linear_k.bias"):      # (rounding noise: it moves all scores of a query alike)
                assert o <= (2e-2 if dtype == torch.bfloat16 else 1e-6 if name == "output" else (2 * n) ** -0.5), f"{name}: {o}"


@pytest.mark.parametrize("n,heads", [(65536, 8), (65537, 4), (81920, 2), (81921, 8), (131072, 4), (131073, 8), (163841, 2)])
def test_rows_beside_the_rounds_of_a_forward(cuda, n, heads):
    """Sixteen or thirty-two rows per wave by the rounds they take: 65536, 81920 and 131072 rows each on 256 CUs"""
    for dtype in (torch.float32, torch.bfloat16):
        print(f"rows beside the rounds: n={n} heads={heads} {dtype}", flush=True)
        model = scaled(Graphormer(1, heads, 32, 64, 5, 1, 0.0, 0.0, 0.0, 64, 1), n, dtype, cuda)
        x = torch.randn(n - 1, 32, generator=torch.Generator().manual_seed(n)).to(cuda, dtype)      # (one more row: the global token)
        compare(Graphormer, model, x, GraphPlan(random_edges(n - 1, 1, n + 2, cuda), n), n + 3)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,heads", [(17, 2), (65, 4), (1000, 8), (16383, 8), (16385, 4), (32767, 2), (40000, 4), (65537, 2)])
def test_gt_gradients_where_no_relu_changes_its_side(cuda, monkeypatch, dtype, n, heads):
    """The rows beside the lines between variants once more: weights in front of a ReLU are small beside its biases of +-2, so its inputs keep their sign
    (2 against at most 0.2 times ten standard deviations) and the two ways of running the model agree to rounding in every gradient, and in the output and the
    input gradient in every element: a row that is lost or another's is off by what a typical element is, a fifth of the largest or more"""
    print(f"gt without ReLUs near 0: n={n} heads={heads} {dtype}", flush=True)
    model = scaled(GT(2, heads, 32, 64, 5, 1, 0.0, 0.0, 0.0, 64, 0), n, dtype, cuda)
    relus = [layer.FFN_layer1 for layer in model.layers] + list(model.MLP_layer.FC_layers[:2])
    with torch.no_grad():
        for linear in relus:
            linear.weight.mul_(0.1)
            linear.bias.copy_(torch.where(torch.arange(linear.bias.numel(), device=cuda) % 3 == 2, -2.0, 2.0))
    seen, relu = [], gt.ReluFunction.apply
    x = torch.randn(n, 32, generator=torch.Generator().manual_seed(n)).to(cuda, dtype)
    plan = GraphPlan(random_edges(n, 0, n + 2, cuda), n)
    with monkeypatch.context() as patch:
        patch.setattr(gt.ReluFunction, "apply", staticmethod(lambda u: seen.append(float(u.detach().abs().min())) or relu(u)))
        patch.setattr(GT, "one_operator", False)
        model(x, None, plan, attn_type="sparse")
    assert len(seen) == len(relus) and min(seen) > 0.2 and model._one_operator(x, plan, "sparse") is not None
    compare(GT, model, x, plan, n + 3)


class NodeFwdArgs(ctypes.Structure):      # tgt_node_fwd_args
    _fields_ = [("rows", ctypes.c_int64)] + [(k, ctypes.c_int32) for k in ("dtype", "tokens", "classes", "linear", "same_bits")] + \
        [(k, ctypes.c_float) for k in ("eps_post", "eps_next")] + \
        [(k, ctypes.c_void_p) for k in ("attn", "s_in", "token", "s_out", "w_post", "w_next", "v_post", "v_next", "q", "k", "v", "logp")]


@pytest.mark.parametrize("scale", [0.3, 1.0, 2.0])
def test_gelu_of_the_fused_layers_is_as_exact_as_the_error_function(cuda, scale):
    """The activation of the fused kernels against 64 bits, next to 0.5 u (1 + erff(u / sqrt 2)) of the separate kernel.  With zero rows,
    W1 = 0 and W2 = 1 the layer's output is the activation of its bias b1, 64 values a launch, behind a product with W2 that rounds a
    little of its own: the separate kernel's values go through the same product."""
    launches, L = 1024, _lib.lib()
    u = (torch.randn(launches, 64, generator=torch.Generator().manual_seed(3)) * scale).to(cuda)
    zero, one = torch.zeros(64, 64, device=cuda), torch.eye(64, device=cuda)
    frags = torch.empty(L.tgt_node_frag_bytes(3, _lib.DTYPE_F32), dtype=torch.uint8, device=cuda)
    vecs, stream = torch.zeros(5, 64, device=cuda), torch.cuda.current_stream(cuda).cuda_stream      # bo, gamma, beta, b1, b2
    mats, ld = (ctypes.c_void_p * 3)(zero.data_ptr(), zero.data_ptr(), one.data_ptr()), (ctypes.c_int * 3)(64, 64, 64)
    rows, lens, packed = (ctypes.c_void_p * 5)(*[vecs[i].data_ptr() for i in range(5)]), (ctypes.c_int * 5)(*[64] * 5), torch.empty_like(vecs)
    _lib.check(L.tgt_node_pack(ctypes.addressof(mats), ctypes.addressof(ld), ctypes.addressof(ld), 3, ctypes.addressof(rows), ctypes.addressof(lens), 5,
                               _lib.DTYPE_F32, frags.data_ptr(), packed.data_ptr(), stream))
    fused = torch.empty_like(u)
    for i in range(launches):
        vecs[3] = u[i]
        args = NodeFwdArgs(rows=1, dtype=_lib.DTYPE_F32, eps_post=1e-5, attn=zero.data_ptr(), s_in=zero.data_ptr(), s_out=fused[i].data_ptr(), w_post=frags.data_ptr(),
                           v_post=vecs.data_ptr())
        _lib.check(L.tgt_node_fwd(ctypes.addressof(args), stream))
    exact = 0.5 * u.double() * torch.special.erfc(-u.double() * 2 ** -0.5)
    rms = lambda t: float((t.double() - exact).pow(2).mean().sqrt())
    (separate,) = _ext.op("linear")(_ext.op("gelu")(u), [one], [zero[0]])
    print(f"gelu, u ~ N(0, {scale}): rms error {rms(fused):.3e}, of the separate kernel {rms(separate):.3e}", flush=True)
    assert rms(fused) <= rms(separate) and float((fused - exact).abs().max()) <= 5e-7


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,classes,layers", [(1, 1, 1), (63, 64, 3), (64, 5, 2), (65, 7, 3), (127, 3, 2), (128, 40, 2), (16384, 9, 2), (16386, 9, 3), (32769, 4, 2)])
def test_both_sides_of_an_attention_in_one_launch(cuda, dtype, n, classes, layers):
    """The part in front of an attention and the part behind the one before it as one launch (groups of 64 and 128 nodes that end inside, several
    groups per workgroup), against the layers one by one"""
    print(f"both sides: n={n} classes={classes} layers={layers} {dtype}", flush=True)
    model = scaled(Graphormer(layers, 8, 40, 64, classes, 1, 0.0, 0.0, 0.0, 64, 1), n, dtype, cuda)
    x = torch.randn(n, 40, generator=torch.Generator().manual_seed(n)).to(cuda, dtype)
    compare(Graphormer, model, x, GraphPlan(random_edges(n, 1, n + 2, cuda), n + 1), n + 3)


class NodeBwdPreArgs(ctypes.Structure):      # tgt_node_bwd_pre_args
    _fields_ = [("rows", ctypes.c_int64)] + [(k, ctypes.c_int32) for k in ("dtype", "tokens", "classes", "linear")] + [("eps", ctypes.c_float)] + \
        [(k, ctypes.c_void_p) for k in ("dq", "dk", "dv", "g_in", "s", "dlogp", "logp", "w_back", "v_next", "g_out", "d_token", "partial")]


class NodeBwdPostArgs(ctypes.Structure):      # tgt_node_bwd_post_args
    _fields_ = [("rows", ctypes.c_int64)] + [(k, ctypes.c_int32) for k in ("dtype", "heads", "same_bits")] + [("eps", ctypes.c_float)] + \
        [(k, ctypes.c_void_p) for k in ("g_in", "s", "attn", "w_post", "w_back", "v_post", "Z", "g_out", "d_attn", "nd", "partial")]


@pytest.mark.parametrize("n", [32768, 32769, 33024, 49151, 49152, 49153, 131073, 147456, 147457])
def test_backward_of_many_rows_is_that_of_its_parts(cuda, n):
    """bf16 in groups of 192 nodes (32769 to 49152 and 131073 to 147456 rows on 256 CUs) and beside them: every row as in calls of at most 8000 rows (groups of 64), bit
    for bit, and the partial sums add up to theirs.  Bar of the sums: their float32 rounding, some 2^-24 of a sum's terms; a row that is lost, or counted
    twice, is 1 / sqrt(n) of a sum or more."""
    print(f"backward in parts: n={n}", flush=True)
    L, g, st = _lib.lib(), torch.Generator(device=cuda).manual_seed(n), torch.cuda.current_stream(cuda).cuda_stream
    rand = lambda *s: torch.randn(s, generator=g, device=cuda)
    weights, values, vecs = [(rand(64, 64) / 8).bfloat16() for _ in range(3)], (rand(5, 64) / 4).bfloat16(), torch.empty(5, 64, device=cuda)
    frags = torch.empty(L.tgt_node_frag_bytes(3, _lib.DTYPE_BF16), dtype=torch.uint8, device=cuda)
    back = frags.data_ptr() + frags.numel() // 2
    mats, ld = (ctypes.c_void_p * 3)(*[w.data_ptr() for w in weights]), (ctypes.c_int * 3)(64, 64, 64)
    of_vecs, lens = (ctypes.c_void_p * 5)(*[values[i].data_ptr() for i in range(5)]), (ctypes.c_int * 5)(*[64] * 5)
    _lib.check(L.tgt_node_pack(ctypes.addressof(mats), ctypes.addressof(ld), ctypes.addressof(ld), 3, ctypes.addressof(of_vecs), ctypes.addressof(lens), 5, _lib.DTYPE_BF16,
                               frags.data_ptr(), vecs.data_ptr(), st))
    rows = {k: rand(n, 64).bfloat16() for k in ("dq", "dk", "dv", "g_in", "s", "attn")}
    rows["logp"], rows["dlogp"] = torch.log_softmax(rand(n, 40), 1).bfloat16(), rand(n, 40).bfloat16()
    Z = rand(n, 8).abs() + 1

    def run(lo, hi):
        at = {k: t[lo:hi].data_ptr() for k, t in rows.items()}
        workers = L.tgt_node_bwd_workers(hi - lo)
        out = {k: torch.empty(hi - lo, 64, dtype=torch.bfloat16, device=cuda) for k in ("pre", "plain", "classes", "post", "da", "parts", "da_parts")}
        nd, sums = torch.empty(hi - lo, 8, 2, device=cuda), [torch.full((workers, m * 4096 + (m + 2) * 64), float("nan"), device=cuda) for m in (3, 3, 1, 3, 3)]
        qkv = {k: at[k] for k in ("dq", "dk", "dv", "g_in")}
        for g_out, s, more in (("pre", sums[0], dict(qkv, v_next=vecs.data_ptr())), ("plain", sums[1], qkv),      # (without LayerNorm: GT)
                               ("classes", sums[2], dict(dlogp=at["dlogp"], logp=at["logp"], classes=40, v_next=vecs.data_ptr()))):
            pre = NodeBwdPreArgs(rows=hi - lo, dtype=_lib.DTYPE_BF16, eps=1e-5, s=at["s"], w_back=back, g_out=out[g_out].data_ptr(), partial=s.data_ptr(), **more)
            _lib.check(L.tgt_node_bwd_pre(ctypes.addressof(pre), st))
        for same, g_out, da, s in ((1, "post", "da", sums[3]), (0, "parts", "da_parts", sums[4])):
            post = NodeBwdPostArgs(rows=hi - lo, dtype=_lib.DTYPE_BF16, heads=8, same_bits=same, eps=1e-5, g_in=at["g_in"], s=at["s"], attn=at["attn"], w_post=frags.data_ptr(),
                                   w_back=back, v_post=vecs.data_ptr(), Z=Z[lo:hi].data_ptr(), g_out=out[g_out].data_ptr(), d_attn=out[da].data_ptr(), nd=nd.data_ptr(),
                                   partial=s.data_ptr())
            _lib.check(L.tgt_node_bwd_post(ctypes.addressof(post), st))
        return [*out.values(), nd], [s.double().sum(0) for s in sums]

    whole, sums = run(0, n)
    parts = [run(lo, min(lo + 8000, n)) for lo in range(0, n, 8000)]
    for i, t in enumerate(whole):
        assert torch.equal(t, torch.cat([p[0][i] for p in parts])), i
    for i, t in enumerate(sums):
        want = sum(p[1][i] for p in parts)
        sizes = [4096] * (t.numel() // 4096) + [64] * (t.numel() % 4096 // 64)
        for a, b in zip(t.split(sizes), want.split(sizes)):
            assert float((a - b).norm()) <= 1e-5 * float(b.norm())


class NodeSum(ctypes.Structure):      # tgt_node_sum
    _fields_ = [("partial", ctypes.c_void_p)] + [(k, ctypes.c_int32) for k in ("workers", "mats", "rows", "ld")] + [("out", ctypes.c_void_p * 8)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("count,features,outputs,workers", [(1, 1, 64, 1), (9, 128, 64, 250), (26, 500, 64, 17), (27, 51, 64, 512), (3, 100, 40, 33)])
def test_sums_of_a_linear_beside_the_layers(cuda, dtype, count, features, outputs, workers):
    """The same bits as the two launches: sums of more elements than a layer's and of fewer, more descriptors than a launch takes, and elements that
    are no multiple of 64 (a launch of their own)"""
    print(f"sums together: count={count} features={features} outputs={outputs} workers={workers} {dtype}", flush=True)
    g, L, st = torch.Generator(device=cuda).manual_seed(count), _lib.lib(), torch.cuda.current_stream(cuda).cuda_stream
    code = _lib.DTYPE_F32 if dtype == torch.float32 else _lib.DTYPE_BF16
    partials = [torch.randn(max(1, workers // 2), 3 * 4096 + 5 * 64, generator=g, device=cuda) for _ in range(count)]
    n = outputs * features + outputs
    of_linear = torch.randn(workers, n, generator=g, device=cuda)
    outs = []
    for together in (False, True):
        layer = [[torch.full((s,), float("nan"), dtype=dtype, device=cuda) for s in (4096, 4096, 4096, 64, 64, 64, 64, 64)] for _ in range(count)]
        W, b = torch.full((n - outputs,), float("nan"), dtype=dtype, device=cuda), torch.full((outputs,), float("nan"), dtype=dtype, device=cuda)
        sums = (NodeSum * count)(*[NodeSum(partial=p.data_ptr(), workers=p.shape[0], mats=3, rows=64, ld=0, out=(ctypes.c_void_p * 8)(*[t.data_ptr() for t in o]))
                                   for p, o in zip(partials, layer)])
        desc = _lib.ReduceDesc(partial=of_linear.data_ptr(), workers=workers, n=n, n_out=2)
        desc.out[0], desc.out[1], desc.begin[1] = W.data_ptr(), b.data_ptr(), n - outputs
        if together:
            _lib.check(L.tgt_node_sums_and_reduce(ctypes.addressof(sums), count, ctypes.addressof(desc), code, st))
        else:
            _lib.check(L.tgt_node_sums(ctypes.addressof(sums), count, code, st))
            _lib.check(L.tgt_reduce_partials(ctypes.addressof(desc), 1, code, st))
        outs.append([t for o in layer for t in o] + [W, b])
    for x, y in zip(*outs):
        assert torch.equal(x, y) and not x.isnan().any()
