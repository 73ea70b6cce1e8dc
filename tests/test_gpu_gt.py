"""GPU parity of the node-level GT model (models/gt_dist_node_level.py) and its ReLU kernel with the oracle.
ReLU is exact.  The model: max|a - b| / max|b| against float64 on the same inputs, float32 1e-5 on the
log-probabilities and on every parameter gradient;
bf16 three times the single-kernel bar of 2e-2 on the output.
"""
import ctypes

import numpy as np
import pytest
import torch

from oracle import gt as ogt
from torchgt_amd import _lib, workloads
from torchgt_amd.gt import _DT, GT, ReluFunction
from torchgt_amd.multi_head_attention import LinearFunction

pytestmark = pytest.mark.gpu


def err(a, b):
    a, b = a.detach().double().cpu(), b.detach().double().cpu()
    assert a.shape == b.shape, (a.shape, b.shape)
    denom = b.abs().max().item()
    return (a - b).abs().max().item() / (denom if denom > 0 else 1.0)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_relu_forward_backward_is_exact(cuda, dtype):
    g = torch.Generator().manual_seed(0)
    for n in (8, 4096, 100_000 * 8):
        u = torch.randn(n, generator=g).to(dtype)
        u[::7] = 0
        dh = torch.randn(n, generator=g).to(dtype)
        uc = u.to(cuda).requires_grad_(True)
        h = ReluFunction.apply(uc)
        (du,) = torch.autograd.grad(h, uc, dh.to(cuda))
        assert torch.equal(h.cpu(), torch.relu(u))
        assert torch.equal(du.cpu(), torch.where(u > 0, dh, torch.zeros_like(dh)))
    L = _lib.lib()
    assert L.tgt_relu_fwd(None, 3, 0, None, None) == _lib.ERR_UNSUPPORTED       # not a multiple of the vector width
    assert L.tgt_relu_fwd(None, 8, 0, None, None) == _lib.ERR_INVALID_ARG


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_relu_keeps_nan_as_torch_does(cuda, dtype):
    """F.relu and its backward: a NaN stays one, its slope is 1; an infinity stays or becomes 0"""
    u = torch.randn(256, generator=torch.Generator().manual_seed(1)).to(dtype)
    u[3], u[5], u[70], u[71] = float("nan"), float("inf"), -float("inf"), -0.0
    dh = torch.randn(256, generator=torch.Generator().manual_seed(2)).to(dtype)
    ref, uc = u.clone().requires_grad_(True), u.to(cuda).requires_grad_(True)
    want, got = torch.relu(ref), ReluFunction.apply(uc)
    for a, b in ((got, want), (torch.autograd.grad(got, uc, dh.to(cuda))[0], torch.autograd.grad(want, ref, dh)[0])):
        assert torch.equal(a.isnan().cpu(), b.isnan()) and torch.equal(a.nan_to_num(7.).cpu(), b.nan_to_num(7.))
    # the same in the epilogue of a 64 -> 64 linear, and in the fused layers: a NaN of one feed-forward feature reaches every row
    L, code = _lib.lib(), _DT[dtype]
    x, W, b = torch.randn(70, 64, device=cuda).to(dtype), torch.randn(64, 64, device=cuda).to(dtype), torch.zeros(64, device=cuda, dtype=dtype)
    b[9] = float("nan")
    v, h = torch.empty_like(x), torch.empty_like(x)
    _lib.check(L.tgt_linear_act_fwd(x.data_ptr(), W.data_ptr(), b.data_ptr(), 70, 64, 64, code, 2, v.data_ptr(), h.data_ptr(), None))
    assert h[:, 9].isnan().all() and int(h.isnan().sum()) == 70
    m = GT(2, 8, 32, 64, 5, 1, 0.0, 0.0, 0.0, 64, 0)
    with torch.no_grad():
        m.layers[1].FFN_layer1.bias[17] = float("nan")
    m = m.to(cuda, dtype)
    loops = torch.arange(100).repeat(2, 1).to(cuda)
    for one in (True, False):
        m.one_operator = one
        out = m(torch.randn(100, 32, device=cuda).to(dtype), None, loops, attn_type="sparse")
        assert out.isnan().all(), one


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_gt_forward_backward_matches_oracle(cuda, dtype):
    """GT of the node-level scripts (4 layers, hidden 64, 8 heads, 128-d input, 40 classes) on a 2 000-node power-law
    graph with self-loops: log-probabilities and the gradient of every parameter that takes part."""
    print(f"GT model case: {dtype}", flush=True)
    torch.manual_seed(2)
    rng = np.random.default_rng(4)
    S = 2000
    e, n = workloads.power_law_graph(n=S - 1, directed_edges=20000)
    assert n == S
    n_layers, H = 4, 8
    m = GT(n_layers, H, 128, 64, 40, 1, 0.0, 0.0, 0.0, 64, 0)
    keys = set(m.state_dict())
    assert {"node_encoder.weight", "downstream_out_proj.weight", "MLP_layer.FC_layers.2.bias", "layers.0.O.weight",
            "layers.0.self_attention_norm.weight", "layers.0.layer_norm1.weight", "layers.0.layer_norm2.bias",
            "layers.0.FFN_layer1.weight", "layers.0.FFN_layer2.bias", "layers.3.self_attention.linear_q.weight"} <= keys
    assert not any("output_layer" in k for k in keys)                      # the GT attention has no output layer
    assert m.layers[0].FFN_layer1.weight.shape == (128, 64) and m.MLP_layer.FC_layers[1].weight.shape == (16, 32)
    with torch.no_grad():
        for p in m.parameters():
            if p.dim() == 2:
                p.normal_(0, 0.15)
    m = m.to(dtype)
    x = torch.randn(S, 128).to(dtype)
    names = [k for k, _ in m.named_parameters()]
    pd = {k: v.detach().double().requires_grad_(True) for k, v in m.named_parameters()}
    ei = torch.as_tensor(e)
    want = ogt.gt_forward(pd, x.double(), ei, n_layers, H)
    y = torch.as_tensor(rng.integers(0, 40, S))
    ref = torch.autograd.grad(torch.nn.functional.nll_loss(want, y), [pd[k] for k in names], allow_unused=True)
    mc = m.to(cuda)
    got = mc(x.to(cuda), None, ei.to(cuda), attn_type="sparse")
    assert got.shape == (S, 40) and got.dtype == dtype
    tol = 1e-5 if dtype == torch.float32 else 6e-2
    assert err(got, want) <= tol, err(got, want)
    got_g = torch.autograd.grad(torch.nn.functional.nll_loss(got.float(), y.to(cuda)), [p for _, p in mc.named_parameters()],
                                allow_unused=True)
    scale = max(r.abs().max().item() for r in ref if r is not None)
    unused, errs = [], {}
    for k, a, r in zip(names, got_g, ref):
        assert (a is None) == (r is None), k
        if r is None:
            unused.append(k)
            continue
        if r.abs().max().item() < 1e-3 * scale:          # the key bias: cancelled by the normalisation, rounding noise only
            assert a.detach().double().abs().max().item() <= 2e-2 * scale, k
            continue
        errs[k] = err(a, r)
    # constructed but not used by the reference's forward: the first LayerNorm of every layer and the plain output layer
    assert sorted(unused) == sorted([f"layers.{l}.self_attention_norm.{w}" for l in range(n_layers) for w in ("weight", "bias")]
                                    + ["downstream_out_proj.weight", "downstream_out_proj.bias"])
    print("gradient errs", {k: round(v, 6) for k, v in errs.items()}, flush=True)
    if dtype == torch.float32:
        bad = {k: v for k, v in errs.items() if v > tol}
        assert not bad, bad
    else:
        # bf16 tensors between all kernels of four layers: the gradients of the last layers stay within the module bar
        tail = {k: v for k, v in errs.items() if k.startswith("MLP_layer")}
        assert tail and max(tail.values()) <= 6e-2, tail
        assert np.median(list(errs.values())) <= 6e-2


@pytest.mark.parametrize("attn_type", ["sparse", "full"])
def test_graph_level_gt_matches_oracle(cuda, attn_type):
    """GT of models/gt_graph_level.py (3 layers, hidden 64, 8 heads, ZINC table) on 10 padded ER graphs whose edges
    index the flattened batch: outputs [b, 1] and every parameter gradient, float32.  With attn_type 'full' the
    reference attends densely over all rows of a graph, padding included (no bias, no mask); that path runs on bf16
    matrix instructions here: the bf16 module bar."""
    from torchgt_amd.gt import GraphLevelGT
    import types
    from oracle import dense_attention as oda
    print(f"graph-level GT case: {attn_type}", flush=True)
    data = workloads.erdos_renyi_batch(batch=10, seed=31)
    sizes = data["n_nodes"]
    b, s = len(sizes), data["spatial_pos"].shape[1]
    rng = np.random.default_rng(5)
    x = np.zeros((b, s, 2), np.int64)
    edges = []
    for g in range(b):
        n = int(sizes[g])
        x[g, :n] = rng.integers(1, 64, size=(n, 2))
        src, dst = np.nonzero(data["spatial_pos"][g][:n, :n] == 2)
        loops = np.arange(n)
        edges.append(np.stack([np.concatenate([src, loops]), np.concatenate([dst, loops])]) + g * s)
    ei = torch.from_numpy(np.concatenate(edges, 1))
    x = torch.from_numpy(x)
    torch.manual_seed(3)
    n_layers, H = 3, 8
    m = GraphLevelGT(n_layers, H, 64, 0.0, 0.0, 64, "ZINC", "single_hop", 5, 0.0, 1)
    assert {"embedding_h.weight", "graph_token.weight", "MLP_layer.FC_layers.0.weight", "layers.2.O.bias"} <= set(m.state_dict())
    with torch.no_grad():
        for k, p in m.named_parameters():
            if p.dim() == 2:
                p.normal_(0, 0.05 if ("linear_q" in k or "linear_k" in k) and attn_type == "full" else 0.15)
    names = [k for k, _ in m.named_parameters()]
    pd = {k: v.detach().double().requires_grad_(True) for k, v in m.named_parameters()}
    if attn_type == "sparse":
        want = ogt.gt_graph_level_forward(pd, x, ei, n_layers, H)
    else:
        # the same layers with the dense attention of the graph-level CoreAttention (q * sqrt(d), softmax over all s keys)
        out = pd["embedding_h.weight"][x].sum(-2)
        lin = lambda v, nme: v @ pd[nme + ".weight"].t() + pd[nme + ".bias"]
        for l in range(n_layers):
            pre = f"layers.{l}."
            q, k, v = (lin(out, pre + "self_attention." + nme).view(b, s, H, 8) for nme in ("linear_q", "linear_k", "linear_v"))
            y = lin(oda.dense_attention(q, k, v, None), pre + "O")
            out = ogt.layer_norm(out + y, pd[pre + "layer_norm1.weight"], pd[pre + "layer_norm1.bias"])
            y = lin(ogt.relu(lin(y, pre + "FFN_layer1")), pre + "FFN_layer2")
            out = ogt.layer_norm(out + y, pd[pre + "layer_norm2.weight"], pd[pre + "layer_norm2.bias"])
        want = ogt.mlp_readout(out.mean(1), pd)
    target = torch.randn(want.shape, generator=torch.Generator().manual_seed(6)).double()
    ref = torch.autograd.grad(((want - target) ** 2).mean(), [pd[k] for k in names], allow_unused=True)
    mc = m.to(cuda)
    got = mc(types.SimpleNamespace(x=x.to(cuda), edge_index=ei.to(cuda)), attn_type=attn_type)
    assert got.shape == want.shape == (b, 1)
    tol = 1e-5 if attn_type == "sparse" else 6e-2
    assert err(got, want) <= tol, err(got, want)
    # the same upstream gradient on both sides (the oracle's dL/d output), so that the backward is compared by itself
    dl = (2 * (want - target) / want.numel()).detach()
    got_g = torch.autograd.grad(got, [p for _, p in mc.named_parameters()], dl.to(cuda, got.dtype), allow_unused=True)
    scale = max(r.abs().max().item() for r in ref if r is not None)
    unused, errs = [], {}
    for k, a, r in zip(names, got_g, ref):
        assert (a is None) == (r is None), k
        if r is None:
            unused.append(k)
        elif r.abs().max().item() < 1e-3 * scale:
            assert a.detach().double().abs().max().item() <= 2e-2 * scale, k
        else:
            errs[k] = err(a, r)
    assert sorted(unused) == sorted([f"layers.{l}.self_attention_norm.{w}" for l in range(n_layers) for w in ("weight", "bias")]
                                    + ["graph_token.weight"])
    print("gradient errs", {k: round(v, 6) for k, v in errs.items()}, flush=True)
    # 'full': the activations carry bf16-sized noise from the dense attention, and a ReLU unit whose input is within
    # that noise of zero takes the other branch: with ten graphs one such unit of the readout moves its layer's
    # gradient by several percent.  The bar there is 0.15 on every tensor and the module bar on the median.
    gtol = tol if attn_type == "sparse" else 0.15
    bad = {k: v for k, v in errs.items() if v > gtol}
    assert not bad, bad
    assert np.median(list(errs.values())) <= tol
    assert "embedding_h.weight" in errs and got_g[names.index("embedding_h.weight")][0].abs().max() > 0     # row 0 is an ordinary row


class _ReadoutFwd(ctypes.Structure):
    _fields_ = [("rows", ctypes.c_int64)] + [(k, ctypes.c_int32) for k in ("dtype", "m1", "m2", "out", "classes")] + [(k, ctypes.c_void_p) for k in ("x", "w", "v", "logp")]


class _ReadoutBwd(ctypes.Structure):
    _fields_ = ([("rows", ctypes.c_int64)] + [(k, ctypes.c_int32) for k in ("dtype", "m1", "m2", "out", "classes")] +
                [(k, ctypes.c_void_p) for k in ("x", "dlogp", "logp", "w", "w_back", "v", "dx")] + [("grads", ctypes.c_void_p * 6), ("partial", ctypes.c_void_p)])


def run_readout(x, W, b, dlogp, classes, logp_back=None):
    """log-probabilities, dx and the gradients of W and b from tgt_readout_fwd and tgt_readout_bwd (logp_back: the log-probabilities it is told)"""
    L, dtype, code, st = _lib.lib(), x.dtype, _DT[x.dtype], ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    n, (m1, m2, out) = x.shape[0], [t.shape[0] for t in W]
    ints = lambda *a: (ctypes.c_int * len(a))(*a)
    ptrs = lambda ts: (ctypes.c_void_p * len(ts))(*[t.data_ptr() for t in ts])
    unit = L.tgt_node_frag_bytes(3, code)
    frags, vecs = torch.empty(unit, dtype=torch.uint8, device=x.device), torch.empty(192, device=x.device)
    _lib.check(L.tgt_node_pack_parts(ptrs(W), ints(64, m1, m2), ints(m1, m2, out), ints(64, m1, m2), 3, ptrs(b), ints(m1, m2, out), 3, code, frags.data_ptr(), vecs.data_ptr(), st))
    logp, dx, grads = torch.full((n, classes), 7., device=x.device).to(dtype), torch.full_like(x, 7), [torch.full_like(t, 7) for t in W + b]
    f = _ReadoutFwd(n, code, m1, m2, out, classes, x.data_ptr(), frags.data_ptr(), vecs.data_ptr(), logp.data_ptr())
    _lib.check(L.tgt_readout_fwd(ctypes.byref(f), st))
    partial = torch.empty(L.tgt_readout_partial_floats(n, m1, m2, out), device=x.device)
    r = _ReadoutBwd(n, code, m1, m2, out, classes, x.data_ptr(), dlogp.data_ptr(), (logp if logp_back is None else logp_back).data_ptr(), frags.data_ptr(), frags.data_ptr() + unit // 2, vecs.data_ptr(), dx.data_ptr(),
                    ptrs(grads), partial.data_ptr())
    _lib.check(L.tgt_readout_bwd(ctypes.byref(r), st))
    return logp, dx, grads


# Weights and rows of -1, 0, 1 (times a power of two): the inputs of both ReLUs and the logits are the same numbers whatever the order of
# the sums, so no activation changes its side.  What is left: a log-softmax (2^-8 of a bfloat16 result, 1e-5 in float32) and, backward, one rounding of
# every d logits, du (bfloat16: 2^-9 each of three in a row, and of the results): 1e-2 of the largest; float32 1e-5.
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,m1,m2,out,classes", [(1, 32, 16, 40, 40), (15, 5, 3, 7, 7), (16, 64, 64, 64, 63), (17, 33, 17, 8, 1), (63, 32, 16, 48, 47), (65, 32, 16, 1, 1),
                                                 (129, 1, 1, 2, 2), (4097, 32, 16, 40, 40), (16385, 64, 32, 16, 13), (32769, 32, 16, 40, 40), (49152, 64, 64, 64, 63), (70001, 32, 16, 40, 40)])
def test_readout_in_one_kernel(cuda, dtype, n, m1, m2, out, classes):
    print(f"readout n={n} widths {m1} {m2} {out} classes={classes} {dtype}", flush=True)
    g = torch.Generator(device=cuda).manual_seed(n + out)
    grid = lambda *s: torch.randint(-1, 2, s, generator=g, device=cuda).to(dtype)
    W = [grid(m1, 64) * 0.25, grid(m2, m1) * 0.5, grid(out, m2) * 0.25]
    b = [grid(m1), grid(m2), grid(out)]
    x, dlogp = grid(n, 64), torch.randn(n, classes, generator=g, device=cuda).to(dtype)
    logp, dx, grads = run_readout(x, W, b, dlogp, classes)
    held = lambda t: t.to(dtype).double()      # as a row of this type holds it
    Wd, bd, a0 = [t.double() for t in W], [t.double() for t in b], x.double()
    a1 = held(a0 @ Wd[0].T + bd[0]).relu()
    a2 = held(a1 @ Wd[1].T + bd[1]).relu()
    want = torch.log_softmax(held(a2 @ Wd[2].T + bd[2])[:, :classes], 1)
    assert float((logp.double() - want).abs().max()) <= (2 ** -8 if dtype == torch.bfloat16 else 1e-5) * max(1.0, float(want.abs().max()))
    d = torch.zeros(n, out, dtype=torch.double, device=cuda)
    d[:, :classes] = dlogp.double() - logp.double().exp() * dlogp.double().sum(1, keepdim=True)
    d1 = (d @ Wd[2]) * (a2 > 0)
    d0 = (d1 @ Wd[1]) * (a1 > 0)
    for name, got, ref in zip(("dx", "Wa", "Wb", "Wc", "ba", "bb", "bc"), [dx, *grads], [d0 @ Wd[0], d0.T @ a0, d1.T @ a1, d.T @ a2, d0.sum(0), d1.sum(0), d.sum(0)]):
        top = max(float(ref.abs().max()), 1e-30)
        # a bias of many rows: n terms of either sign, each rounded; their sum is as large as sqrt(n) of them
        assert float((got.double() - ref).abs().max()) <= (1e-2 if dtype == torch.bfloat16 else 1e-5) * max(top, 1.0 if name[0] == "b" or n < 3 else 0.0), name


@pytest.mark.parametrize("n", [4096, 64000, 300000])
def test_readout_weight_gradients_are_as_exact_as_float32_products(cuda, n):
    """rms error of the three weight gradients against 64 bits, of the rms of the result.  Weights of 1, positive rows and log-probabilities of -inf (d logits =
    dlogp) hand the same two matrices of random float32 numbers to each of the three products, without an error in front of them and with no ReLU near 0.
    Bound: float32 matrix instructions round the running sum once per two products, which leaves 2^-24 sqrt(1 + k / 12) after the k rows of a worker
    (test_gpu_projections.py).  Also dx, whose products are exact here."""
    g = torch.Generator(device=cuda).manual_seed(n)
    x, dlogp = torch.randn(n, 64, generator=g, device=cuda).abs() + 2.0 ** -20, torch.randn(n, 64, generator=g, device=cuda)
    one, none = torch.eye(64, device=cuda), torch.zeros(64, device=cuda)
    _, dx, grads = run_readout(x, [one, one, one], [none, none, none], dlogp, 64, logp_back=torch.full_like(dlogp, -float("inf")))
    assert torch.equal(dx, dlogp)
    want = dlogp.double().t().contiguous() @ x.double()
    errs = [float((a.double() - want).norm() / want.norm()) for a in grads[:3]]
    k = 64 if n <= 16384 else -(-n // (128 * 256)) * 128      # groups of 64 or 128 rows over 256 CUs
    bound = 2 ** -24 * (1 + k / 12) ** 0.5
    print(f"readout exactness n={n}: " + " ".join(f"{e:.2e}" for e in errs) + f" (bound {bound:.2e})", flush=True)
    assert max(errs) <= bound


@pytest.mark.parametrize("n,m1,m2,out", [(4096, 32, 16, 40), (4096, 64, 64, 64), (16400, 36, 20, 12)])
def test_readout_is_as_exact_as_its_linears_and_log_softmax(cuda, n, m1, m2, out):
    """float32: rms error of log-probabilities and dx against 64 bits, next to that of the separate linears, ReLUs and torch's log_softmax on the same operands: no
    larger than theirs, 5 % for sums in another order.  (dx of rows without a ReLU input within 1e-5 of 0: those may change their side.)"""
    def run(dtype, linear, relu):
        xs = x.to(dtype).requires_grad_(True)
        y, near = xs, torch.ones(n, dtype=torch.bool, device=cuda)
        for i in range(3):
            y = linear(y, W[i].to(dtype), b[i].to(dtype))
            if i < 2:
                near &= y.detach().abs().min(1).values > 1e-5
                y = relu(y)
        lp = torch.log_softmax(y, 1)
        return lp.detach(), torch.autograd.grad(lp, xs, dlogp.to(dtype))[0], near

    errs = {"fused": [0.0, 0.0], "separate": [0.0, 0.0]}
    for seed in range(3):
        g = torch.Generator(device=cuda).manual_seed(seed + out)
        rand = lambda *s: torch.randn(*s, generator=g, device=cuda)
        W, b = [rand(m1, 64) / 8, rand(m2, m1) / m1 ** 0.5, rand(out, m2) / m2 ** 0.5], [rand(m) * 0.1 for m in (m1, m2, out)]
        x, dlogp = rand(n, 64), rand(n, out)
        lp, dx, near = run(torch.float64, lambda y, w, c: y @ w.t() + c, torch.relu)
        fused = run_readout(x, W, b, dlogp, out)
        for name, (p, d) in (("fused", fused[:2]), ("separate", run(torch.float32, lambda y, w, c: LinearFunction.apply(y, w, c)[0], ReluFunction.apply)[:2])):
            for i, (a, r) in enumerate(((p, lp), (d[near], dx[near]))):
                errs[name][i] += float((a.double() - r).norm() / r.norm()) / 3
    print(f"readout n={n} widths {m1} {m2} {out}: {errs}", flush=True)
    for a, s in zip(errs["fused"], errs["separate"]):
        assert a <= 1.05 * s


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,m1,m2,out,classes", [(20, 32, 16, 40, 40), (70, 5, 3, 7, 6), (130, 64, 64, 64, 64), (33, 33, 17, 8, 8), (300, 32, 16, 1, 1)])
@pytest.mark.parametrize("what", ["x", "Wa", "Wb", "Wc", "bias", "killed", "overflow", "dlogp"])
def test_infinities_go_through_the_readout_as_through_three_linears(cuda, dtype, n, m1, m2, out, classes, what):
    """Every log-probability and gradient is +-inf, NaN or finite as the products and sums have it, widths of less than 64 and rows past a tile's end
    included.  `killed`: infinite weights whose pre-activations are all -inf, so that the ReLU ends them; `overflow`: finite operands, infinite products.
    Weights and rows of -1, 0, 1 times a power of two elsewhere: no ReLU changes its side (see test_readout_in_one_kernel, also for the bars)."""
    print(f"readout infinities n={n} widths {m1} {m2} {out} classes={classes} {what} {dtype}", flush=True)
    g = torch.Generator().manual_seed(n + m1)
    grid = lambda *s: torch.randint(-1, 2, s, generator=g).to(dtype)
    W, b = [grid(m1, 64) * 0.25, grid(m2, m1) * 0.5, grid(out, m2) * 0.25], [grid(m1), grid(m2), grid(out)]
    x, dlogp, inf = grid(n, 64), torch.randn(n, classes, generator=g).to(dtype), float("inf")
    W[0][0, 0] = 0.25
    if what == "x":
        x[n // 2, 1], x[n - 1, 63], x[0, 0], x[3, 5], x[3, 6] = inf, -inf, float("nan"), inf, inf
    elif what in ("Wa", "Wb", "Wc"):
        w = W["abc".index(what[1])]
        w[w.shape[0] // 2, w.shape[1] - 1], w[0, 0] = inf, -inf
    elif what == "bias":
        b[0][m1 - 1], b[1][0], b[2][out // 2] = -inf, inf, -inf
    elif what == "killed":
        x[:, 7] = 1
        W[0][m1 // 2, 7], W[0][0, 7] = -inf, -inf
        b[1][m2 - 1] = -inf
    elif what == "overflow":
        x[:, 5], x[n - 1], W[0][m1 - 1, 5] = 0, 0, 2.0 ** 100
        x[n - 1, 5] = 2.0 ** 100
    else:
        dlogp[n - 1, classes - 1], dlogp[0, 0] = inf, -inf
    logp, dx, grads = run_readout(x.to(cuda), [w.to(cuda) for w in W], [t.to(cuda) for t in b], dlogp.to(cuda), classes)

    def product(p, q):      # every product formed and added, in the order and the range of float32
        s = torch.zeros(p.shape[0], q.shape[1])
        for k in range(p.shape[1]):
            s += p[:, k:k + 1].float() * q[k:k + 1].float()
        return s.double()

    held = lambda t: t.to(dtype).double()
    Wd, bd = [t.double() for t in W], [t.double() for t in b]
    a1 = held(product(x, W[0].T) + bd[0]).relu()
    a2 = held(product(a1, W[1].T) + bd[1]).relu()
    want = torch.log_softmax(held(product(a2, W[2].T) + bd[2])[:, :classes], 1)
    back = logp.double().cpu()
    d = torch.zeros(n, out, dtype=torch.double)
    d[:, :classes] = dlogp.double() - back.exp() * dlogp.double().sum(1, keepdim=True)
    d = held(d)
    d1 = held(torch.where(a2 <= 0, 0.0, product(d, W[2])))
    d0 = held(torch.where(a1 <= 0, 0.0, product(d1, W[1])))
    bar, seen = 1e-2 if dtype == torch.bfloat16 else 1e-5, 0
    refs = [want, product(d0, W[0]), product(d0.T, x), product(d1.T, a1), product(d.T, a2), d0.sum(0), d1.sum(0), d.sum(0)]
    for name, a, r in zip(("logp", "dx", "Wa", "Wb", "Wc", "ba", "bb", "bc"), [logp, dx, *grads], refs):
        a = a.double().cpu()
        assert torch.equal(a.isnan(), r.isnan()) and torch.equal(a.isposinf(), r.isposinf()) and torch.equal(a.isneginf(), r.isneginf()), name
        fin = r.isfinite()
        seen += int((~fin).sum())
        assert not fin.any() or float((a - r)[fin].abs().max()) <= bar * max(1.0, float(r[fin].abs().max())), name
    assert seen > 0 or what == "killed"


@pytest.mark.parametrize("where", ["MLP_layer.FC_layers.0.weight", "MLP_layer.FC_layers.1.weight", "MLP_layer.FC_layers.2.weight", "MLP_layer.FC_layers.1.bias", "x"])
def test_an_infinity_in_the_model_gives_what_its_modules_give(cuda, where):
    """float32 GT of hidden size 64 as one operator and module by module: the same infinities and NaN in the log-probabilities, the loss and every gradient"""
    print(f"gt with an infinity in {where}", flush=True)
    torch.manual_seed(1)
    n, model = 300, GT(2, 8, 32, 64, 7, 1, 0.0, 0.0, 0.0, 64, 0)
    with torch.no_grad():
        for p in model.parameters():
            if p.dim() == 2:
                p.normal_(0, p.shape[1] ** -0.5)
    x, y = torch.randn(n, 32), torch.randint(0, 7, (n,), device=cuda)
    if where == "x":
        x[n // 2, 3] = float("inf")
    else:
        with torch.no_grad():
            p = dict(model.named_parameters())[where]
            p[(p.shape[0] // 2, p.shape[1] - 1) if p.dim() == 2 else 3] = -float("inf") if p.dim() == 2 else float("inf")
    model, loops, got = model.to(cuda), torch.arange(n).repeat(2, 1).to(cuda), []
    for one in (True, False):
        model.one_operator = one
        model.zero_grad(set_to_none=True)
        out = model(x.to(cuda), None, loops, attn_type="sparse")
        loss = torch.nn.functional.nll_loss(out, y)
        loss.backward()
        got.append([("output", out.detach()), ("loss", loss.detach())] + [(k, p.grad) for k, p in model.named_parameters() if p.grad is not None])
    assert not got[0][0][1].isfinite().all()
    for (name, a), (_, r) in zip(*got):
        assert torch.equal(a.isnan(), r.isnan()) and torch.equal(a.isposinf(), r.isposinf()) and torch.equal(a.isneginf(), r.isneginf()), name
        fin = r.isfinite()
        assert not fin.any() or float((a - r)[fin].abs().max()) <= 1e-4 * max(1.0, float(r[fin].abs().max())), name


def test_readout_refuses_other_widths():
    L = _lib.lib()
    assert L.tgt_readout_partial_floats(10, 65, 16, 40) == -1 and L.tgt_readout_partial_floats(10, 32, 0, 40) == -1
    assert L.tgt_readout_fwd(None, None) != 0 and L.tgt_readout_bwd(None, None) != 0
    f = _ReadoutFwd(0, 0, 32, 16, 40, 41, None, None, None, None)
    assert L.tgt_readout_fwd(ctypes.byref(f), None) != 0      # more classes than outputs
    f.classes = 40
    assert L.tgt_readout_fwd(ctypes.byref(f), None) == 0      # no rows
