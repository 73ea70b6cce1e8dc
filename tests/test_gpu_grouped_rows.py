"""GPU: rows of 5 to 32 edges that the backward walks with one lane group each (graphs whose neighbours are near each other), at the
edges of its steps of four: against the oracle in float64 on the dtype-rounded inputs.  Bars as for the other walks: the result's own
rounding, 2^-9 of its size for bf16, is a tenth of them; float32 adds at most 32 terms in a row, 32 * 2^-24 = 2e-6."""
import numpy as np
import pytest
import torch

from oracle import sparse_attention as osa
from torchgt_amd import GraphPlan, _lib, sparse_attention

pytestmark = pytest.mark.gpu
TOL = {torch.float32: 1e-5, torch.bfloat16: 2e-2}
LENGTHS = [5, 6, 7, 8, 9, 12, 13, 16, 17, 31, 32, 33, 0, 1, 4, 29, 40, 256, 257, 11]      # the last row's edges end the list


def near_graph(n, lengths, seed, reach=600):
    """Rows of the given lengths in turn; the k-th edge of row r comes from a node at most `reach` away."""
    rng = np.random.default_rng(seed)
    dst = np.repeat(np.arange(n), np.resize(lengths, n))
    src = np.clip(dst + rng.integers(-reach, reach + 1, dst.size), 0, n - 1)
    order = rng.permutation(dst.size)
    return torch.from_numpy(np.stack([src[order], dst[order]]))


def inputs(n, E, H, d, dtype, bias_kind, seed):
    g = torch.Generator().manual_seed(seed)
    q, k, v, dout = (torch.randn(n, H, d, generator=g).to(dtype) for _ in range(4))
    shape = {"none": None, "edge": (E,), "edge_head": (E, H)}[bias_kind]
    return q, k, v, None if shape is None else (torch.randn(shape, generator=g) * 0.5).to(dtype), dout


def reference(q, k, v, bias, ei, dout, dev="cpu"):
    t = [x.to(dev).double().requires_grad_(True) for x in (q, k, v)]
    b = None if bias is None else bias.to(dev).double().requires_grad_(True)
    out, _ = osa.sparse_attention(t[0], t[1], t[2], ei.to(dev), b)
    return [out] + list(torch.autograd.grad(out, t + ([] if b is None else [b]), dout.to(dev).double()))


def close(got, want, tol):
    for name, a, b in zip(("out", "dq", "dk", "dv", "dbias"), got, want):
        a, b = a.detach().double().cpu(), b.detach().cpu()
        assert float((a - b).abs().max()) <= tol * float(b.abs().max()), name


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H,d,bias_kind", [(8, 8, "none"), (4, 16, "none"), (2, 32, "none"), (8, 8, "edge_head"), (8, 16, "none"),
                                           (8, 16, "edge_head"), (16, 8, "edge"), (4, 32, "edge_head")])
def test_rows_of_one_lane_group(cuda, H, d, bias_kind, dtype):
    n, ei = 16384, near_graph(16384, LENGTHS, 1)
    print(f"case {H}x{d} {bias_kind} {dtype} E={ei.shape[1]}", flush=True)
    q, k, v, bias, dout = inputs(n, ei.shape[1], H, d, dtype, bias_kind, 2)
    plan = GraphPlan(ei.to(cuda), n)
    t = [x.to(cuda).requires_grad_(True) for x in (q, k, v)] + ([] if bias is None else [bias.to(cuda).requires_grad_(True)])
    out = sparse_attention(t[0], t[1], t[2], edge_bias=t[3] if bias is not None else None, plan=plan)
    got = [out] + list(torch.autograd.grad(out, t, dout.to(cuda)))
    close(got, reference(q, k, v, bias, ei, dout), TOL[dtype])


def test_many_edges_with_a_bias(cuda):
    # from 2 Mi edges and 16 edges a row on 64-element rows with a bias take this list as well
    n = 110_000
    ei = near_graph(n, [20, 17, 32, 9, 24], 3)
    assert ei.shape[1] >= 16 * n and ei.shape[1] >= 2 << 20
    q, k, v, bias, dout = inputs(n, ei.shape[1], 8, 8, torch.bfloat16, "edge_head", 4)
    t = [x.to(cuda).requires_grad_(True) for x in (q, k, v, bias)]
    out = sparse_attention(t[0], t[1], t[2], edge_bias=t[3], plan=GraphPlan(ei.to(cuda), n))
    got = [out] + list(torch.autograd.grad(out, t, dout.to(cuda)))
    close(got, reference(q, k, v, bias, ei, dout, cuda), TOL[torch.bfloat16])


@pytest.mark.parametrize("H,d", [(8, 8), (8, 16)])
@pytest.mark.parametrize("dtype,bias_kind", [(torch.float32, "none"), (torch.float32, "edge_head"), (torch.bfloat16, "edge_head"), (torch.bfloat16, "none")])
def test_first_backward_inside_a_capture(cuda, dtype, bias_kind, H, d):
    """Creating the plan (64 elements a row) and the first call of another shape make every list that a backward of the shape may take: one that is
    captured before any other backward ran takes the same list as an eager one, and gives its bits."""
    n = 16384
    print(f"captured first: {H}x{d} {bias_kind} {dtype}", flush=True)
    ei = near_graph(n, LENGTHS, 5)
    q, k, v, bias, dout = inputs(n, ei.shape[1], H, d, dtype, bias_kind, 6)
    L, P = _lib.lib(), lambda x: None if x is None else x.data_ptr()
    plan = GraphPlan(ei.to(cuda), n)
    dev = [None if x is None else x.to(cuda) for x in (q, k, v, bias, dout)]
    out, dq, dk, dv = (torch.empty_like(dev[0]) for _ in range(4))
    db = None if bias is None else torch.empty_like(dev[3])
    Z, ws = torch.empty(n, H, device=cuda), plan.workspace(H, d)
    code = _lib.DTYPE_F32 if dtype == torch.float32 else _lib.DTYPE_BF16
    mode = _lib.BIAS_NONE if bias is None else _lib.BIAS_EDGE_HEAD
    results = [x for x in (out, dq, dk, dv, db) if x is not None]

    def forward(stream):
        _lib.check(L.tgt_sparse_attn_fwd(plan.handle, P(dev[0]), P(dev[1]), P(dev[2]), P(dev[3]), mode, H, d, code, P(out), P(Z), P(ws), ws.numel(), stream))

    def step(stream):
        forward(stream)
        _lib.check(L.tgt_sparse_attn_bwd(plan.handle, P(dev[0]), P(dev[1]), P(dev[2]), P(dev[3]), mode, H, d, code, P(out), P(Z), P(dev[4]), P(dq),
                                         P(dk), P(dv), P(db), P(ws), ws.numel(), stream))

    if H * d != 64:
        forward(torch.cuda.current_stream().cuda_stream)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step(torch.cuda.current_stream().cuda_stream)
    step(torch.cuda.current_stream().cuda_stream)
    eager = [x.clone() for x in results]
    close(eager, reference(q, k, v, bias, ei, dout), TOL[dtype])
    for replay in range(3):
        for x in results:
            x.zero_()
        graph.replay()
        torch.cuda.synchronize()
        for name, x, want in zip(("out", "dq", "dk", "dv", "dbias"), results, eager):
            assert torch.equal(x, want), f"{name} of replay {replay}"
        step(torch.cuda.current_stream().cuda_stream)
    plan.close()
