"""The whole-model operators against the oracle in float64: outputs and the gradients of all parameters and of the input, as one vector.

Bars, relative errors in the 2-norm.  float32: 4e-6; a model of two layers passes each row through some twenty sums of 64 to 300 terms
one behind the other, forward and backward, each within a few 2^-24 of its row (measured: 1e-7 for outputs, 4e-7 to 1e-6 for gradients).
A ReLU whose input is nearly 0 may open on one side and not on the other: one of n * 128 units a layer, and the gradients of two
layers, each unit's share alike, move by about 1 / sqrt(2 * 128 n) of their norm - that much is allowed on top for a GT.
bf16: what the same model gives layer by layer is the measure, the kernels that round at the same places: no more than a quarter above
its distance, or 2e-3."""
import types

import pytest
import torch

from oracle import graph_level as ogl
from oracle import gt as ogt
from oracle import sparse_attention as osa
from torchgt_amd import GT, GraphLevelGraphormer, Graphormer, GraphPlan, workloads

pytestmark = pytest.mark.gpu


def edges_of(n, tokens, seed):
    g = torch.Generator().manual_seed(seed)
    e = torch.cat([torch.randint(0, n, (2, 4 * n), generator=g), torch.arange(n).repeat(2, 1)], 1)
    if tokens:
        rows = torch.arange(n + 1)
        e = torch.cat([e + 1, torch.stack([torch.zeros_like(rows), rows]), torch.stack([rows, torch.zeros_like(rows)])], 1)
    return e


def scaled(model, seed, dtype):
    g = torch.Generator().manual_seed(seed)
    with torch.no_grad():
        for p in model.parameters():
            p.copy_(p + torch.randn(p.shape, generator=g) * 0.1 if p.dim() == 1 else torch.randn(p.shape, generator=g) / p.shape[-1] ** 0.5)
    return model.to(dtype)


def node_graphormer(p, x, edges, layers, heads):
    """Graphormer.forward (models/graphormer_dist_node_level.py:355-392) with one global token, by the oracle's parts."""
    linear, norm = ogt._linear, lambda t, name: ogl.layer_norm(t, p[name + ".weight"], p[name + ".bias"])
    h = torch.cat([p["graph_token.weight"], linear(x, p, "node_encoder")])
    for i in range(layers):
        at = f"layers.{i}."
        y = norm(h, at + "self_attention_norm")
        q, k, v = (linear(y, p, f"{at}self_attention.linear_{c}").view(1, h.shape[0], heads, -1) for c in "qkv")
        h = h + linear(osa.sparse_attention(q, k, v, edges)[0].reshape(h.shape[0], -1), p, at + "self_attention.output_layer")
        h = h + linear(ogl.gelu(linear(norm(h, at + "ffn_norm"), p, at + "ffn.layer1")), p, at + "ffn.layer2")
    return torch.log_softmax(linear(norm(h, "final_ln")[1:], p, "downstream_out_proj"), dim=1)


def compare(model, run, exact, weights, flips, cuda):
    """run(model) -> (output, input or None) on the GPU; exact(p) -> (output, input or None) in float64 from the parameters by name."""
    dtype = next(model.parameters()).dtype
    p = {k: v.detach().double().requires_grad_(True) for k, v in model.named_parameters()}
    want, xin = exact(p)
    (want * weights).sum().backward()
    model = model.to(cuda)
    errors = []
    for one in (True, False):
        model.one_operator = one
        model.zero_grad(set_to_none=True)
        out, x = run(model)
        (out.double() * weights.to(cuda)).sum().backward()
        names = [k for k, v in model.named_parameters() if v.grad is not None]
        assert all(p[k].grad is not None for k in names) and len(names) > 20
        got = [model.get_parameter(k).grad for k in names] + ([] if x is None else [x.grad])
        ref = [p[k].grad for k in names] + ([] if x is None else [xin.grad])
        for k, r in zip(names, ref):
            if k.startswith("graph_") and k.endswith("encoder.weight") and "edge_dis" not in k:
                r[0] = 0      # nn.Embedding(padding_idx=0)
        flat = lambda ts: torch.cat([t.detach().double().cpu().flatten() for t in ts])
        far = lambda a, b: float((a - b).norm() / b.norm())
        errors.append((far(out.detach().double().cpu(), want.detach()), far(flat(got), flat(ref))))
    print(f"  output {errors[0][0]:.2e} (layers {errors[1][0]:.2e})  gradients {errors[0][1]:.2e} (layers {errors[1][1]:.2e})", flush=True)
    for (mine, layers), extra in zip(zip(*errors), (0.0, flips)):
        assert mine <= (4e-6 + extra if dtype == torch.float32 else max(1.25 * layers, 2e-3))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("kind,n,features,classes,hidden,heads", [("graphormer", 700, 100, 47, 64, 8), ("graphormer", 257, 32, 5, 64, 2), ("graphormer", 300, 128, 40, 128, 8),
                                                                  ("gt", 700, 100, 47, 64, 8), ("gt", 300, 128, 40, 128, 8)])
def test_node_models(cuda, dtype, kind, n, features, classes, hidden, heads):
    print(f"oracle case: {kind} n={n} features={features} classes={classes} hidden={hidden} heads={heads} {dtype}", flush=True)
    tokens, layers = (0, 2) if kind == "gt" else (1, 2)
    torch.manual_seed(n)
    model = scaled((Graphormer if tokens else GT)(layers, heads, features, hidden, classes, 1, 0.0, 0.0, 0.0, hidden, tokens), n + 1, dtype)
    g = torch.Generator().manual_seed(n + 2)
    x, e, weights = torch.randn(n, features, generator=g).to(dtype), edges_of(n, tokens, n + 3), torch.randn(n, classes, generator=g).double()
    plan = GraphPlan(e.to(cuda), n + tokens)

    def run(m):
        xc = x.to(cuda).requires_grad_(True)
        assert (m._one_operator(*((xc, None, plan, None, "sparse") if tokens else (xc, plan, "sparse"))) is not None) == m.one_operator
        return m(xc, None, plan, attn_type="sparse"), xc

    def exact(p):
        xd = x.double().requires_grad_(True)
        return (node_graphormer(p, xd, e, layers, heads) if tokens else ogt.gt_forward(p, xd, e, layers, heads)), xd

    compare(model, run, exact, weights, 0.0 if tokens else (2 * 128 * n) ** -0.5, cuda)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("edge_type,outputs", [("single_hop", 1), ("multi_hop", 17)])
def test_graph_models(cuda, dtype, edge_type, outputs):
    print(f"oracle case: graph-level {edge_type} outputs={outputs} {dtype}", flush=True)
    layers, heads, b = 3, 8, 12
    data = workloads.erdos_renyi_batch(batch=b, seed=31)
    s = data["spatial_pos"].shape[1]
    torch.manual_seed(5)
    model = scaled(GraphLevelGraphormer(layers, heads, 64, 0.0, 0.0, 64, "ZINC", edge_type, 3, 0.0, outputs), 6, dtype)
    with torch.no_grad():      # (the attention multiplies queries by sqrt(d): scores of a few units)
        for layer in model.layers:
            layer.self_attention.linear_q.weight.mul_(0.1)
    g = torch.Generator().manual_seed(7)
    ids = lambda hi, *shape: torch.randint(1, hi, shape, generator=g)
    batch = dict(x=ids(64, b, s, 1), in_degree=ids(64, b, s), out_degree=ids(64, b, s), attn_bias=torch.from_numpy(data["attn_bias"]).to(dtype),
                 spatial_pos=torch.from_numpy(data["spatial_pos"]).long(), attn_edge_type=torch.from_numpy(data["edge_type"]).long().unsqueeze(-1),
                 edge_input=ids(64, b, s, s, 4, 1))
    weights = torch.randn(b, outputs, generator=g).double()
    on_gpu = types.SimpleNamespace(**{k: v.to(cuda) for k, v in batch.items()})

    def run(m):
        assert (m._one_operator(on_gpu) is not None) == m.one_operator
        return m(on_gpu), None

    def exact(p):
        return ogl.graphormer_forward(p, dict(batch, attn_bias=batch["attn_bias"].double()), layers, heads, edge_type, 3), None

    compare(model, run, exact, weights, 0.0, cuda)
