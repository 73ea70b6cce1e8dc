"""What is timed: the work that training and evaluation scripts of this framework spend their time on, through its
public entry points.

Kinds of cases
  attention    one layer's sparse attention, forward + backward, on a prebuilt plan (the kernel-level benchmark)
  block        the same over cluster tiles plus the edges outside them
  dense        the biased dense attention of a graph-level batch, forward + backward
  node_train   a training step of a node-level model: forward, nll loss, backward to every parameter
  node_eval    the evaluation pass of a node-level model
  graph_train  a training step of the graph-level Graphormer
  batch        what a training loop does with a new batch of nodes before its first step: sub-graph, global node,
               cluster reordering, plan

Graphs, features, labels and weights are synthetic and made on the GPU from the seed alone.  Weights have the scale of a
trained layer (attention scores of order one), not the near-zero scale of a fresh initialisation.
"""
import math
import types

import torch

from torchgt_amd import (GT, GraphLevelGraphormer, GraphPlan, Graphormer, TileSet, block_attention, dense_attention,
                         floyd_warshall, gen_edge_input, nll_loss, sparse_attention)
from torchgt_amd.graph_prep import fix_edge_index, prepare_batch

DEV = "cuda"
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}
BLOCK = 16              # tile edge of the cluster reordering
SPD_CLAMP = 20          # longest shortest-path distance that has an embedding of its own


def listed():
    return [
        # a citation-sized graph, one scalar bias per edge (a shortest-path embedding): launches and latency count
        {"name": "attention_4k_f32", "kind": "attention", "nodes": 4096, "degree": 8.0, "exponent": 2.5, "clusters": 1,
         "heads": 8, "dim": 8, "dtype": "f32", "bias": "edge"},
        # the headline: one sequence of 64 K nodes, bias per edge and head with gradient
        {"name": "attention_64k_f32", "kind": "attention", "nodes": 64000, "degree": 5.3, "exponent": 2.1, "clusters": 1,
         "heads": 8, "dim": 8, "dtype": "f32", "bias": "edge_head"},
        # a large clustered graph in bf16 without bias, four heads of 16
        {"name": "attention_262k_bf16", "kind": "attention", "nodes": 262144, "degree": 16.0, "exponent": 2.1, "clusters": 64,
         "heads": 4, "dim": 16, "dtype": "bf16", "bias": "none"},
        # cluster tiles on the matrix cores, inter-cluster edges beside them, one softmax
        {"name": "block_262k_bf16", "kind": "block", "nodes": 262144, "clusters": 64, "degree": 8.0, "outside": 0.05,
         "heads": 8, "dim": 8, "dtype": "bf16"},
        # a batch of 256 small graphs padded to 128 nodes and a virtual node
        {"name": "dense_b256_bf16", "kind": "dense", "batch": 256, "smallest": 16, "largest": 128, "heads": 8, "dim": 8,
         "dtype": "bf16"},
        # training steps of the slim node-level Graphormer: a small graph, a 64 K-node sequence, one of 870 K nodes with
        # 44 M edges
        {"name": "graphormer_train_4k_f32", "kind": "node_train", "model": "graphormer", "nodes": 4096, "degree": 8.0,
         "exponent": 2.5, "clusters": 1, "layers": 4, "heads": 8, "hidden": 64, "features": 128, "classes": 40, "dtype": "f32"},
        {"name": "graphormer_train_64k_f32", "kind": "node_train", "model": "graphormer", "nodes": 64000, "degree": 5.3,
         "exponent": 2.1, "clusters": 1, "layers": 4, "heads": 8, "hidden": 64, "features": 128, "classes": 40, "dtype": "f32"},
        {"name": "graphormer_train_870k_bf16", "kind": "node_train", "model": "graphormer", "nodes": 870000, "degree": 48.0,
         "exponent": 2.0, "clusters": 64, "layers": 4, "heads": 8, "hidden": 64, "features": 100, "classes": 47,
         "dtype": "bf16"},
        # a training step of the node-level GT in bf16
        {"name": "gt_train_64k_bf16", "kind": "node_train", "model": "gt", "nodes": 64000, "degree": 5.3, "exponent": 2.1,
         "clusters": 1, "layers": 4, "heads": 8, "hidden": 64, "features": 128, "classes": 40, "dtype": "bf16"},
        # evaluation of the ragged last part of an epoch
        {"name": "graphormer_eval_37605_f32", "kind": "node_eval", "model": "graphormer", "nodes": 37605, "degree": 5.3,
         "exponent": 2.1, "clusters": 1, "layers": 4, "heads": 8, "hidden": 64, "features": 128, "classes": 40, "dtype": "f32"},
        # a training step of the graph-level Graphormer on the batch of the dense case
        {"name": "graph_train_b256_bf16", "kind": "graph_train", "batch": 256, "smallest": 16, "largest": 128, "layers": 4,
         "heads": 8, "hidden": 64, "edge_type": "single_hop", "dtype": "bf16"},
        # a new batch of 64 000 nodes out of a larger graph, reordered into 8 clusters
        {"name": "batch_64k_of_256k", "kind": "batch", "nodes": 256000, "degree": 12.0, "exponent": 2.1, "clusters": 8,
         "take": 64000, "reorder": True},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["attention", "attention", "block", "dense", "node_train", "node_train", "node_train", "node_eval",
                       "graph_train", "graph_train", "batch"])
    dtype = rng.choice(["f32", "bf16"])
    if kind == "dense":
        largest = _log(rng, 12, 200)
        return {"kind": kind, "batch": _log(rng, 4, 256), "smallest": max(2, largest // 8), "largest": largest, "heads": 8,
                "dim": rng.choice([8, 8, 16]), "dtype": dtype}
    if kind == "graph_train":
        largest = _log(rng, 12, 160)
        return {"kind": kind, "batch": _log(rng, 4, 256), "smallest": max(2, largest // 8), "largest": largest, "layers": 4,
                "heads": 8, "hidden": 64, "edge_type": rng.choice(["single_hop", "single_hop", "multi_hop"]), "dtype": dtype}
    nodes = _log(rng, 1000, 500_000)
    degree = round(math.exp(rng.uniform(math.log(4), math.log(min(50, 1e7 / nodes)))), 1)
    if kind == "block":
        clusters = _log(rng, 4, 64)
        size = max(64, nodes // clusters)
        return {"kind": kind, "nodes": clusters * size, "clusters": clusters, "degree": degree,
                "outside": rng.choice([0.0, 0.02, 0.05, 0.2]), "heads": 8, "dim": 8, "dtype": "bf16"}
    case = {"kind": kind, "nodes": nodes, "degree": degree, "exponent": rng.choice([2.0, 2.1, 2.5]),
            "clusters": rng.choice([1, 8, 64])}
    if kind == "attention":
        heads, dim = rng.choice([(8, 8), (8, 8), (4, 16), (8, 16)])
        return dict(case, heads=heads, dim=dim, dtype=dtype, bias=rng.choice(["none", "edge", "edge_head"]))
    if kind == "batch":
        return dict(case, clusters=8, take=max(200, int(nodes * rng.uniform(0.1, 1.0))), reorder=rng.choice([True, True, False]))
    # features and classes: those of the node-level configurations and odd ones
    return dict(case, model=rng.choice(["graphormer", "graphormer", "gt"]), layers=4, heads=8, hidden=rng.choice([64, 64, 64, 128]),
                features=rng.choice([100, 128, 128, rng.randint(32, 500)]), classes=rng.choice([40, 47, rng.randint(3, 64)]),
                dtype=dtype)


# ---- inputs -------------------------------------------------------------------------------------------------------------

def _generator(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _edges(nodes, degree, exponent, clusters, g):
    """int64 [2, E]: power-law graph (expected degrees, simple, both directions, in random order), four of five edges inside
    the contiguous cluster of their first end when there are clusters, and a self-loop on every node at the end.  E depends
    on the sizes only: pairs lost to duplicates are replaced by spare draws, the last ones by pairs of any two nodes."""
    u = torch.rand(nodes, generator=g, device=DEV, dtype=torch.float64)
    w = u.pow(-1.0 / (exponent - 1.0))
    for _ in range(4):                      # the structural cut-off of a simple graph
        w = (w * (degree / w.mean())).clamp(max=math.sqrt(nodes * degree))
    cdf = torch.cumsum(w, 0)
    m = int(nodes * degree / 2)
    tries = m + m // 4 + 64
    rand = lambda: torch.rand(tries, generator=g, device=DEV, dtype=torch.float64)
    pick = lambda r: torch.searchsorted(cdf, r).clamp(max=nodes - 1)
    a, r = pick(rand() * cdf[-1]), rand()
    if clusters > 1:
        size = -(-nodes // clusters)
        ends = torch.arange(1, clusters + 1, device=DEV).mul(size).clamp(max=nodes)
        hi = cdf[ends - 1]
        lo = torch.cat([hi.new_zeros(1), hi[:-1]])
        c = a // size
        b = pick(torch.where(rand() < 0.8, lo[c] + r * (hi[c] - lo[c]), r * cdf[-1]))
    else:
        b = pick(r * cdf[-1])
    key = torch.unique((torch.minimum(a, b) * nodes + torch.maximum(a, b))[a != b])
    while key.numel() < m:
        a, b = torch.randint(0, nodes, (2, 2 * (m - key.numel()) + 64), generator=g, device=DEV)
        key = torch.unique(torch.cat([key, (torch.minimum(a, b) * nodes + torch.maximum(a, b))[a != b]]))
    key = key[torch.randperm(key.numel(), generator=g, device=DEV)[:m]]
    a, b = key // nodes, key % nodes
    loops = torch.arange(nodes, device=DEV)
    return torch.stack([torch.cat([a, b, loops]), torch.cat([b, a, loops])])


def _randn(shape, g, dtype):
    return torch.randn(shape, generator=g, device=DEV).to(dtype)


def _settle(model, dtype, seed):
    """The model on the GPU with weights of a trained layer's scale."""
    gen = torch.Generator().manual_seed(int(seed))
    with torch.no_grad():
        for p in model.parameters():
            if p.dim() == 1:
                p.add_(torch.randn(p.shape, generator=gen) * 0.05)
            else:
                p.copy_(torch.randn(p.shape, generator=gen) / math.sqrt(p.shape[-1]))
    return model.to(DEV, dtype)


def _small_graphs(case, g, dtype):
    """Collated batch of random graphs (edge probability 0.1) as the graph-level data loader hands it over."""
    b, s = case["batch"], case["largest"]
    sizes = torch.randint(case["smallest"], s + 1, (b,), generator=g, device=DEV)
    sizes[0] = s
    valid = torch.arange(s, device=DEV)[None, :] < sizes[:, None]
    upper = torch.triu(torch.rand(b, s, s, generator=g, device=DEV) < 0.1, 1)
    adj = (upper | upper.transpose(1, 2)) & valid[:, :, None] & valid[:, None, :]
    dist, path = floyd_warshall(adj.to(torch.uint8), sizes)
    pairs = valid[:, :, None] & valid[:, None, :]
    spatial = torch.where(pairs, dist.clamp(max=SPD_CLAMP) + 1, 0)
    kinds = torch.triu(torch.randint(1, 5, (b, s, s), generator=g, device=DEV), 1)
    kinds = ((kinds + kinds.transpose(1, 2)) * adj).unsqueeze(-1)
    bias = torch.zeros(b, s + 1, s + 1, device=DEV)
    bias[:, :, 1:].masked_fill_(~valid[:, None, :], float("-inf"))
    degree = torch.where(valid, (adj.sum(-1) + 1).clamp(max=63), 0)
    atoms = torch.randint(1, 64, (b, s, 1), generator=g, device=DEV) * valid.unsqueeze(-1)
    hops = gen_edge_input(5, path, kinds, sizes) + 1 if case.get("edge_type") == "multi_hop" else None
    return types.SimpleNamespace(x=atoms, in_degree=degree, out_degree=degree, attn_bias=bias.to(dtype), spatial_pos=spatial,
                                 attn_edge_type=kinds, edge_input=hops)


def prepare(case, seed):
    g = _generator(seed)
    dtype = DTYPES.get(case.get("dtype"))
    s = types.SimpleNamespace(kind=case["kind"])
    if s.kind == "attention":
        n, H, d = case["nodes"] + 1, case["heads"], case["dim"]
        edges = fix_edge_index(_edges(case["nodes"], case["degree"], case["exponent"], case["clusters"], g), case["nodes"])
        s.plan = GraphPlan(edges, n)
        s.q, s.k, s.v = (_randn((n, H, d), g, dtype).requires_grad_(True) for _ in range(3))
        s.grad = _randn((n, H, d), g, dtype)
        s.bias = None
        if case["bias"] == "edge_head":
            s.bias = (_randn((edges.shape[1], H), g, torch.float32) * 0.5).to(dtype).requires_grad_(True)
        elif case["bias"] == "edge":        # an embedding of a few distances
            table = _randn((7,), g, torch.float32) * 0.5
            s.bias = table[torch.randint(0, 7, (edges.shape[1],), generator=g, device=DEV)].to(dtype).requires_grad_(True)
    elif s.kind == "block":
        n, c = case["nodes"], case["clusters"]
        size = n // c
        tiles = int(n * case["degree"]) // (BLOCK * BLOCK * c) + 1
        first = torch.randint(0, size // BLOCK, (2, c, tiles), generator=g, device=DEV) * BLOCK
        first += (torch.arange(c, device=DEV) * size)[None, :, None]
        m = int(n * case["degree"] * case["outside"])
        rest = torch.randint(0, n, (2, m), generator=g, device=DEV)
        rest = rest[:, rest[0] // size != rest[1] // size].contiguous()
        s.tiles = TileSet(first.reshape(2, -1).t().cpu().numpy(), n, torch.device(DEV, torch.cuda.current_device()))
        s.plan = GraphPlan(rest, n, rows_with_edges_only=True)
        shape = (n, case["heads"], case["dim"])
        s.q, s.k, s.v = (_randn(shape, g, dtype).requires_grad_(True) for _ in range(3))
        s.grad = _randn(shape, g, dtype)
    elif s.kind == "dense":
        H, d = case["heads"], case["dim"]
        batch = _small_graphs(case, g, torch.float32)
        b, S = batch.attn_bias.shape[:2]
        # the layer multiplies q by sqrt(d): queries of this scale give logits of order one
        s.q = (_randn((b, S, H, d), g, torch.float32) / d).to(dtype).requires_grad_(True)
        s.k, s.v = (_randn((b, S, H, d), g, dtype).requires_grad_(True) for _ in range(2))
        table = _randn((SPD_CLAMP + 2, H), g, torch.float32) * 0.5
        bias = torch.zeros(b, S, S, H, device=DEV)
        bias[:, 1:, 1:] = table[batch.spatial_pos]
        s.bias = (bias.permute(0, 3, 1, 2) + batch.attn_bias.unsqueeze(1)).to(dtype).contiguous().requires_grad_(True)
        s.grad = _randn((b, S, H * d), g, dtype)
    elif s.kind in ("node_train", "node_eval"):
        n = case["nodes"]
        edges = _edges(n, case["degree"], case["exponent"], case["clusters"], g)
        build, tokens = (GT, 0) if case["model"] == "gt" else (Graphormer, 1)
        if tokens:
            edges = fix_edge_index(edges, n)
        s.plan = GraphPlan(edges, n + tokens)
        s.model = _settle(build(case["layers"], case["heads"], case["features"], case["hidden"], case["classes"], 1, 0.0, 0.0, 0.0,
                                case["hidden"], tokens), dtype, seed)
        s.model.train(s.kind == "node_train")
        s.x = _randn((n, case["features"]), g, dtype)
        s.y = torch.randint(0, case["classes"], (n,), generator=g, device=DEV)
    elif s.kind == "graph_train":
        s.batch = _small_graphs(case, g, dtype)
        s.model = _settle(GraphLevelGraphormer(case["layers"], case["heads"], case["hidden"], 0.0, 0.0, case["hidden"], "ZINC",
                                               case["edge_type"], 5, 0.0, 1), dtype, seed)
        s.model.train()
        s.y = torch.randn(case["batch"], generator=g, device=DEV)
    else:
        n = case["nodes"]
        s.n, s.reorder, s.k = n, case["reorder"], case["clusters"]
        # one graph and one choice of nodes per case, under other node names and in another edge order for every seed: the
        # number of edges that stay in the batch is a property of the case
        fixed = _generator(20)
        edges = _edges(n, case["degree"], case["exponent"], case["clusters"], fixed)
        take = torch.randperm(n, generator=fixed, device=DEV)[:case["take"]]
        name = torch.randperm(n, generator=g, device=DEV)
        s.edges = name[edges][:, torch.randperm(edges.shape[1], generator=g, device=DEV)].contiguous()
        take = take[torch.randperm(take.numel(), generator=g, device=DEV)]
        s.take = name[take]
        # what the graph partitioner says about the batch: the global node and the clusters of its nodes
        s.parts = torch.cat([take.new_zeros(1), take * s.k // n])
        s.x = _randn((n, 128), g, torch.float32)
        s.y = torch.randint(0, 40, (n,), generator=g, device=DEV)
    return s


# ---- one pass -----------------------------------------------------------------------------------------------------------

def _gradients(model):
    """The gradients as the one flat vector that an all-reduce or a gradient clip takes."""
    return torch._utils._flatten_dense_tensors([p.grad for p in model.parameters() if p.grad is not None])


def run(s):
    if s.kind == "attention":
        out = sparse_attention(s.q, s.k, s.v, edge_bias=s.bias, plan=s.plan)
        leaves = [s.q, s.k, s.v] + ([] if s.bias is None else [s.bias])
        return [out, *torch.autograd.grad(out, leaves, s.grad)]
    if s.kind == "block":
        out = block_attention(s.q, s.k, s.v, s.tiles, plan=s.plan)
        return [out, *torch.autograd.grad(out, [s.q, s.k, s.v], s.grad)]
    if s.kind == "dense":
        out = dense_attention(s.q, s.k, s.v, s.bias)
        return [out, *torch.autograd.grad(out, [s.q, s.k, s.v, s.bias], s.grad)]
    if s.kind == "node_train":
        s.model.zero_grad(set_to_none=True)
        out = s.model(s.x, None, s.plan, attn_type="sparse")
        loss = nll_loss(out.float(), s.y)
        loss.backward()
        return {"loss": loss, "out": out, "gradients": _gradients(s.model)}
    if s.kind == "node_eval":
        with torch.no_grad():
            return s.model(s.x, None, s.plan, attn_type="sparse")
    if s.kind == "graph_train":
        s.model.zero_grad(set_to_none=True)
        out = s.model(s.batch)
        loss = torch.nn.functional.l1_loss(out.float().view(-1), s.y)
        loss.backward()
        return {"loss": loss, "out": out, "gradients": _gradients(s.model)}
    x, y, edges, _ = prepare_batch(s.x, s.y, s.take, s.edges, s.n, s.k, BLOCK, s.parts, reorder=s.reorder)
    plan = GraphPlan(edges, s.take.numel() + 1)
    return {"x": x, "y": y, "edges": edges, "by_destination": plan.edge_order(), "by_source": plan.edge_order_src()}


# ---- what a pass cannot do without ----------------------------------------------------------------------------------------

def _edge_count(case, tokens):
    return int(case["nodes"] * case["degree"]) + case["nodes"] + 2 * tokens * case["nodes"]


def work(case):
    size = 2 if case.get("dtype") == "bf16" else 4
    kind = case["kind"]
    if kind == "attention":
        n, E, row = case["nodes"] + 1, _edge_count(case, 1), case["heads"] * case["dim"]
        bias = {"none": 0, "edge": size, "edge_head": size * case["heads"]}[case["bias"]]
        # q, k, v, out and the gradients once each, three index walks, the bias and its gradient
        return {"bytes": 8 * n * row * size + 3 * E * 4 + 2 * E * bias, "flops": 14 * E * row}
    if kind == "block":
        n, row = case["nodes"], case["heads"] * case["dim"]
        E = n * case["degree"] * (1 + case["outside"])
        return {"bytes": 8 * n * row * size, "flops": 14 * E * row}
    if kind == "dense":
        b, S, row = case["batch"], case["largest"] + 1, case["heads"] * case["dim"]
        return {"bytes": 8 * b * S * row * size + 2 * b * case["heads"] * S * S * size, "flops": 14 * b * S * S * row}
    if kind in ("node_train", "node_eval"):
        n, C, L, tokens = case["nodes"], case["hidden"], case["layers"], 0 if case["model"] == "gt" else 1
        E, wide = _edge_count(case, tokens), 2 * C if case["model"] == "gt" else C
        forward = L * (2 * n * C * (4 * C + 2 * wide) + 4 * E * C) + 2 * n * C * (case["features"] + case["classes"])
        # the features, the edges and the labels in, the log-probabilities out; a training step also writes each layer's
        # input, q, k, v and attention rows for its backward and reads them there
        once = n * case["features"] * size + 8 * E + n * case["classes"] * size
        kept = 2 * L * 5 * n * C * size + 8 * n
        train = kind == "node_train"
        return {"bytes": once + (kept if train else L * 4 * n * C * size), "flops": forward * (3 if train else 1)}
    if kind == "graph_train":
        b, S, C, L = case["batch"], case["largest"] + 1, case["hidden"], case["layers"]
        pairs = b * S * S
        forward = L * (2 * b * S * C * 6 * C + 4 * pairs * C)
        ids = 8 * pairs * (6 if case["edge_type"] == "multi_hop" else 2)
        return {"bytes": ids + pairs * size + 2 * L * 5 * b * S * C * size, "flops": 3 * forward}
    E, t = _edge_count(case, 0), case["take"]
    kept = int(E * (t / case["nodes"]) ** 2) + 3 * t
    return {"bytes": 16 * E + 32 * kept + t * (2 * 128 * 4 + 16), "flops": 0}


def tolerance(case):
    if case["kind"] == "batch":
        return "exact"
    if case["dtype"] == "bf16":
        return {"rel": 2e-2 if case["kind"] in ("node_train", "node_eval", "graph_train") else 1e-2}
    return {"rel": 5e-5 if case["kind"] in ("node_train", "node_eval", "graph_train") else 1e-5}
