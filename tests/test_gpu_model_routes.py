"""Which calls the whole-model operators take: a call that they do not cover gives what the layers one by one give."""
import types

import pytest
import torch

from oracle import encoder_layer as oel
from torchgt_amd import GT, GraphLevelGraphormer, Graphormer, GraphPlan
from torchgt_amd.encoder import EncoderLayer

pytestmark = pytest.mark.gpu


def edges_of(n, tokens, seed):
    g = torch.Generator().manual_seed(seed)
    e = torch.cat([torch.randint(0, n, (2, 4 * n), generator=g), torch.arange(n).repeat(2, 1)], 1)
    for t in range(tokens):      # a token is joined to every row in front of it
        old = torch.arange(n + t)
        e = torch.cat([e + 1, torch.stack([torch.zeros_like(old), old + 1]), torch.stack([old + 1, torch.zeros_like(old)])], 1)
    return e


def scaled(model, seed, dtype, device):
    g = torch.Generator().manual_seed(seed)
    with torch.no_grad():
        for p in model.parameters():
            p.copy_(p + torch.randn(p.shape, generator=g) * 0.1 if p.dim() == 1 else torch.randn(p.shape, generator=g) / p.shape[-1] ** 0.5)
    return model.to(device, dtype)


@pytest.mark.parametrize("hidden", [64, 128])
@pytest.mark.parametrize("tokens", [0, 1, 2, 3])
def test_token_counts(cuda, tokens, hidden):
    """Rows 1 .. of the sequence come back (models/graphormer_dist_node_level.py:391) for any number of global tokens."""
    n, layers, heads, classes = 100, 2, 8, 7
    print(f"tokens case: {tokens} hidden={hidden}", flush=True)
    torch.manual_seed(tokens)
    model = scaled(Graphormer(layers, heads, 20, hidden, classes, 1, 0.0, 0.0, 0.0, hidden, tokens), 2, torch.float32, cuda)
    x, e = torch.randn(n, 20), edges_of(n, tokens, 3)
    want = torch.from_numpy(oel.graphormer_forward(x.numpy(), {k: v.double().cpu().numpy() for k, v in model.state_dict().items()}, e.numpy(), layers, heads))
    plan = GraphPlan(e.to(cuda), n + tokens)
    w = torch.randn(want.shape, generator=torch.Generator().manual_seed(4)).to(cuda)
    grads = []
    for one in (True, False):
        model.one_operator = one
        model.zero_grad(set_to_none=True)
        out = model(x.to(cuda), None, plan, attn_type="sparse")
        assert out.shape == want.shape == (n + tokens - 1, classes)
        assert float((out.double().cpu() - want).abs().max()) <= 3e-5 * float(want.abs().max())
        (out * w).sum().backward()
        grads.append(torch.cat([p.grad.flatten() for p in model.parameters() if p.grad is not None]))
    assert float((grads[0] - grads[1]).norm()) <= 2e-5 * float(grads[1].norm())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("kind,hidden,classes", [("gt", 64, 40), ("gt", 128, 47), ("graphormer", 64, 40), ("graphormer", 128, 40)])
def test_autocast(cuda, kind, hidden, classes, dtype):
    """Under autocast the log-probabilities are float32, whichever way the model runs, and the gradients those of the model's dtype."""
    n, layers, heads = 200, 2, 8
    print(f"autocast case: {kind} hidden={hidden} {dtype}", flush=True)
    cls, tokens = (GT, 0) if kind == "gt" else (Graphormer, 1)
    torch.manual_seed(1)
    model = scaled(cls(layers, heads, 32, hidden, classes, 1, 0.0, 0.0, 0.0, hidden, tokens), 2, dtype, cuda)
    x, plan = torch.randn(n, 32).to(cuda, dtype), GraphPlan(edges_of(n, tokens, 3).to(cuda), n + tokens)
    w = torch.randn(n, classes, generator=torch.Generator().manual_seed(4)).to(cuda)
    got = []
    for one in (True, False):
        model.one_operator = one
        model.zero_grad(set_to_none=True)
        with torch.autocast("cuda", torch.bfloat16):
            out = model(x, None, plan, attn_type="sparse")
            loss = (out.float() * w).sum()
        loss.backward()
        assert out.dtype == torch.float32
        got.append([out.detach(), torch.cat([p.grad.float().flatten() for p in model.parameters() if p.grad is not None])])
    for a, b in zip(*got):      # two orders of float32 sums; bf16: two orders of roundings
        assert float((a - b).norm()) <= (2e-5 if dtype == torch.float32 else 3e-2) * float(b.norm())


class OwnLayer(EncoderLayer):
    calls = 0

    def forward(self, *args, **kwargs):
        OwnLayer.calls += 1
        return super().forward(*args, **kwargs)


@pytest.mark.parametrize("path", ["input_dropout", "layers.0", "layers.1.self_attention", "layers.1.self_attention.dist_attn", "layers.0.self_attention.dist_attn.local_attn",
                                  "layers.0.self_attention_dropout", "layers.1.ffn", "layers.1.ffn_dropout"])
def test_hooks_fire_and_may_change_what_they_see(cuda, path):
    """A hook on a module of the model sees one call a pass, and what it returns goes on through the model."""
    n = 100
    torch.manual_seed(1)
    model = scaled(Graphormer(2, 8, 32, 64, 5, 1, 0.0, 0.0, 0.0, 64, 1), 2, torch.float32, cuda)
    x, plan = torch.randn(n, 32).to(cuda), GraphPlan(edges_of(n, 1, 3).to(cuda), n + 1)
    before = model(x, None, plan, attn_type="sparse")
    seen = []
    handle = model.get_submodule(path).register_forward_hook(lambda m, args, out: seen.append(1) or (tuple(0.5 * t for t in out) if isinstance(out, tuple) else 0.5 * out))
    changed = model(x, None, plan, attn_type="sparse")
    assert seen == [1] and float((changed - before).abs().max()) > 1e-3
    handle.remove()
    after = model(x, None, plan, attn_type="sparse")
    assert seen == [1] and torch.equal(after, before)


def test_a_subclass_of_the_layer_keeps_its_forward(cuda):
    n = 100
    torch.manual_seed(1)
    model = scaled(Graphormer(2, 8, 32, 64, 5, 1, 0.0, 0.0, 0.0, 64, 1), 2, torch.float32, cuda)
    x, plan = torch.randn(n, 32).to(cuda), GraphPlan(edges_of(n, 1, 3).to(cuda), n + 1)
    before = model(x, None, plan, attn_type="sparse")
    model.layers[1].__class__ = OwnLayer
    OwnLayer.calls = 0
    out = model(x, None, plan, attn_type="sparse")
    assert OwnLayer.calls == 1 and float((out - before).abs().max()) <= 1e-5 * float(before.abs().max())


@pytest.mark.parametrize("where", ["input_dropout", "layers.1.ffn_dropout", "layers.0.self_attention_dropout"])
def test_one_dropout_in_training_mode(cuda, where):
    """A dropout module set to training in a model in eval mode drops (and the others don't), as does none in a model in training mode
    whose dropouts are in eval mode."""
    n = 100
    torch.manual_seed(1)
    model = scaled(Graphormer(2, 8, 32, 64, 5, 1, 0.2, 0.2, 0.0, 64, 1), 2, torch.float32, cuda).eval()
    x, plan = torch.randn(n, 32).to(cuda), GraphPlan(edges_of(n, 1, 3).to(cuda), n + 1)
    run = lambda: model(x, None, plan, attn_type="sparse").detach()
    still = run()
    dropout = model.get_submodule(where)
    dropout.train()
    with torch.random.fork_rng(devices=[cuda]):
        torch.manual_seed(5)
        dropped = run()
        seen = []
        handle = dropout.register_forward_hook(lambda m, args, out: seen.append(int((out == 0).sum()) > args[0].numel() // 10))
        torch.manual_seed(5)
        assert torch.equal(run(), dropped) and seen == [True]
        handle.remove()
    assert float((dropped - still).abs().max()) > 1e-3
    model.train()
    for m in model.modules():
        if isinstance(m, torch.nn.Dropout):
            m.eval()
    assert torch.equal(run(), still)


def test_bias_gradients_of_a_large_batch_go_into_a_running_sum(cuda):
    """The layers share one bias; where its gradient is large only a running sum and the next layer's are held."""
    b, s, layers = 64, 384, 5
    torch.manual_seed(1)
    model = scaled(GraphLevelGraphormer(layers, 8, 64, 0.0, 0.0, 64, "ZINC", "single_hop", 5, 0.0, 1), 2, torch.float32, cuda)
    g = torch.Generator().manual_seed(3)
    ids = lambda hi, *shape: torch.randint(0, hi, shape, generator=g).to(cuda)
    batch = types.SimpleNamespace(x=ids(64, b, s, 1), in_degree=ids(64, b, s), out_degree=ids(64, b, s), attn_bias=torch.zeros(b, s + 1, s + 1, device=cuda),
                                  spatial_pos=ids(40, b, s, s), attn_edge_type=ids(64, b, s, s, 1))
    one_bias = b * 8 * (s + 1) ** 2 * 4
    assert one_bias > 256 << 20
    got = []
    for one in (True, False):
        model.one_operator = one
        model.zero_grad(set_to_none=True)
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        model(batch).sum().backward()
        torch.cuda.synchronize()
        got.append((torch.cuda.max_memory_allocated() - before, torch.cat([p.grad.flatten() for p in model.parameters() if p.grad is not None])))
    assert got[0][0] <= 4.5 * one_bias      # the bias, the sum, one layer's gradient, all rows of the step (1 to 1.5 of a bias)
    assert float((got[0][1] - got[1][1]).norm()) <= 3e-5 * float(got[1][1].norm())


@pytest.mark.parametrize("kind,hidden", [("gt", 64), ("gt", 128), ("graphormer", 64), ("graphormer", 128)])
def test_forward_mode_is_refused_not_dropped(cuda, kind, hidden):
    """A tangent of x that no operator carries on raises, with gradients off too."""
    n, tokens = 50, 0 if kind == "gt" else 1
    torch.manual_seed(1)
    model = (Graphormer if tokens else GT)(2, 8, 32, hidden, 5, 1, 0.0, 0.0, 0.0, hidden, tokens).to(cuda).requires_grad_(False)
    x, plan = torch.randn(n, 32).to(cuda), GraphPlan(edges_of(n, tokens, 3).to(cuda), n + tokens)
    for one in (True, False):
        model.one_operator = one
        with torch.autograd.forward_ad.dual_level(), torch.no_grad():
            with pytest.raises(RuntimeError, match="jvp"):
                model(torch.autograd.forward_ad.make_dual(x, torch.ones_like(x)), None, plan, attn_type="sparse")
        assert model(x, None, plan, attn_type="sparse").shape == (n, 5)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("hidden", [64, 128])
def test_a_batch_without_nodes(cuda, dtype, hidden):
    """No node, the global token alone: no rows come back, and every gradient is zero."""
    torch.manual_seed(1)
    model = Graphormer(2, 8, 32, hidden, 5, 1, 0.0, 0.0, 0.0, hidden, 1).to(cuda, dtype)
    x, plan = torch.zeros(0, 32, device=cuda, dtype=dtype), GraphPlan(torch.zeros(2, 1, dtype=torch.long, device=cuda), 1)
    for one in (True, False):
        model.one_operator = one
        model.zero_grad(set_to_none=True)
        out = model(x, None, plan, attn_type="sparse")
        assert out.shape == (0, 5)
        out.float().sum().backward()
        grads = [p.grad for p in model.parameters() if p.grad is not None]
        assert len(grads) > 30 and not any(g.any() for g in grads)
        with torch.no_grad():
            assert model(x, None, plan, attn_type="sparse").shape == (0, 5)
