"""What keeps a model off the whole-model operators, as far as the model itself decides it (no GPU needed): a model that they do not
cover has to run module by module, not raise and not lose what its modules do."""
import pytest
import torch
import torch.nn as nn

from torchgt_amd import GT, GraphLevelGraphormer, Graphormer
from torchgt_amd.module_tree import model_parameters


def build(kind, dropout=0.0, input_dropout=0.0, attention_dropout=0.0, layers=2):
    if kind == "graph":
        return GraphLevelGraphormer(layers, 8, 64, dropout, input_dropout, 64, "ZINC", "single_hop", 5, attention_dropout, 1)
    cls, tokens = (GT, 0) if kind == "gt" else (Graphormer, 1)
    return cls(layers, 8, 16, 64, 4, 1, dropout, input_dropout, attention_dropout, 64, tokens)


def parameters(model):
    return model._operator_parameters() if isinstance(model, GraphLevelGraphormer) else model_parameters(model, torch.float32)


KINDS = ["graphormer", "gt", "graph"]


class Attention(nn.Module):      # a module of the user's own, without the parameters of the library's
    def forward(self, x, attn_bias=None, edge_index=None, attn_type=None):
        return x


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("where", ["layer", "attention", "last", "no layers"])
def test_a_module_of_another_kind_in_the_tree(kind, where):
    """``parameters`` says no, before and after, and yes again once the library's module is back."""
    model = build(kind)
    assert parameters(model) is not None
    owner, name = {"layer": (model.layers, "0"), "attention": (model.layers[1], "self_attention"), "no layers": (model, "layers"),
                   "last": (model, "MLP_layer" if kind == "gt" else "final_ln")}[where]
    kept = owner._modules[name]
    setattr(owner, name, {"last": nn.Identity(), "no layers": nn.ModuleList()}.get(where, Attention()))
    assert parameters(model) is None and parameters(model) is None
    setattr(owner, name, kept)
    assert parameters(model) is not None


def called(model):
    return [(path, model.get_submodule(path)) for path, _ in model._called_modules()]


LISTENERS = {
    "forward hook": lambda m: m.register_forward_hook(lambda *a: None),
    "forward pre-hook": lambda m: m.register_forward_pre_hook(lambda *a: None),
    "backward hook": lambda m: m.register_full_backward_hook(lambda *a: None),
    "backward pre-hook": lambda m: m.register_full_backward_pre_hook(lambda *a: None),
}


@pytest.mark.parametrize("kind", KINDS)
def test_modules_that_somebody_listens_to_are_called(kind):
    model = build(kind)
    assert len(called(model)) >= 2 * 5 + 1
    for path, m in called(model):
        for name, listen in LISTENERS.items():
            handle = listen(m)
            assert parameters(model) is None, (path, name)
            handle.remove()
            assert parameters(model) is not None, (path, name)
        m.forward = lambda *a, **k: None
        assert parameters(model) is None, path
        del m.forward
        cls = type(m)
        m.__class__ = type("Own", (cls,), {"forward": lambda *a, **k: None})
        assert parameters(model) is None, path
        m.__class__ = cls
        assert parameters(model) is not None, path
        forward = cls.forward
        cls.forward = lambda *a, **k: None
        try:
            assert parameters(model) is None, path
        finally:
            cls.forward = forward
    for listen in (nn.modules.module.register_module_forward_hook, nn.modules.module.register_module_forward_pre_hook,
                   nn.modules.module.register_module_full_backward_hook):
        handle = listen(lambda *a: None)
        assert parameters(model) is None
        handle.remove()
    assert parameters(model) is not None


def test_layers_of_unlike_head_counts():
    """Every layer has its own number of heads: the operators take one for all."""
    for kind in KINDS:
        model, other = build(kind), build(kind)
        other.layers[1].self_attention.num_heads = 4
        model.layers[1] = other.layers[1]
        assert parameters(model) is None


@pytest.mark.parametrize("kind", KINDS)
def test_every_dropout_has_its_own_mode(kind):
    model = build(kind, dropout=0.1, input_dropout=0.3)
    assert parameters(model) is None
    model.eval()
    assert parameters(model) is not None
    dropouts = [m for _, m in called(model) if isinstance(m, nn.Dropout)]
    assert len(dropouts) == (3 if kind == "gt" else 5)
    for m in dropouts:
        m.train()      # drops in a model in eval mode
        assert parameters(model) is None
        m.eval()
    model.train()
    for m in dropouts:
        m.eval()       # (the model's own flag says nothing)
    assert model.training and parameters(model) is not None


def test_attention_dropout_has_each_modules_mode():
    model = build("graph", attention_dropout=0.5)
    cores = [layer.self_attention.dist_attn.local_attn for layer in model.layers]
    assert parameters(model) is not None and cores[0].dropout_at_work() == 0.5
    cores[1].eval()      # the operator has one rate for all layers
    assert parameters(model) is None
    cores[0].eval()
    assert parameters(model) is not None and cores[0].dropout_at_work() == 0.0


@pytest.mark.parametrize("kind", KINDS)
def test_a_data_parallel_wrapper_gets_gradients_layer_by_layer(kind, tmp_path):
    """Its reduction overlaps with the backward only if gradients become ready one after the other; gradients that nobody waits for (no
    wrapper, no gradients wanted) leave the operators their work."""
    model, alone = build(kind), build(kind)
    assert parameters(model) is not None
    torch.distributed.init_process_group("gloo", init_method=f"file://{tmp_path}/store", rank=0, world_size=1)
    try:
        assert parameters(model) is not None
        wrapped = torch.nn.parallel.DistributedDataParallel(model, find_unused_parameters=True)
        assert parameters(model) is None and parameters(alone) is not None
        with torch.no_grad():
            assert parameters(model) is not None
        del wrapped
        handle = alone.layers[0].self_attention.linear_q.weight.register_post_accumulate_grad_hook(lambda p: None)
        assert parameters(alone) is None
        handle.remove()
    finally:
        torch.distributed.destroy_process_group()
