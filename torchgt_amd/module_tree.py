"""What the whole-model and whole-layer operators need to know of the modules they pass by.

An operator that does the work of a tree of modules reads their parameters and calls none of them.  That is the same thing only while
every module it passes by is the library's own and nobody listens to it: ``plain`` looks at that on every call."""
import weakref

import torch
import torch.distributed
import torch.nn as nn
from torch.nn.modules import module as _torch_module

from . import _ext


def kind(cls):
    """A class with the ``forward`` it has now, for ``plain``."""
    return cls, cls.forward


DROPOUT = kind(nn.Dropout)


def plain(module, cls, forward):
    """Whether calling the module would run ``forward`` of exactly this class and nothing else: no subclass, no ``forward`` put on the
    object or the class, no hook, no compiled call."""
    d = module.__dict__
    return type(module) is cls and cls.forward is forward and "forward" not in d and not (
        d["_forward_hooks"] or d["_forward_pre_hooks"] or d["_backward_hooks"] or d["_backward_pre_hooks"] or "_compiled_call_impl" in d)


def all_plain(*pairs):
    """``plain`` for (module, kind) pairs, and no hook on every module of the process."""
    return not watched_everywhere() and all(plain(m, *k) for m, k in pairs)


def at_work(dropout):
    return dropout.training and dropout.p > 0


def watched_everywhere():
    m = _torch_module
    return bool(m._global_forward_hooks or m._global_forward_pre_hooks or m._global_backward_hooks or m._global_backward_pre_hooks)


class OneWalk(nn.Module):
    """``parameters()`` of a model in one walk over its modules.  ``zero_grad``, a gradient clip and a flattening all-reduce each ask for
    them on every step, and ``nn.Module`` spells out the name of every parameter through a generator per module for it: 92 us for
    the 72 parameters of four layers, 43 here (half a step of 4 K nodes is host time).  Names are only left out where nobody could
    see them: a class or an object that brings its own ``named_parameters`` or ``named_modules`` is asked in the general way."""

    def parameters(self, recurse=True):
        if not recurse or not _plain_names(type(self)) or not _NAMES.isdisjoint(self.__dict__):
            yield from super().parameters(recurse)
            return
        seen, parents, known, stack = set(), set(), {type(self)}, [self]
        while stack:
            m = stack.pop()
            d = m.__dict__
            if type(m) not in known or "named_modules" in d:      # (that is all the general way asks a child for)
                if not _plain_names(type(m)) or "named_modules" in d or "_parameters" not in d or "_modules" not in d:
                    yield from [q for q in super().parameters() if id(q) not in seen]
                    return
                known.add(type(m))
            own, children = d["_parameters"], d["_modules"]
            if children:
                if id(m) in parents:      # (a leaf that is there twice has nothing new the second time)
                    continue
                parents.add(id(m))
            if own:
                for p in own.values():
                    if p is not None and id(p) not in seen:
                        seen.add(id(p))
                        yield p
            if children:
                for child in reversed(children.values()):
                    if child is not None:
                        stack.append(child)


_NAMES = {"named_parameters", "named_modules", "_named_members"}


def _plain_names(cls):
    M = nn.Module
    return cls.named_parameters is M.named_parameters and cls.named_modules is M.named_modules and cls._named_members is M._named_members


class ModuleTree:
    """Where a model's parameters are: for the whole-model operators, whose host time is counted in microseconds, the
    attribute look-ups of seventy parameters through ``nn.Module`` would be a third of it.  Remembers the dictionaries of the
    modules, not the parameters, and notices when a module of the tree was exchanged (``current``).

    names: the parameters in the operator's order; norms: the modules whose ``eps`` it takes; called: (path, kind) of the modules that
    the model calls when it runs module by module."""

    def __init__(self, root, names, norms, called):
        self.links, self.slots, self.norms, self.called, self.dropouts, self.layers = [], [], [], [], [], []
        seen = set()

        def step(module, name):
            child = module._modules.get(name)
            if (id(module), name) not in seen:
                seen.add((id(module), name))
                self.links.append((module._modules, name, child))
            return child

        def at(path):
            m = root
            for part in path:
                m = step(m, part) if m is not None else None
            return m

        self.count = len(root.layers)
        self.all_layers = step(root, "layers")._modules
        self.missing = self.count == 0      # a module of the names is not there: somebody's own module stands in its place
        for full in names:
            *path, leaf = full.split(".")
            m = at(path)
            if m is None:
                self.missing = True
                return
            self.slots.append((m._parameters, leaf))
        for path in norms:
            m = at(path.split("."))
            if m is None or "eps" not in m.__dict__:
                self.missing = True
                return
            self.norms.append(m.__dict__)
        for path, (cls, forward) in called:
            m = at(path.split("."))
            if m is None:
                self.missing = True
                return
            self.called.append((m, m.__dict__, cls))
            if cls is nn.Dropout:
                self.dropouts.append(m.__dict__)
        self.classes = list({kind for _, kind in called})
        self.layers = [(layer, layer.__dict__, layer._modules.get("self_attention")) for layer in self.all_layers.values()]

    def current(self):
        if len(self.all_layers) != self.count:
            return False
        for d, name, child in self.links:
            if d.get(name) is not child:
                return False
        return True

    def parameters(self, dtype):
        """(parameters, eps of the norms), each in order, or None: one is absent or has another dtype, a module is not plain or was asked
        to run step by step, or dropout is at work (each dropout module has its own mode, whatever the model's)."""
        if self.missing or watched_everywhere():
            return None
        for cls, forward in self.classes:
            if cls.forward is not forward:
                return None
        for m, d, cls in self.called:      # ``plain``, without a call for each of the thirty
            if type(m) is not cls or "forward" in d or d["_forward_hooks"] or d["_forward_pre_hooks"] or d["_backward_hooks"] or \
                    d["_backward_pre_hooks"] or "_compiled_call_impl" in d:
                return None
        for d in self.dropouts:
            if d["training"] and d["p"] > 0:
                return None
        heads = None
        for layer, d, att in self.layers:
            if "one_operator" in d or not layer.one_operator or not att.one_operator or att.num_heads != (heads or att.num_heads):
                return None
            heads = att.num_heads
        P = [d.get(name) for d, name in self.slots]
        for p in P:
            if p is None or p.dtype is not dtype:
                return None
        return P, [d["eps"] for d in self.norms]


def gradients_watched(parameters):
    """Whether a data-parallel wrapper reduces these gradients while the backward goes on.  An operator for the whole model hands over
    all of them at its end, its layers one by one hand over a layer's at a time: such a wrapper gets the layers.  Asked in jobs with a
    process group only; gradients that are reduced after the backward (one flat all-reduce) do not ask for anything else."""
    d = torch.distributed
    return d.is_available() and d.is_initialized() and torch.is_grad_enabled() and _ext.op("gradients_watched")(parameters)


_TREES = weakref.WeakKeyDictionary()      # model -> ModuleTree (which holds the model's modules, not the model)


def model_parameters(model, dtype):
    """(parameters, eps of the norms) of a model in the order of its whole-model operators, or None where they do not cover its state."""
    tree = _TREES.get(model)
    if tree is None or not tree.current():
        tree = _TREES[model] = ModuleTree(model, model._parameter_names(), model._norm_names(), model._called_modules())
    found = tree.parameters(dtype)
    return None if found is None or gradients_watched(found[0]) else found
