"""The state of a model's modules as it is now, for calls that read parameters past ``nn.Module.__call__`` and compute
what the methods of the package's classes would.

A program may exchange any parameter or module between two calls (``load_state_dict(assign=True)``, a new
``nn.Parameter``, another head).  What a call has prepared from the modules is used again only while
``ModelState`` sees the same ones in the same state; each call looks at all of them (12 layers: 0.12 ms)."""

from __future__ import annotations

from operator import attrgetter, is_

import torch
from torch import nn

from ._lib import raw_stream

__all__ = ["Methods", "ModelState", "Prepared", "Sources", "plain_modules", "walk"]

_hooks_of = attrgetter("_forward_hooks", "_forward_pre_hooks", "_backward_hooks", "_backward_pre_hooks")
_global_hooks = tuple(getattr(nn.modules.module, f"_global_{n}_hooks") for n in ("forward", "forward_pre", "backward", "backward_pre"))
_forwards = tuple((c, c.forward) for c in (nn.Linear, nn.LayerNorm, nn.GELU, nn.Sequential, nn.Embedding))


def plain_modules(modules, classes) -> bool:
    """Whether calling these modules is nothing but the forward of these classes: no subclass, no hook, no function of
    a program's own in the place of a method."""
    return (list(map(type, modules)) == list(classes) and not any(map(any, map(_hooks_of, modules))) and not any(_global_hooks)
            and not any("forward" in m.__dict__ for m in modules) and all(c.forward is f for c, f in _forwards)
            and all(m.approximate == "none" for m in modules if type(m) is nn.GELU))


class Methods:
    """The methods of a class that a prepared call stands for, as they are at import: ``of(obj)`` while nothing
    has taken the place of one of them, in a subclass, in the class or in the object."""

    def __init__(self, cls, *names):
        self._functions, self._names = [(n, getattr(cls, n)) for n in names], frozenset(names)

    def of(self, *objects) -> bool:
        return (all(getattr(t, n, None) is f for t in set(map(type, objects)) for n, f in self._functions)
                and all(self._names.isdisjoint(o.__dict__) for o in objects))


def walk(roots):
    """The modules of the trees below ``roots`` at the moment, and the entries of their parameter tables."""
    modules, parameters = list(roots), []
    for m in modules:  # (grows while it is walked)
        below, own = m._modules, m._parameters
        if below:
            modules += [c for c in below.values() if c is not None]
        if own:
            parameters += own.values()
    return modules, parameters


def _same(a, b) -> bool:
    return a is not None and len(a) == len(b) and all(map(is_, a, b))


def _values_at(tensors) -> tuple:
    """Where the tensors' values lie and how often they were written to."""
    return [p._version for p in tensors], list(map(torch.Tensor.data_ptr, tensors))


class Sources:
    """The tensors that something was prepared from: ``unchanged(tensors)`` while the same objects hold the same
    values at the same place.  They and their memory are held, so that neither an object nor an address
    that the comparison knows can come back as something else."""

    def __init__(self, tensors):
        self._tensors, self._facts = list(tensors), _values_at(tensors)
        self._storages = [t.untyped_storage() for t in self._tensors]

    def unchanged(self, tensors) -> bool:
        return _same(self._tensors, tensors) and _values_at(tensors) == self._facts


def capturing(device) -> bool:
    return device.type == "cuda" and torch.cuda.is_current_stream_capturing()


class Prepared:
    """Tensors that are made once, on the current stream, and read by calls on any: ``use()`` in front of every call
    on the current stream orders it behind the making, and keeps the memory from being given away under it
    when the tensors are dropped."""

    def __init__(self, tensors):
        self.tensors = tuple(tensors)
        self._device = next((t.device for t in self.tensors if t.is_cuda), None)
        if self._device is not None:
            self._home = raw_stream(self._device)
            self._streams = {self._home}

    def use(self) -> tuple:
        # (a recording cannot wait for what lies outside of it; it begins with everything in front of it done)
        if (self._device is not None and raw_stream(self._device) not in self._streams
                and not torch.cuda.is_current_stream_capturing()):
            stream = torch.cuda.current_stream(self._device)
            # behind what the making stream has been given so far: no event has to be kept for calls that stay on it
            try:
                home = (torch.cuda.ExternalStream(self._home, device=self._device) if self._home
                        else torch.cuda.default_stream(self._device))
                stream.wait_event(home.record_event())
            except RuntimeError:  # a stream of somebody else's making, gone since
                torch.cuda.synchronize(self._device)
            for t in self.tensors:
                if t.is_cuda:
                    t.record_stream(stream)
            self._streams.add(stream.cuda_stream)
        return self.tensors


class ModelState:
    """``look(roots, *tensors)`` gives a number that is another one whenever anything that a prepared call may have
    taken from the modules below ``roots`` has changed since the last look: which modules and parameters
    there are, where their values lie, whether they were written to, the constants of norms, attention
    and head."""

    # attributes of the package's modules, of LayerNorm and of GELU that enter the computation
    CONSTANTS = ("eps", "n_heads", "head_dim", "std_min", "num_components", "dim_y", "approximate")

    def __init__(self):
        self.generation = 0
        self._modules = self._types = self._parameters = self._sources = self._constants = self._values = None

    def look(self, roots, *tensors) -> int:
        modules, parameters = walk(roots)
        parameters += tensors
        types = list(map(type, modules))
        if not (_same(self._modules, modules) and types == self._types and _same(self._parameters, parameters)
                and self._sources.unchanged(self._tensors) and [d.get(n) for d, n in self._constants] == self._values):
            self.generation += 1
            self._modules, self._types, self._parameters = modules, types, parameters
            self._tensors = [p for p in parameters if p is not None]
            self._sources = Sources(self._tensors)
            self._constants = [(m.__dict__, n) for m in modules for n in self.CONSTANTS if n in m.__dict__]
            self._values = [d[n] for d, n in self._constants]
        return self.generation
