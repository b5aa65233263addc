"""When a fused form may stand for the calls of several modules, and the loops that take it."""
from __future__ import annotations

import torch.nn as nn
from torch.nn.modules import module as _module

_FUSED: set = set()
_GLOBAL_HOOKS = (_module._global_forward_hooks, _module._global_forward_pre_hooks, _module._global_backward_hooks,
                 _module._global_backward_pre_hooks)


def fused(cls):
    """Class decorator: :func:`as_called` may say yes of objects of this class."""
    _FUSED.add(cls)
    return cls


def as_called(*modules) -> bool:
    """Whether a call of each of these modules is its class's ``forward`` and nothing else, so that a fused form may stand for the call: a
    class that is declared :func:`fused` itself (one derived from it may have another ``forward``), no hooks, no ``forward`` of the
    object's."""
    a, b, c, e = _GLOBAL_HOOKS
    if a or b or c or e:
        return False
    for m in modules:
        d = m.__dict__
        if (type(m) not in _FUSED or "forward" in d or d["_forward_hooks"] or d["_forward_pre_hooks"] or d["_backward_hooks"]
                or d["_backward_pre_hooks"]):
            return False
    return True


def then_norm(m: nn.Module, norm: nn.Module, x, *args, residual, **kw):
    """(y, norm(y)) of y = m(x, *args, residual=residual, **kw): in one call where nothing hooks into either."""
    if as_called(m, norm):
        return m.forward_norm(x, *args, residual=residual, norm=norm, **kw)
    y = m(x, *args, residual=residual, **kw)
    return y, norm(y)


def chain(layers, norms, x, *args):
    """(y, norm(y)) of y = x through ``layers``; ``norms``: the one that each layer begins with, and the one behind them all.  A layer's
    last product makes the next layer's norm as well (``forward_next``), unless something hooks into the layer's call."""
    n = None
    for layer, own, following in zip(layers, norms, norms[1:]):
        if as_called(layer):
            n = own(x) if n is None else n
            x, n = layer.forward_next(x, n, *args, next_norm=following)
        else:
            x, n = layer(x, *args), None
    return x, norms[-1](x) if n is None else n
