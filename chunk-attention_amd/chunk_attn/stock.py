"""Whether the module classes that the layer and the model stand in for are as their files wrote them: adapters,
tracers and profilers replace forwards, what a module call goes through before them, and the functions they compute
with.  What is remembered at import is checked to come from its own file, so that a replacement made before the
import is seen too."""
from __future__ import annotations

import torch
from torch import nn
from torch.nn import functional as F


def _at_home(function, module):
    """The function if `module` is where it was defined, None (which is no class's forward) otherwise."""
    return function if getattr(function, "__globals__", None) is vars(module) else None


_CALL = _at_home(nn.Module.__call__, nn.modules.module)
_CALL_IMPL = _at_home(nn.Module._call_impl, nn.modules.module)
_LINEAR = _at_home(nn.Linear.forward, nn.modules.linear)
_EMBEDDING = _at_home(nn.Embedding.forward, nn.modules.sparse)
_F_LINEAR = torch._C._nn.linear
_F_EMBEDDING = _at_home(F.embedding, F)


def is_stock(cls, forward) -> bool:
    """Calls of the module class run `forward`, the one its file gave it, and nothing else."""
    return cls.forward is forward and cls.__call__ is _CALL and cls._call_impl is _CALL_IMPL


def linear_is_stock() -> bool:
    return F.linear is _F_LINEAR and is_stock(nn.Linear, _LINEAR)


def embedding_is_stock() -> bool:
    return F.embedding is _F_EMBEDDING and is_stock(nn.Embedding, _EMBEDDING)
