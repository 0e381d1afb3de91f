"""Device-ready copies of module parameters, cached until a parameter changes."""

from __future__ import annotations

import torch
import torch.nn as nn
from torch import Tensor


def _find(module: nn.Module, path: tuple[str, ...]) -> nn.Parameter:
    """``module.get_parameter``, through the modules' own tables (a few lookups instead of attribute protocols)."""
    owner = module
    for name in path[:-1]:
        owner = owner._modules.get(name)
        if owner is None:
            break
    else:
        p = owner._parameters.get(path[-1])
        if isinstance(p, nn.Parameter):
            return p
    return module.get_parameter(".".join(path))   # anything unusual: its answer, or its error


class PreparedParams:
    """Caches ``(param.detach().to(dtype).contiguous(), ...)`` for a module.

    The cache key is the identity and (data_ptr, version counter, device,
    dtype) of every source parameter, so in-place updates (optimizer steps,
    ``load_state_dict``), ``.to()`` moves and replaced parameters invalidate it.
    The sources stay referenced: a new parameter cannot take the identity of
    one that was freed, as it can take its address.
    """

    def __init__(self, spec: list[tuple[str, torch.dtype]]):
        self.spec = spec
        self._paths = [tuple(name.split(".")) for name, _ in spec]
        self._key: tuple | None = None
        self._src: list[nn.Parameter] | None = None
        self._val: tuple[Tensor, ...] | None = None

    def __getstate__(self) -> dict:
        return {"spec": self.spec}   # a copy or a saved module has parameters of its own, and prepares them itself

    def __setstate__(self, state: dict) -> None:
        PreparedParams.__init__(self, state["spec"])

    def get(self, module: nn.Module) -> tuple[Tensor, ...]:
        params = [_find(module, path) for path in self._paths]
        key = tuple((id(p), p.data_ptr(), p._version, p.device, p.dtype) for p in params)
        if key != self._key or self._val is None:
            self._val = tuple(
                p.detach().to(dtype=dt).contiguous() for p, (_, dt) in zip(params, self.spec)
            )
            self._key, self._src = key, params
        return self._val
