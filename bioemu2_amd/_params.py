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
        # (prepared copies, [(parameter, data_ptr, version, device index, dtype)]), replaced as one
        self._cache: tuple[tuple[Tensor, ...], list[tuple]] | None = None

    def __getstate__(self) -> dict:
        return {"spec": self.spec}   # a copy or a saved module has parameters of its own, and prepares them itself

    def __setstate__(self, state: dict) -> None:
        PreparedParams.__init__(self, state["spec"])

    def get(self, module: nn.Module) -> tuple[Tensor, ...]:
        cache = self._cache
        if cache is not None:
            for path, (src, ptr, version, device, dtype) in zip(self._paths, cache[1]):
                p = _find(module, path)
                if (p is not src or p.data_ptr() != ptr or p._version != version or p.dtype != dtype
                        or p.get_device() != device):
                    break
            else:
                return cache[0]
        params = [_find(module, path) for path in self._paths]
        val = self._pack(*(p.detach().to(dtype=dt).contiguous() for p, (_, dt) in zip(params, self.spec)))
        self._cache = val, [(p, p.data_ptr(), p._version, p.get_device(), p.dtype) for p in params]
        return val

    def _pack(self, *prepared: Tensor) -> tuple[Tensor, ...]:
        """What is kept of the copies: themselves, or what a subclass lays out from them."""
        return prepared
