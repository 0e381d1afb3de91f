"""The prepared copies of a module's parameters follow the parameters (CPU)."""

import copy

import numpy as np
import pytest
import torch
from torch.func import functional_call

from bioemu2_amd.transition import Transition


class _Prepared(Transition):
    def forward(self):
        return self.prepared_params()


def _weights(module, value, kind):
    return {name: kind(torch.full_like(p, value).detach()) for name, p in module.named_parameters()}


@pytest.mark.parametrize("grad", [False, True])
def test_plain_tensors_in_a_parameters_place_are_refused(grad):
    m = _Prepared(128, 256)
    m()
    with torch.set_grad_enabled(grad), pytest.raises(AttributeError):
        functional_call(m, _weights(m, 1.0, lambda t: t), ())


def test_replaced_and_freed_parameters_are_seen():
    """A new parameter at a freed one's address (here for certain: both over one array) has the same address, version,
    device and dtype."""
    m = _Prepared(128, 256)
    memory = {name: np.zeros(p.shape, dtype=np.float32) for name, p in m.named_parameters()}
    for value in range(1, 5):
        params = {}
        for name, a in memory.items():
            a.fill(value)
            params[name] = torch.nn.Parameter(torch.from_numpy(a))
        assert all(bool((t == value).all()) for t in functional_call(m, params, ()))
    for value in range(1, 5):
        memory["fc2.weight"].fill(value)
        m.fc2.weight = torch.nn.Parameter(torch.from_numpy(memory["fc2.weight"]))
        assert bool((m()[3] == value).all())


def test_copies_and_updates_are_seen():
    m = _Prepared(128, 256)
    first = m()
    assert all(a is b for a, b in zip(first, m()))
    other = copy.deepcopy(m)
    with torch.no_grad():
        other.fc1.weight.fill_(3.0)
    assert bool((other()[2] == 3.0).all()) and m()[2] is first[2]
    m.load_state_dict(other.state_dict())
    assert bool((m()[2] == 3.0).all())
