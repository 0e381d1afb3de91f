"""The prepared copies of a module's parameters follow the parameters (CPU)."""

import copy

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
