"""The prepared copies of a module's parameters follow the parameters (CPU)."""

import copy
import io
import pickle

import numpy as np
import pytest
import torch
from torch.func import functional_call

from bioemu2_amd._params import PreparedParams
from bioemu2_amd.transition import Transition
from bioemu2_amd.triangle_attention import TriangleAttentionHip


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


class _Saved:
    """Pickles as a prepared-parameter object with the given attributes."""

    def __init__(self, cls, state):
        self.cls, self.state = cls, state

    def __reduce__(self):
        return object.__new__, (self.cls,), self.state


def test_whole_modules_saved_with_other_attributes_load():
    """A module saved in whole brings the attributes that its helper objects had then: the names alone, or a key and
    the prepared copies too."""
    m = _Prepared(128, 256)
    m()
    spec = m._prepared.spec
    for state in ({"spec": spec, "_key": None, "_val": None}, {"spec": spec, "_key": (1,), "_val": m(), "_src": None}):
        m._prepared = pickle.loads(pickle.dumps(_Saved(PreparedParams, state)))
        assert bool((m()[2] == m.fc1.weight.to(m()[2].dtype)).all())


def test_saved_and_copied_modules_prepare_their_own():
    m = TriangleAttentionHip(128, 4)
    first = m.prepared_params()
    buffer = io.BytesIO()
    torch.save(m, buffer)
    buffer.seek(0)
    for other in (torch.load(buffer, weights_only=False), copy.deepcopy(m)):
        with torch.no_grad():
            other.proj_k.weight.fill_(2.0)
        packed = other.prepared_params()[2]
        assert bool((packed[128:256] == 2.0).all()) and torch.equal(packed[:128], first[2][:128])
    assert all(a is b for a, b in zip(first, m.prepared_params()))
    with torch.no_grad():
        m.proj_b.weight.zero_()
    packed = m.prepared_params()[2]
    assert bool((packed[512:] == 0).all()) and torch.equal(packed[:512], first[2][:512])
