"""Which calls reach an op's body directly and which go through the dispatcher, and that both give the same result."""

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from bioemu2_amd import _ops
from bioemu2_amd.attention_pair_bias import AttentionPairBias, AttentionPairBiasSlidingWindow
from bioemu2_amd.outer_product_mean import OuterProductMeanHip
from bioemu2_amd.pair_weighted_averaging import PairWeightedAveraging
from bioemu2_amd.transition import Transition
from bioemu2_amd.triangle_attention import TriangleAttentionHip
from bioemu2_amd.triangle_multiplication import TriangleMultiplicationHip
from tests._helpers import randomize_params

pytestmark = pytest.mark.gpu


@pytest.fixture
def counted(monkeypatch):
    """Counts dispatcher calls of the trimul op."""
    calls = []
    op = _ops.trimul.op
    monkeypatch.setattr(_ops.trimul, "op", lambda *a: (calls.append(1), op(*a))[1])
    return calls


def _case(device):
    torch.manual_seed(0)
    m = randomize_params(TriangleMultiplicationHip(128), 1).to(device).eval()
    x = torch.randn(1, 20, 20, 128, device=device).to(torch.bfloat16)
    return m, x, torch.rand(1, 20, 20, device=device) < 0.8


def test_inference_calls_skip_the_dispatcher(gpu_device, counted):
    m, x, mask = _case(gpu_device)
    with torch.no_grad():
        direct = m(x, mask)
    with torch.inference_mode():
        m(x, mask)
    assert not counted
    assert torch.equal(direct, m(x, mask).detach())   # gradients enabled: through the op
    assert len(counted) == 1


class _Seen(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.names.append(str(func))
        return func(*args, **(kwargs or {}))


def test_onlookers_see_the_op(gpu_device, counted):
    m, x, mask = _case(gpu_device)
    with torch.no_grad():
        want = m(x, mask)
        with _Seen() as mode:
            got = m(x, mask)
        assert any("bioemu_mi355x.trimul" in n for n in mode.names) and torch.equal(got, want)

        class Sub(torch.Tensor):
            pass

        m(x.as_subclass(Sub), mask)
        with torch.autograd.forward_ad.dual_level():
            m(x, mask)
    assert len(counted) == 3


def test_profilers_see_the_op(gpu_device, counted):
    m, x, mask = _case(gpu_device)
    with torch.no_grad(), torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as prof:
        m(x, mask)
    assert len(counted) == 1
    assert any("bioemu_mi355x::trimul" in e.key for e in prof.key_averages())


def test_kernels_put_over_the_op_are_called(gpu_device):
    def body(x: torch.Tensor) -> torch.Tensor:
        return x + 1

    op = _ops._Op("test_direct_call_override", body)
    x = torch.zeros(3, device=gpu_device)
    with torch.no_grad():
        assert op(x)[0] == 1
        torch.library.register_kernel("bioemu_mi355x::test_direct_call_override", "cuda", lambda x: x + 2)
        assert op(x)[0] == 2
        op = _ops._Op("test_direct_call_autocast", body)
        torch.library.register_autocast("bioemu_mi355x::test_direct_call_autocast", "cuda", torch.float16)
        with torch.autocast("cuda"):
            assert op(x).dtype == torch.float16


def test_uint8_masks_mean_nonzero(gpu_device):
    m, x, mask = _case(gpu_device)
    with torch.no_grad():
        want = m(x, mask)
        assert torch.equal(m(x, mask.to(torch.uint8) * 255), want)
        assert torch.equal(m(x, mask.to(torch.uint8).transpose(1, 2).contiguous().transpose(1, 2)), want)
        assert torch.equal(m(x, mask.float()), want)


def test_sliding_window_mask_of_any_alignment(gpu_device):
    torch.manual_seed(1)
    m = randomize_params(AttentionPairBiasSlidingWindow(128, 16, 4, initial_norm=False), 2).to(gpu_device).eval()
    nw = 3
    s = torch.randn(nw, 32, 128, device=gpu_device)
    z = torch.randn(1, nw, 32, 128, 16, device=gpu_device)
    mask = torch.rand(nw, 32, device=gpu_device) < 0.9
    shifted = torch.zeros(nw * 32 + 3, dtype=torch.bool, device=gpu_device)[3:].view(nw, 32).copy_(mask)
    with torch.no_grad():
        for dt in (torch.bfloat16, torch.float32):
            assert torch.equal(m(s.to(dt), z.to(dt), mask), m(s.to(dt), z.to(dt), shifted))


def test_replaced_parameters_are_seen(gpu_device):
    m = randomize_params(Transition(128, 256), 3).to(gpu_device).eval()
    x = torch.randn(1, 40, 128, device=gpu_device)
    with torch.no_grad():
        before = m(x)
        m.fc3.weight = torch.nn.Parameter(2.0 * m.fc3.weight)
        assert torch.equal(m(x), 2.0 * before)
        m.norm = torch.nn.LayerNorm(128).to(gpu_device)
        assert not torch.equal(m(x), 2.0 * before)
        del m.fc3.weight
        with pytest.raises(AttributeError):
            m(x)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("kind", ["trimul", "triatt", "apb", "swa", "opm", "pwa"])
def test_any_nonzero_byte_is_valid(gpu_device, kind, dtype):
    """uint8 masks reach every kernel as they are."""
    torch.manual_seed(4)
    n, d = 37, gpu_device
    z, pair = torch.randn(1, n, n, 128).to(dtype), torch.rand(1, n, n) < 0.7
    pair[0, 3] = False
    if kind == "trimul":
        m, args, mask = TriangleMultiplicationHip(128), (z,), pair
    elif kind == "triatt":
        m, args, mask = TriangleAttentionHip(128, 4), (z,), pair
    elif kind == "apb":
        m, args, mask = AttentionPairBias(384, 128, 16), (torch.randn(1, n, 384).to(dtype), z), torch.rand(1, n) < 0.7
    elif kind == "swa":
        m = AttentionPairBiasSlidingWindow(128, 16, 4)
        args = (torch.randn(3, 32, 128).to(dtype), torch.randn(1, 3, 32, 128, 16).to(dtype))
        mask = torch.rand(3, 32) < 0.7
    elif kind == "opm":
        m, args, mask = OuterProductMeanHip(64, 32, 128), (torch.randn(1, 9, n, 64).to(dtype),), torch.rand(1, 9, n) < 0.7
        mask[0, 2] = False
    else:
        m, args, mask = PairWeightedAveraging(64, 128, 32, 8), (torch.randn(1, 9, n, 64).to(dtype), z), pair
    m = randomize_params(m, 5).to(d).eval()
    args = [a.to(d) for a in args]
    values = torch.randint(1, 256, mask.shape, dtype=torch.uint8) * mask.to(torch.uint8)
    with torch.no_grad():
        want = m(*args, mask.to(d))
        assert torch.isfinite(want).all() and torch.equal(m(*args, values.to(d)), want)
