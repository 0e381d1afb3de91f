"""LayerNorm biases folded into the projection that follows: W beta is summed with channels c and c + 64 first.

Channels c and c + 64 of some pairs cancel exactly and are 2^20 times the others, so that a sum that meets them in
another order keeps 2^-4 of its bias (the spacing of fp32 there), where this order loses nothing of it.
"""

import pytest
import torch

import oracle
from bioemu2_amd.triangle_attention import TriangleAttentionHip
from bioemu2_amd.triangle_multiplication import TriangleMultiplicationHip
from tests._helpers import randomize_params, rel_l2, state

pytestmark = pytest.mark.gpu
ATOL, RTOL_L2 = 2e-2, 1e-2   # the repository's bf16 bound against the fp32 oracle
BIG = [c for c in range(64) if c % 8 < 2]   # the first two of every eight channels


def _cancelling(beta, *weights):
    """beta large on BIG and BIG + 64, the weights' columns there opposite (and exact in bf16)."""
    lo = torch.tensor(BIG)
    beta[lo] = beta[lo + 64] = 2.0**20
    for w in weights:
        w[:, lo] = 0.25 * torch.sign(w[:, lo])
        w[:, lo + 64] = -w[:, lo]


def _check(got, want):
    got = got.float().cpu()
    assert (got - want).abs().max().item() <= ATOL * max(1.0, want.abs().max().item())
    assert rel_l2(got, want) <= RTOL_L2


def _double(params):
    return {k: v.double() for k, v in params.items()}


@pytest.mark.parametrize("starting", [True, False])
def test_triangle_attention_bias(gpu_device, monkeypatch, starting):
    torch.manual_seed(0)
    m = randomize_params(TriangleAttentionHip(128, 4, starting=starting), 1)
    with torch.no_grad():
        m.norm.weight[[c + o for c in BIG for o in (0, 64)]] = 0.0   # only the biases reach the large channels
        _cancelling(m.norm.bias, m.proj_q.weight, m.proj_k.weight, m.proj_v.weight, m.proj_g.weight, m.proj_b.weight)
    z = torch.randn(1, 37, 37, 128).to(torch.bfloat16)
    mask = torch.rand(1, 37, 37) < 0.8
    monkeypatch.setattr(oracle.pairformer_ref, "_f32", lambda t: t.double())
    want = oracle.triangle_attention(z.double(), mask, _double(state(m)), 4, starting)
    m = m.to(gpu_device).eval()
    with torch.no_grad():
        _check(m(z.to(gpu_device), mask.to(gpu_device)), want)


def test_triangle_multiplication_output_bias(gpu_device, monkeypatch):
    torch.manual_seed(1)
    m = randomize_params(TriangleMultiplicationHip(128, "outgoing"), 2)
    with torch.no_grad():
        both = [c + o for c in BIG for o in (0, 64)]
        for norm in (m.norm_in, m.norm_out):
            norm.weight[both] = 0.0
        for w in (m.p_in.weight, m.g_in.weight):   # the input projections take LN(x) whole
            w[:, both] = 0.0
        _cancelling(m.norm_in.bias, m.g_out.weight)
        _cancelling(m.norm_out.bias, m.p_out.weight)
    x = torch.randn(1, 37, 37, 128).to(torch.bfloat16)
    mask = torch.rand(1, 37, 37) < 0.8
    monkeypatch.setattr(oracle.pairformer_ref, "_f32", lambda t: t.double())
    want = oracle.trimul(x.double(), mask, _double(state(m)), "outgoing")
    m = m.to(gpu_device).eval()
    with torch.no_grad():
        _check(m(x.to(gpu_device), mask.to(gpu_device)), want)
