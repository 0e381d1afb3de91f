"""fp32 products on split operands where magnitudes are unlike: weight rows, normalised rows.

Bound: TOL of test_split_gpu.py against float64, for each output channel or row by itself, because each weight row and
each row has its own scale.
"""

import pytest
import torch

from bioemu2_amd import _ops
from bioemu2_amd.attention_pair_bias import AttentionPairBias
from bioemu2_amd.glue import PairwiseConditioning
from bioemu2_amd.transition import Transition
from bioemu2_amd.triangle_multiplication import TriangleMultiplicationHip
from tests._helpers import randomize_params
from tests.test_split_gpu import TOL, _apb64, _ln, _params, _transition

pytestmark = pytest.mark.gpu


def _unlike(weight):
    """Rows of 1, 1e-1 .. 1e-9 of their magnitude, in turn."""
    with torch.no_grad():
        weight.mul_(torch.logspace(0, -9, 10).repeat(-(-weight.shape[0] // 10))[: weight.shape[0], None])


def _worst_channel(got, want):
    """The largest relative error (2-norm) of an output channel."""
    got, want = got.double().cpu().flatten(0, -2), want.flatten(0, -2)
    return float(((got - want).norm(dim=0) / want.norm(dim=0)).max())


@pytest.mark.parametrize("dim,rows", [(128, 200), (128, 18500), (64, 12300), (384, 70), (384, 4300)])
def test_output_rows_of_a_transition(gpu_device, dim, rows):
    torch.manual_seed(0)
    m = randomize_params(Transition(dim, 2 * dim), 3)
    _unlike(m.fc3.weight)
    x = torch.randn(rows, dim)
    want = _transition(x.double(), _params(m))
    with torch.no_grad():
        got = m.to(gpu_device)(x.to(gpu_device))
    assert _worst_channel(got, want) <= TOL


@pytest.mark.parametrize("c_s,heads,n", [(128, 4, 40), (384, 16, 40), (384, 16, 1500)])
def test_output_rows_of_an_attention(gpu_device, c_s, heads, n):
    torch.manual_seed(1)
    m = randomize_params(AttentionPairBias(c_s, 16, heads, initial_norm=False), 4)
    _unlike(m.proj_o.weight)
    s, z = torch.randn(1, n, c_s), torch.randn(1, n, n, 16)
    mask = torch.ones(1, n, dtype=torch.bool)
    want = _apb64(s.double(), z.double(), mask, _params(m), heads, 1, False)
    with torch.no_grad():
        got = m.to(gpu_device)(s.to(gpu_device), z.to(gpu_device), mask.to(gpu_device))
    assert _worst_channel(got, want) <= TOL


@pytest.mark.parametrize("rows", [500, 17000])
def test_output_rows_of_the_conditioning_projection(gpu_device, rows):
    torch.manual_seed(2)
    m = randomize_params(PairwiseConditioning(128, 128), 5)
    _unlike(m.dim_pairwise_init_proj[1].weight)
    z, rel = torch.randn(rows, 128), torch.randn(rows, 128)
    p = _params(m)
    want = _ln(torch.cat([z, rel], -1).double(), p, "dim_pairwise_init_proj.0") @ p["dim_pairwise_init_proj.1.weight"].T
    m = m.to(gpu_device)
    got = _ops.launch_pair_cond_proj_f32(z.to(gpu_device), rel.to(gpu_device), *m.prepared_params_f32(),
                                         torch.empty(rows, 128, device=gpu_device))
    assert _worst_channel(got, want) <= TOL


@pytest.mark.parametrize("n", [33, 130])
def test_output_rows_of_a_triangle_multiplication(gpu_device, n):
    torch.manual_seed(3)
    m = randomize_params(TriangleMultiplicationHip(128, "outgoing"), 6)
    _unlike(m.p_out.weight)
    p = _params(m)
    x = torch.randn(1, n, n, 128)
    xn = _ln(x.double(), p, "norm_in")
    a, b = ((xn @ p["p_in.weight"].T) * torch.sigmoid(xn @ p["g_in.weight"].T)).permute(0, 3, 1, 2).chunk(2, 1)
    o = (a @ b.transpose(2, 3)).permute(0, 2, 3, 1)
    want = (_ln(o, p, "norm_out") @ p["p_out.weight"].T) * torch.sigmoid(xn @ p["g_out.weight"].T)
    mask = torch.ones(1, n, n, dtype=torch.bool)
    with torch.no_grad():
        got = m.to(gpu_device)(x.to(gpu_device), mask.to(gpu_device))
    assert _worst_channel(got, want) <= TOL


def _worst_row(got, want):
    """The largest relative error (2-norm) of a row."""
    got, want = got.double().cpu().flatten(0, -2), want.flatten(0, -2)
    return float(((got - want).norm(dim=1) / want.norm(dim=1)).max())


def _zero_biases(module):
    with torch.no_grad():
        for name, p in module.named_parameters():
            if p.ndim == 1 and name.endswith("bias"):
                p.zero_()


@pytest.mark.parametrize("rows", [500, 17000])
def test_rows_of_little_deviation_in_the_conditioning_projection(gpu_device, rows):
    """Deviations from 1 to 1e-12 next to each other: normalised rows far below the LayerNorm's epsilon."""
    torch.manual_seed(4)
    m = randomize_params(PairwiseConditioning(128, 128), 7)
    _zero_biases(m)
    dev = torch.logspace(0, -12, 13).repeat(-(-rows // 13))[:rows, None]
    z, rel = torch.randn(rows, 128) * dev, torch.randn(rows, 128) * dev
    p = _params(m)
    want = _ln(torch.cat([z, rel], -1).double(), p, "dim_pairwise_init_proj.0") @ p["dim_pairwise_init_proj.1.weight"].T
    m = m.to(gpu_device)
    got = _ops.launch_pair_cond_proj_f32(z.to(gpu_device), rel.to(gpu_device), *m.prepared_params_f32(),
                                         torch.empty(rows, 128, device=gpu_device))
    assert _worst_row(got, want) <= TOL


@pytest.mark.parametrize("dev", [1e-3, 1e-5, 1e-7, 1e-9, 1e-12])
def test_rows_of_little_deviation_in_an_attention(gpu_device, dev):
    torch.manual_seed(5)
    m = randomize_params(AttentionPairBias(128, 16, 4), 8)
    _zero_biases(m)
    s, z = torch.randn(1, 40, 128) * dev, torch.randn(1, 40, 40, 16)
    mask = torch.ones(1, 40, dtype=torch.bool)
    want = _apb64(s.double(), z.double(), mask, _params(m), 4, 1, True)
    with torch.no_grad():
        got = m.to(gpu_device)(s.to(gpu_device), z.to(gpu_device), mask.to(gpu_device))
    assert _worst_row(got, want) <= TOL


@pytest.mark.parametrize("n", [33, 130])
@pytest.mark.parametrize("small", [1e-2, 1e-4, 1e-6])
def test_rows_of_little_deviation_in_a_triangle_multiplication(gpu_device, n, small):
    """Input projections so small that the contraction's rows lie far below the output LayerNorm's epsilon."""
    torch.manual_seed(6)
    m = randomize_params(TriangleMultiplicationHip(128, "outgoing"), 9)
    _zero_biases(m)
    with torch.no_grad():
        m.p_in.weight.mul_(small)
    p = _params(m)
    x = torch.randn(1, n, n, 128)
    xn = _ln(x.double(), p, "norm_in")
    a, b = ((xn @ p["p_in.weight"].T) * torch.sigmoid(xn @ p["g_in.weight"].T)).permute(0, 3, 1, 2).chunk(2, 1)
    o = (a @ b.transpose(2, 3)).permute(0, 2, 3, 1)
    want = (_ln(o, p, "norm_out") @ p["p_out.weight"].T) * torch.sigmoid(xn @ p["g_out.weight"].T)
    mask = torch.ones(1, n, n, dtype=torch.bool)
    with torch.no_grad():
        got = m.to(gpu_device)(x.to(gpu_device), mask.to(gpu_device))
    assert _worst_row(got, want) <= TOL


# rows of each form of the transition: separate products (32 x 64 tiles, 128 x 128 tiles), one kernel
TRANSITIONS = [(128, 200), (128, 18500), (64, 12300), (384, 70), (384, 4300)]


@pytest.mark.parametrize("dim,rows", TRANSITIONS)
@pytest.mark.parametrize("factor", [256.0, 4096.0])
def test_hidden_outliers(gpu_device, dim, rows, factor):
    """One fc1 row and another fc2 row large, their fc3 columns small in turn: the product of the largest norms says
    nothing about any hidden value."""
    torch.manual_seed(7)
    m = randomize_params(Transition(dim, 2 * dim), 10)
    with torch.no_grad():
        for w, unit in ((m.fc1.weight, 3), (m.fc2.weight, 37)):
            w[unit] *= factor
            m.fc3.weight[:, unit] /= factor
    x = torch.randn(rows, dim)
    want = _transition(x.double(), _params(m))
    with torch.no_grad():
        got = m.to(gpu_device)(x.to(gpu_device))
    assert _worst_row(got, want) <= TOL


@pytest.mark.parametrize("dim,rows", TRANSITIONS)
def test_gamma_outlier(gpu_device, dim, rows):
    """A LayerNorm weight of 1024 on a channel that is near its row's mean."""
    torch.manual_seed(8)
    m = randomize_params(Transition(dim, 2 * dim), 11)
    with torch.no_grad():
        m.norm.weight[5] = 1024.0
    x = torch.randn(rows, dim)
    x[:, 5] = 0.0
    x -= x.mean(1, keepdim=True)
    x[:, 5] = 0.0
    want = _transition(x.double(), _params(m))
    with torch.no_grad():
        got = m.to(gpu_device)(x.to(gpu_device))
    assert _worst_row(got, want) <= 2.5 * TOL   # the mean is rounded, 1024 times: 7.4e-6 with fp32 operands


@pytest.mark.parametrize("dim,rows", TRANSITIONS)
def test_closed_gates_and_small_rows(gpu_device, dim, rows):
    """Hidden values far below what the weights' norms allow: gates near -25, and rows of deviation down to 1e-12."""
    torch.manual_seed(9)
    m = randomize_params(Transition(dim, 2 * dim), 12)
    _zero_biases(m)
    x = torch.randn(rows, dim) * torch.logspace(0, -12, 13).repeat(-(-rows // 13))[:rows, None]
    want = _transition(x.double(), _params(m))
    d = m.to(gpu_device)
    with torch.no_grad():
        assert _worst_row(d(x.to(gpu_device)), want) <= TOL
        x = torch.randn(rows, dim)
        x[:, 0] = 30.0
        d.fc1.weight.mul_(0.02)
        d.fc1.weight[:, 0] = -25.0 * (1.0 + 900.0 / dim) ** 0.5 / 30.0   # the channel, normalised, times this: -25
        want = _transition(x.double(), _params(d))
        assert float((want.norm(dim=1) / _transition(-x.double(), _params(d)).norm(dim=1)).max()) < 1e-6
        assert _worst_row(d(x.to(gpu_device)), want) <= 4 * TOL   # the argument is rounded, 25 times: 1.3e-5 with fp32 operands


@pytest.mark.parametrize("dim,rows", TRANSITIONS)
def test_hidden_overflow(gpu_device, dim, rows):
    """Infinite hidden values give infinite outputs of the weights' signs."""
    torch.manual_seed(10)
    m = randomize_params(Transition(dim, 2 * dim, use_norm=False), 13)
    with torch.no_grad():
        m.fc1.weight[3] = m.fc2.weight[3] = 0.0
        m.fc1.weight[3, 0] = m.fc2.weight[3, 0] = 1e20
    x = torch.randn(rows, dim)
    x[:, 0] = 1.0
    x[7, 0] = 0.0
    with torch.no_grad():
        got = m.to(gpu_device)(x.to(gpu_device)).cpu()
    assert torch.isfinite(got[7]).all()
    got[7] = got[8]
    assert torch.equal(got, (float("inf") * torch.sign(m.fc3.weight[:, 3].cpu())).expand_as(got))


@pytest.mark.parametrize("c_s,heads", [(384, 16), (128, 4)])
@pytest.mark.parametrize("n,masked", [(40, range(5, 9)), (97, range(60, 97)), (200, range(0, 199))])
def test_valid_keys_below_the_masked_ones(gpu_device, c_s, heads, n, masked):
    """Queries whose valid keys' logits are near -5e6 attend to the masked keys, whose logit is -1e6; the others next to
    them do not."""
    torch.manual_seed(11)
    m = randomize_params(AttentionPairBias(c_s, 16, heads, initial_norm=False), 14)
    d = c_s // heads
    low = 5e6 / (d / d**0.5)
    with torch.no_grad():
        m.proj_q_bias.zero_()
        m.proj_qkv.weight[: 2 * c_s] = 0.0
        m.proj_qkv.weight[:c_s, 0] = low**0.5
        m.proj_qkv.weight[c_s : 2 * c_s, 1] = -(low**0.5)
    s, z = torch.randn(1, n, c_s), torch.randn(1, n, n, 16)
    s[..., 0] = (torch.arange(n) % 3 == 0).float()
    s[..., 1] = 1.0
    mask = torch.ones(1, n, dtype=torch.bool)
    mask[:, list(masked)] = False
    want = _apb64(s.double(), z.double(), mask, _params(m), heads, 1, False)
    with torch.no_grad():
        got = m.to(gpu_device)(s.to(gpu_device), z.to(gpu_device), mask.to(gpu_device))
    assert _worst_row(got, want) <= TOL


def _trimul64(x, p, mode):
    xn = _ln(x.double(), p, "norm_in")
    a, b = ((xn @ p["p_in.weight"].T) * torch.sigmoid(xn @ p["g_in.weight"].T)).permute(0, 3, 1, 2).chunk(2, 1)
    o = (a @ b.transpose(2, 3) if mode == "outgoing" else a.transpose(2, 3) @ b).permute(0, 2, 3, 1)
    return (_ln(o, p, "norm_out") @ p["p_out.weight"].T) * torch.sigmoid(xn @ p["g_out.weight"].T)


@pytest.mark.parametrize("mode", ["outgoing", "incoming"])
@pytest.mark.parametrize("n", [33, 130])
def test_triangle_planes_far_below_their_bound(gpu_device, mode, n):
    """Rows of deviation down to 1e-9, and input gates near -25: the planes' values lie far below what the weights'
    norms allow, in all lines and in some."""
    torch.manual_seed(12)
    m = randomize_params(TriangleMultiplicationHip(128, mode), 15)
    _zero_biases(m)
    mask = torch.ones(1, n, n, dtype=torch.bool, device=gpu_device)
    d = m.to(gpu_device)
    line = torch.randn(1, n, n, 128)
    for dev in (1e-5, 1e-7, 1e-9):
        for x in (line * dev, line * torch.where(torch.arange(n) % 5 == 0, 1.0, dev)[:, None, None],
                  line * torch.where(torch.arange(n) % 5 == 0, 1.0, dev)[:, None]):
            with torch.no_grad():
                assert _worst_row(d(x.to(gpu_device), mask), _trimul64(x, _params(d), mode)) <= TOL
    x = line.clone()
    x[..., 0] = 30.0
    with torch.no_grad():
        d.g_in.weight.mul_(0.02)
        d.g_in.weight[:, 0] = -25.0 * (1.0 + 900.0 / 128) ** 0.5 / 30.0
        assert _worst_row(d(x.to(gpu_device), mask), _trimul64(x, _params(d), mode)) <= 8 * TOL   # two gates' arguments
        d.g_in.weight[::2, 0] = 0.0   # every other channel open
        assert _worst_row(d(x.to(gpu_device), mask), _trimul64(x, _params(d), mode)) <= TOL
