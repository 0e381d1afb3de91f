"""fp32 row kernels on few rows and on many: which form runs, both sides of each rule's line, and what both give.

Bound: TOL of test_split_gpu.py (float64 reference).
"""

import pytest
import torch
import torch.nn.functional as F

from bioemu2_amd import _ops
from bioemu2_amd.attention_pair_bias import AttentionPairBiasSlidingWindow
from bioemu2_amd.glue import PairwiseConditioning
from bioemu2_amd.timing import KernelTimer
from bioemu2_amd.transition import Transition
from bioemu2_amd.triangle_multiplication import TriangleMultiplicationHip
from tests._helpers import randomize_params, rel_l2
from tests.test_split_gpu import TOL, _params, _transition

pytestmark = pytest.mark.gpu


def _run(module, *args, **kwargs):
    """The module's output and the names of the kernels that made it."""
    with torch.no_grad(), KernelTimer() as t:
        out = module(*args, **kwargs)
    return out, set(t.results())


@pytest.mark.parametrize(
    "dim,hidden,use_norm,rows",
    [
        (128, 256, True, 200),
        (128, 256, True, 18431),      # the last row count of the separate products
        (128, 256, True, 18432),      # one kernel: 72 whole workgroups
        (128, 32, True, 18433),       # ... one row more, one hidden chunk
        (128, 512, False, 18687),     # ... a workgroup less one row
        (128, 2048, True, 18500),     # ... its widest hidden dimension
        (64, 128, False, 12287),
        (64, 128, False, 12289),
        (64, 256, True, 12543),
    ],
)
def test_transition_forms(gpu_device, dim, hidden, use_norm, rows):
    torch.manual_seed(0)
    m = randomize_params(Transition(dim, hidden, use_norm=use_norm), 3)
    x = torch.randn(rows, dim)
    want = _transition(x.double(), _params(m), use_norm)
    got, names = _run(m.to(gpu_device), x.to(gpu_device))
    assert rel_l2(got.cpu(), want) <= TOL
    assert ("f32_transition_rows" in names) == (rows >= (18432 if dim == 128 else 12288))


def test_fused_transition_ranges(gpu_device):
    """Row magnitudes from 1e-12 to 1e12 in one call, checked row by row; other rows' values leave a row's bits alone."""
    torch.manual_seed(1)
    rows = 18500
    m = randomize_params(Transition(128, 256, use_norm=False), 3)
    x = torch.randn(rows, 128) * torch.logspace(-12, 12, rows)[:, None]
    x[5] = 0.0
    want = _transition(x.double(), _params(m), False)
    got, names = _run(m.to(gpu_device), x.to(gpu_device))
    assert "f32_transition_rows" in names and torch.equal(got[5].cpu(), torch.zeros(128))
    err = (got.cpu().double() - want).norm(dim=1) / want.norm(dim=1).clamp_min(1e-300)
    err[5] = 0.0
    assert float(err.max()) <= TOL
    y = x.clone()
    y[9000:] = torch.randn(rows - 9000, 128)
    with torch.no_grad():
        assert torch.equal(m(y.to(gpu_device))[:9000], got[:9000])


@pytest.mark.parametrize("norm", [False, True])
def test_sliding_window_copies_do_not_depend_on_their_number(gpu_device, norm):
    """The projections deal their 16 (and 4) column blocks to as many workgroups as the rows leave room for: every
    block by itself, three at a time with one left over, all in one."""
    torch.manual_seed(2)
    m = randomize_params(AttentionPairBiasSlidingWindow(128, 16, 4, initial_norm=norm), 4).to(gpu_device).eval()
    nw = 12
    s, z = torch.randn(nw, 32, 128, device=gpu_device), torch.randn(1, nw, 32, 128, 16, device=gpu_device)
    mask = torch.rand(nw, 32, device=gpu_device) < 0.9
    with torch.no_grad():
        alone = m(s, z, mask)
        for copies in (2, 17, 37, 260):
            got = m(s.repeat(copies, 1, 1), z, mask, multiplicity=copies).view(copies, nw, 32, 128)
            assert torch.equal(got, alone.expand_as(got))


def test_pair_conditioning_rows_do_not_depend_on_their_number(gpu_device):
    """A column block a workgroup up to 512 tiles of 32 rows, all four beyond; ragged last tiles of both."""
    torch.manual_seed(3)
    m = randomize_params(PairwiseConditioning(128, 128), 5).to(gpu_device).eval()
    p = m.prepared_params_f32()
    z, rel = torch.randn(16385, 128, device=gpu_device), torch.randn(16385, 128, device=gpu_device)

    def proj(rows):
        out = torch.empty(rows, 128, device=gpu_device)
        return _ops.launch_pair_cond_proj_f32(z[:rows], rel[:rows], *p, out)

    want = proj(16385)
    x = F.layer_norm(torch.cat([z, rel], -1).double(), (256,), p[0].double(), p[1].double(), 1e-5) @ p[2].double().T
    assert rel_l2(want.cpu(), x.cpu()) <= TOL
    for rows in (1, 31, 33, 129, 16384):
        assert torch.equal(proj(rows), want[:rows])


@pytest.mark.parametrize("rows", [70, 17000])
@pytest.mark.parametrize("which", [0, 1])
def test_pair_conditioning_in_place(gpu_device, which, rows):
    """The output over one of the inputs, and over rows shifted by one."""
    torch.manual_seed(4)
    m = randomize_params(PairwiseConditioning(128, 128), 6).to(gpu_device).eval()
    p = m.prepared_params_f32()
    base = [torch.randn(rows + 1, 128, device=gpu_device) for _ in range(2)]
    want = _ops.launch_pair_cond_proj_f32(base[0][:rows], base[1][:rows], *p, torch.empty(rows, 128, device=gpu_device))
    for shift in (0, 1):
        x = [t.clone() for t in base]
        out = x[which][shift : shift + rows]
        _ops.launch_pair_cond_proj_f32(x[0][:rows], x[1][:rows], *p, out)
        assert rel_l2(out.cpu(), want.cpu()) <= TOL


@pytest.mark.parametrize("mode", ["outgoing", "incoming"])
@pytest.mark.parametrize("n,few,many", [(2, 1, 129), (33, 3, 4), (40, 1, 13)])
def test_triangle_multiplication_forms(gpu_device, mode, n, few, many):
    """Line tiles (32 pairs) on both sides of the 256 up to which a workgroup takes one: the same bits, out of place and
    over the input."""
    torch.manual_seed(5)
    m = randomize_params(TriangleMultiplicationHip(128, mode), 7).to(gpu_device).eval()
    p = m.prepared_params_f32()
    x = torch.randn(many, n, n, 128, device=gpu_device)
    mask = (torch.rand(many, n, n, device=gpu_device) < 0.8).to(torch.uint8)

    def run(b, out, residual):
        return _ops.launch_trimul_f32(x[:b] if out is None else out, mask[:b], *p,
                                      torch.empty_like(x[:b]) if out is None else out, mode == "outgoing",
                                      residual=residual)

    for residual in (False, True):
        assert torch.equal(run(few, None, residual), run(many, None, residual)[:few])
    for b in (few, many):
        assert torch.equal(run(b, x[:b].clone(), True), run(b, None, True))


@pytest.mark.parametrize("dim,rows", [(128, 18432), (128, 73729), (64, 49153)])
def test_transition_of_another_width_many_rows(gpu_device, dim, rows):
    """As many rows as the one-kernel form takes, with an output width it does not: the separate products, a part of the
    rows at a time in a workspace that does not grow with them."""
    torch.manual_seed(6)
    m = randomize_params(Transition(dim, 96, out_dim=dim + 32), 8)
    x = torch.randn(rows, dim)
    want = _transition(x.double(), _params(m))
    got, names = _run(m.to(gpu_device), x.to(gpu_device))
    assert rel_l2(got.cpu(), want) <= TOL and "f32_transition_rows" not in names
    need = [_ops.transition_f32_workspace_bytes(r, dim, 96) for r in (200, 12287, 12288, 18432, 73728, 600000)]
    assert need == sorted(need) and need[-1] == need[-2]
