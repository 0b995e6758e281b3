"""The segmented scans of large grids against the lane-state scans of small ones.

Grids of more than 8192 scan wavefronts run each row in segments of 2048 sample
blocks (the state carried from block to block); the same rows alone in a small
batch keep lane states.  Both evaluate the same recursions in float64 and
round once to float32, so the filtered signals agree to a unit in the last
place of the row's peak (6e-8; 2e-7 allowed) and the gradients, whose filters
spread those units, to 1e-6 of their peak.  Lengths at the edges: one sample
around segment blocks, aggregate blocks and the 15 sample ramps, odd rows
(misaligned), rows of a single segment (no aggregate and prefix launches) and
of one more than that.  The backward's scans run as many rows as there are
gradient rows, so its segments at these lengths are those of both gradients.
"""

import pytest
import torch

from torch_pesq import PesqLoss, _lib
from torch_pesq.hip_ops.pipeline import pipeline_backward, pipeline_forward, pipeline_region

pytestmark = pytest.mark.gpu


def _run(model, ref, deg, mask=_lib.GRAD_DEG):
    batch, n = ref.shape
    both = mask == _lib.GRAD_REF | _lib.GRAD_DEG
    out, ws = pipeline_forward(ref, deg, model.model_table, 0.5, mask)
    ones = torch.ones(batch, device="cuda")
    g_ref, g_deg = pipeline_backward([None, None, None, ones], ws, model.model_table, batch, n,
                                     0.5, mask)

    def region(name, rows):
        off, _ = pipeline_region(batch, n, mask, name)
        return ws[off:off + rows * n * 4].view(torch.float32).view(rows, n)

    grad = torch.cat([g_ref, g_deg]) if both else g_deg
    return out[3], region("p", 2 * batch), region("f", grad.shape[0]), grad


@pytest.mark.parametrize("batch, n", [
    (700, 6143), (700, 6144), (700, 6145), (700, 6159), (640, 8191), (640, 8193),
    (600, 7168), (600, 7183), (2100, 5401), (37, 116961), (130, 40961), (10, 960001),
])
def test_segmented_scans_match_the_small_grid_scans(batch, n):
    model = PesqLoss(0.5, sample_rate=16000).cuda()
    assert 2 * batch * -(-n // 1024) > 8192
    gen = torch.Generator(device="cuda").manual_seed(n)
    ref = torch.randn(batch, n, generator=gen, device="cuda") * 0.05
    deg = ref + 0.02 * torch.randn(batch, n, generator=gen, device="cuda")
    loss, p, f, grad = _run(model, ref, deg)
    for first in (0, batch // 2, batch - 3):
        item = slice(first, first + 3)
        loss1, p1, f1, grad1 = _run(model, ref[item].contiguous(), deg[item].contiguous())
        p_big = torch.cat([p[item], p[batch + first:batch + first + 3]])
        for got, want, bound in ((p_big, p1, 2e-7), (f[item], f1, 2e-7), (grad[item], grad1, 1e-6)):
            peak = want.abs().amax(1, keepdim=True)
            assert float(((got - want).abs() / peak).max()) < bound
        assert float(((loss[item] - loss1).abs() / loss1).max()) < 1e-6


@pytest.mark.parametrize("batch, n", [
    (700, 6143), (700, 6144), (700, 6145), (700, 6159), (640, 8191), (640, 8193),
    (600, 7168), (600, 7183), (700, 6151), (37, 116961), (130, 40961), (5, 960001),
])
def test_segmented_backward_scans_match_the_small_grid_scans(batch, n):
    """Both gradients: the reversed segments run over 2 batch rows, whose ends lie
    at the row's first samples."""

    both = _lib.GRAD_REF | _lib.GRAD_DEG
    assert 2 * batch * -(-n // 1024) > 8192
    names = _lib.pipeline_kernels(batch, n, both, backward=True)
    assert "iir_output_kernel<5, 1, PipeBwdMode, false, 0, false>" in names
    assert not any("PipeBwdMode, true" in k for k in names)
    model = PesqLoss(0.5, sample_rate=16000).cuda()
    gen = torch.Generator(device="cuda").manual_seed(n + 1)
    ref = torch.randn(batch, n, generator=gen, device="cuda") * 0.05
    deg = ref + 0.02 * torch.randn(batch, n, generator=gen, device="cuda")
    loss, p, f, grad = _run(model, ref, deg, both)
    for first in (0, batch // 2, batch - 3):
        item = slice(first, first + 3)
        loss1, p1, f1, grad1 = _run(model, ref[item].contiguous(), deg[item].contiguous(), both)
        for big, want, bound in ((p, p1, 2e-7), (f, f1, 2e-7), (grad, grad1, 1e-6)):
            got = torch.cat([big[item], big[batch + first:batch + first + 3]])
            peak = want.abs().amax(1, keepdim=True)
            assert float(((got - want).abs() / peak).max()) < bound
        assert float(((loss[item] - loss1).abs() / loss1).max()) < 1e-6


def test_rows_of_one_segment_launch_no_aggregate_pass():
    names = _lib.pipeline_kernels(2100, 5401, _lib.GRAD_DEG, backward=False)
    assert not any("aggregate" in k or "prefix" in k for k in names)
    assert "iir_output_kernel<5, 1, PipeFwdMode, false, 0, false>" in names
