"""GPU: a slice's result does not depend on the slices that share its call, bit for bit: each slice of a
batch equals its own call, over the group sizes and their paddings, remainders and launches."""
import numpy as np
import pytest
import torch

from fanbeamctrecon_tensorflowop_amd import workloads
from fanbeamctrecon_tensorflowop_amd.plan import FanBeamPlan

pytestmark = pytest.mark.gpu


def _plan(side, views, cols, ny=None):
    half = np.arcsin(0.5 * side / (2.3 * side)) * 1.1
    p, a = workloads.scan(nx=side, ny=ny, rfov=0.5 * side, sid=2.3 * side, sdd=4.0 * side, n_cols=cols,
                          dcol_rad=2.0 * half / cols, n_views=views)
    return FanBeamPlan(p, a)


@pytest.mark.parametrize("storage", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("side,views,cols,slices", [
    (33, 40, 50, 2), (50, 31, 70, 7), (64, 90, 96, 21), (120, 50, 190, 9), (211, 70, 300, 17), (211, 64, 310, 27)])
def test_fp_adjoint(side, views, cols, slices, storage):
    plan = _plan(side, views, cols)
    y = torch.randn((slices,) + plan.sino_shape, generator=torch.Generator().manual_seed(side)).to(storage).cuda()
    for n in sorted({2, 3, 5, slices}):
        got = plan.fp_adjoint(y[:n])
        for s in range(min(n, slices)):
            assert torch.equal(got[s], plan.fp_adjoint(y[s:s + 1])[0]), (n, s)


# images of fewer rows than columns: per-pixel gathers, in groups of 1, 2, 4, 8 and 16 slices
@pytest.mark.parametrize("side,ny,views,cols,slices", [
    (60, 47, 30, 80, 3), (260, 200, 21, 300, 10), (400, 300, 18, 350, 12), (512, 400, 9, 300, 11), (512, 400, 9, 300, 18)])
def test_fp_adjoint_gather(side, ny, views, cols, slices):
    plan = _plan(side, views, cols, ny=ny)
    y = torch.randn((slices,) + plan.sino_shape, generator=torch.Generator().manual_seed(side)).cuda()
    got = plan.fp_adjoint(y)
    for s in sorted({0, slices // 2, slices - 1}):
        assert torch.equal(got[s], plan.fp_adjoint(y[s:s + 1])[0]), s
