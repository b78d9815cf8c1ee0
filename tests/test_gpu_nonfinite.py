"""GPU: an infinity or NaN in a sinogram reaches only the pixels that its ray's samples touch in FP^T,
in every slice group, from either side of the LDS window, in a uniform and an uneven batch.

The pixels a ray touches are those where the FP64 oracle's adjoint of that ray alone is not 0.  A
sample within an FP32 rounding (3e-4 of a pixel) of a cell's boundary may be credited to the next
cell: about 1e-3 of the cells a ray passes, so 1% more pixels are let through, and one a ray.
"""
import numpy as np
import pytest
import torch

from fanbeamctrecon_tensorflowop_amd import workloads
from fanbeamctrecon_tensorflowop_amd.batch import UnevenBatch
from fanbeamctrecon_tensorflowop_amd.plan import FanBeamPlan

pytestmark = pytest.mark.gpu

SIDE = 64


def _case(cols, views, oracle_mod):
    sid = 2.5 * SIDE
    half = np.arcsin(0.5 * SIDE / sid) * 1.1
    p, a = workloads.scan(nx=SIDE, rfov=0.5 * SIDE, sid=sid, sdd=2 * sid, n_cols=cols, dcol_rad=2 * half / cols,
                          n_views=views)
    rays = [(0, cols // 2), (1, 3), (views // 3, cols // 3), (views // 2, cols // 2 + 5), (views - 1, 2 * cols // 3)]
    one = np.zeros((1, views, cols), dtype=np.float32)
    for r in rays:
        one[(0,) + r] = 1.0
    return FanBeamPlan(p, a), rays, oracle_mod.Oracle(p, a).fp_adjoint(one)[0]


def _check(got, clean, touched, rays):
    bad = ~np.isfinite(got)
    extra = int((bad & (touched == 0)).sum())
    print("%d touched, %d not finite, %d extra" % ((touched > 0).sum(), bad.sum(), extra), flush=True)
    assert bad[touched > 1e-3 * touched.max()].all()
    assert extra <= 0.01 * (touched > 0).sum() + len(rays)
    assert np.array_equal(got[~bad], clean[~bad])


@pytest.mark.parametrize("slices", [1, 2, 4, 8, 16])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
@pytest.mark.parametrize("cols,views", [(40, 90), (96, 90), (2000, 12)])  # the last: windows wider than the slots
def test_footprint(slices, value, cols, views, oracle_mod):
    plan, rays, touched = _case(cols, views, oracle_mod)
    x = torch.randn((slices,) + plan.sino_shape, device="cuda")
    for r in rays:
        x[(slices - 1,) + r] = 0.0
    clean = plan.fp_adjoint(x).cpu().numpy()
    for dtype in (torch.float32, torch.bfloat16):
        if dtype != torch.float32:
            x = x.to(dtype)
            clean = plan.fp_adjoint(x).cpu().numpy()
        y = x.clone()
        for r in rays:
            y[(slices - 1,) + r] = value
        got = plan.fp_adjoint(y).cpu().numpy()
        assert np.array_equal(got[:-1], clean[:-1])
        _check(got[-1], clean[-1], touched, rays)


def test_uneven(oracle_mod):
    cases = [_case(c, 90, oracle_mod) for c in (96, 200)]
    batch = UnevenBatch([c[0] for c in cases])
    sinos = [torch.randn(c[0].sino_shape, device="cuda") for c in cases]
    for r in cases[1][1]:
        sinos[1][r] = 0.0
    clean = batch.fp_adjoint(torch.cat([s.reshape(-1) for s in sinos])).cpu().numpy()
    for r in cases[1][1]:
        sinos[1][r] = float("nan")
    got = batch.fp_adjoint(torch.cat([s.reshape(-1) for s in sinos])).cpu().numpy()
    n = SIDE * SIDE
    assert np.array_equal(got[:n], clean[:n])
    _check(got[n:].reshape(SIDE, SIDE), clean[n:].reshape(SIDE, SIDE), cases[1][2], cases[1][1])
