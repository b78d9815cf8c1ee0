"""GPU: the cell-driven FP^T at its edges, against the FP64 oracle.

Slice counts around the group sizes (1, 2, 4, 8, 16 and their padding, as groups of 16 and the rest
and as one launch), images around the 7 x 7
pixel tile, view counts around the quarters, detector windows from a few columns to more than a
wave's 64 slots (fine detectors, and sources close to the image, where the window of a tile near
the source covers the detector), both directions of the columns.

Tolerance on white noise: a sample's FP32 position carries three roundings of a coordinate of
up to `side` texels (start, step times index, sum), 2^-24 side each, which change its bilinear
weights by at most the same on each of two axes: 6 2^-24 side relative, plus 2e-6 for the FP32
sums; BF16 output adds its rounding, 2^-9.
"""
import numpy as np
import pytest
import torch

from conftest import rel_l2
from fanbeamctrecon_tensorflowop_amd import workloads
from fanbeamctrecon_tensorflowop_amd.plan import FanBeamPlan

pytestmark = pytest.mark.gpu


def _scan(side, views, cols, sid, fan, flip=False):
    half = np.arcsin(min(0.5 * side / sid, 0.99)) * fan
    d = (-2.0 if flip else 2.0) * half / cols
    return workloads.scan(nx=side, rfov=0.5 * side, sid=sid, sdd=2.0 * sid, n_cols=cols, dcol_rad=d, n_views=views)


@pytest.mark.parametrize("side,views,cols,sid,fan,slices", [
    (1, 3, 4, 4.0, 1.2, 1), (6, 1, 9, 20.0, 1.2, 2), (7, 2, 11, 20.0, 1.2, 3), (8, 4, 30, 30.0, 1.2, 4),
    (14, 5, 1, 50.0, 1.2, 5), (15, 13, 25, 40.0, 0.8, 8), (29, 17, 64, 80.0, 1.2, 9), (33, 66, 65, 90.0, 1.2, 10),
    (36, 40, 47, 90.0, 1.2, 11), (50, 31, 70, 130.0, 1.2, 17), (41, 64, 90, 100.0, 0.7, 21),
    (32, 20, 200, 80.0, 1.2, 1), (32, 20, 330, 80.0, 1.2, 4),    # 32 and 64 columns a window
    (20, 24, 700, 60.0, 1.2, 1), (20, 24, 500, 60.0, 1.2, 16),   # wider than the slots
    (24, 30, 40, 12.6, 1.0, 1), (24, 30, 400, 12.1, 1.0, 2),     # the source close to the image
    (211, 5, 90, 500.0, 1.2, 17), (211, 4, 91, 500.0, 1.2, 21), (211, 6, 60, 500.0, 1.2, 11),  # groups of 16 and the rest
    (120, 5, 90, 300.0, 1.2, 9), (120, 4, 70, 300.0, 1.2, 41), (90, 4, 70, 300.0, 1.2, 7),     # one padded launch
])
@pytest.mark.parametrize("storage", ["f32", "bf16"])
def test_cells(side, views, cols, sid, fan, slices, storage, oracle_mod):
    p, a = _scan(side, views, cols, sid, fan)
    plan, o = FanBeamPlan(p, a), oracle_mod.Oracle(p, a)
    dt = torch.float32 if storage == "f32" else torch.bfloat16
    y = torch.from_numpy(np.random.default_rng(side).normal(size=(slices,) + plan.sino_shape).astype(np.float32)).to(dt)
    out = plan.fp_adjoint(y.cuda())
    assert torch.equal(plan.fp_adjoint(y.cuda(), out_dtype=dt), out.to(dt))
    got = out.double().cpu().numpy()
    tol = 6 * 2.0 ** -24 * side + 2e-6
    for s in sorted({0, slices // 2, slices - 1}):
        ref = o.fp_adjoint(y[s:s + 1].double().numpy())[0]
        e = rel_l2(got[s], ref)
        print("fp_adjoint %s %d px %d views %d columns sid %g, slice %d of %d: %.2e (%.1e)" % (
            storage, side, views, cols, sid, s, slices, e, tol), flush=True)
        assert e <= tol


def test_reversed_columns(oracle_mod):
    p, a = _scan(30, 33, 51, 80.0, 1.2, flip=True)
    plan, o = FanBeamPlan(p, a), oracle_mod.Oracle(p, a)
    y = np.random.default_rng(2).normal(size=(2,) + plan.sino_shape).astype(np.float32)
    got = plan.fp_adjoint(torch.from_numpy(y).cuda()).double().cpu().numpy()
    assert rel_l2(got, o.fp_adjoint(y)) <= 6 * 2.0 ** -24 * 30 + 2e-6
