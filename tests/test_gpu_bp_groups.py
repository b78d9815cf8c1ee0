"""GPU: backprojection and FBP at the edges of their slice groups, view splits and layouts.

The launch picks by slice count and tiles: blocks of 8 x 8 pixels read directly, 1 to 4 slices
at a time and 4, 8 or 16 waves on a block's views, or 16 x 16 tiles staging 8 or 16 slices with
1, 2 or 4 view groups; FBP reads its filtered sinograms interleaved by up to four slices.

Every slice against its own call, 1e-6: the same FP32 updates summed in another order.  A few
slices against the FP64 oracle, on white noise, where the error is the FP32 column
coordinate's: t = x sin - y cos is off by at most 3 roundings of rFOV (its product, its sum and the
stored cosine and sine), that is 3 2^-24 rFOV / (R - rFOV) / dCol columns, and the angle
polynomial and its scale by 2 roundings of half the detector.  An offset of d columns changes a
value interpolated from white noise by sqrt(2) d against an rms of sqrt(2/3); ramp-filtered
noise has lag-one correlation -0.6, so sqrt(3.2) d against sqrt(7/15).
"""
import numpy as np
import pytest
import torch

from conftest import rel_l2
from fanbeamctrecon_tensorflowop_amd import workloads
from fanbeamctrecon_tensorflowop_amd.plan import FanBeamPlan

pytestmark = pytest.mark.gpu

WIDE = dict(sid=100.0, rfov=32.0)


def _scan(side, views, cols, fan, ny=None):
    # fan: detector over FOV fan (below 1 the fan misses FOV pixels: in-range tests and clamps)
    half = np.arcsin(WIDE["rfov"] / WIDE["sid"]) * fan
    return workloads.scan(nx=side, ny=ny, rfov=WIDE["rfov"], sid=WIDE["sid"], sdd=200.0, n_cols=cols,
                          dcol_rad=2.0 * half / cols, n_views=views)


@pytest.mark.parametrize("side,views,cols,fan,slices", [
    (1, 1, 1, 1.2, 1), (7, 3, 2, 1.2, 2), (9, 5, 33, 0.7, 3), (8, 4, 63, 1.2, 4), (65, 17, 64, 0.8, 5),
    (17, 66, 65, 1.2, 7), (400, 9, 500, 1.2, 1), (300, 6, 410, 0.9, 2),    # 4 and 8 waves a block
    (180, 13, 260, 1.2, 11), (180, 13, 260, 0.6, 19), (181, 7, 60, 1.2, 37),  # four view groups
    (180, 6, 250, 1.2, 64), (180, 5, 250, 0.8, 131),                       # two and one
    (257, 5, 300, 1.2, 16), (256, 9, 300, 0.9, 23),
])
def test_groups(side, views, cols, fan, slices, oracle_mod):
    p, a = _scan(side, views, cols, fan)
    plan, o = FanBeamPlan(p, a), oracle_mod.Oracle(p, a)
    y = np.random.default_rng(side + slices).normal(size=(slices,) + plan.sino_shape).astype(np.float32)
    yd = torch.from_numpy(y).cuda()
    g = plan.geom
    col = 3 * 2.0 ** -24 * g["rFOV"] / (g["R"] - g["rFOV"]) / abs(g["dCol"]) + 2 * 2.0 ** -24 * 0.5 * cols
    tol = {"bp": 1e-6 + 3 ** 0.5 * col, "wbp": 1e-6 + 3 ** 0.5 * col, "fbp": 5e-6 + (3.2 * 15 / 7) ** 0.5 * col}
    for name, fn, ref in (("bp", plan.bp, o.bp), ("wbp", plan.fbp_weighted_bp, lambda s: o.bp(s, weighted=True)),
                          ("fbp", plan.fbp, o.fbp)):
        got = fn(yd)
        one = torch.cat([fn(yd[s:s + 1]) for s in range(slices)])
        worst = max(rel_l2(got[s].double().cpu().numpy(), one[s].double().cpu().numpy()) for s in range(slices))
        errs = [rel_l2(got[s].double().cpu().numpy(), ref(y[s:s + 1])[0]) for s in sorted({0, slices // 2, slices - 1})]
        print("%s %dx%d %d views %d columns %d slices: %.2e, per slice %.2e" % (name, side, side, views, cols, slices,
                                                                          max(errs), worst), flush=True)
        assert max(errs) <= tol[name] and worst <= 1e-6


def test_weighted_fbp_layout(oracle_mod):
    # the pre-weights follow the filter's row order: short scan, odd slice count
    half = np.arcsin(WIDE["rfov"] / WIDE["sid"]) * 1.2
    arc = np.pi + 2.1 * half
    p, a = workloads.scan(nx=50, rfov=WIDE["rfov"], sid=WIDE["sid"], sdd=200.0, n_cols=71, dcol_rad=2.0 * half / 71,
                          n_views=90, angular_range=np.degrees(arc))
    a = (np.arange(90) * (arc / 90)).astype(np.float32)
    plan, o = FanBeamPlan(p, a), oracle_mod.Oracle(p, a)
    y = np.random.default_rng(3).normal(size=(7,) + plan.sino_shape).astype(np.float32)
    got = plan.fbp(torch.from_numpy(y).cuda(), short_scan=True).double().cpu().numpy()
    for s in (0, 3, 4, 6):
        # 71 columns: the coordinate bound of test_groups is 1.3e-5 columns, times 2.6
        assert rel_l2(got[s], o.fbp_short_scan(y[s:s + 1])[0]) <= 4e-5
