"""GPU: rounding of one hat weight of BP^T and FBP^T, against the FP64 oracle.

Images of one pixel each make a sinogram value one weight (or none), 16 columns to a pixel make that
weight 16 times as sensitive to where the ray crosses the pixel's line as to the pixel pitch: an
error of half an ulp of 1 in the crossing (3e-8 of a pixel, 1.7e-8 rms) would show as 2.8e-7.  What is allowed is the
rounding of the weight's own FP32 steps, 12 of them (17 with the distance weight), each 2^-24 / sqrt 3
rms of the column offset, whose rms over the hat is 1 / sqrt 3: 6.9e-8 (8.2e-8); times 1.4 for steps
that are not independent.
"""
import numpy as np
import pytest
import torch

from fanbeamctrecon_tensorflowop_amd import workloads
from fanbeamctrecon_tensorflowop_amd.plan import FanBeamPlan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("views", [60, 200])  # a view's lines shared by four waves; a wave per view
def test_one_weight(weighted, views, oracle_mod):
    side, sid = 32, 200.0
    cols = int(16 * 1.1 * side)
    half = 1.1 * 0.5 * side / sid
    p, a = workloads.scan(nx=side, rfov=0.5 * side, sid=sid, sdd=2.0 * sid, n_cols=cols, dcol_rad=2.0 * half / cols,
                          n_views=views)
    plan, o = FanBeamPlan(p, a), oracle_mod.Oracle(p, a)
    rng = np.random.default_rng(views)
    x = np.zeros((8, side, side), dtype=np.float32)
    for s in range(8):
        j, i = rng.integers(6, side - 6, 2)
        x[s, j, i] = 1.0
    fn = plan.fbp_weighted_bp_adjoint if weighted else plan.bp_adjoint
    got = fn(torch.from_numpy(x).cuda()).double().cpu().numpy()
    ref = o.bp_adjoint(x, weighted=weighted)
    live = ref > 0.0
    e = float(np.sqrt(np.mean((got - ref)[live] ** 2)) / ref.max())
    print("weighted %d, %d views: %d weights, rms %.2e" % (weighted, views, live.sum(), e), flush=True)
    assert live.sum() >= 15 * views
    assert e <= 1.4 * (8.2e-8 if weighted else 6.9e-8)
