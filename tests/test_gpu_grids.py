"""GPU: calls with more workgroups than one axis of a launch grid holds."""
import numpy as np
import pytest
import torch

from conftest import rel_l2
from fanbeamctrecon_tensorflowop_amd import workloads
from fanbeamctrecon_tensorflowop_amd.batch import UnevenBatch
from fanbeamctrecon_tensorflowop_amd.plan import FanBeamPlan

pytestmark = pytest.mark.gpu


def test_uneven_adjoint_of_many_slices():
    # 3070 slices of 512 x 512 pixels: 74 x 74 cell tiles each, 2^24 + 34104 workgroups of 256 threads
    p, a = workloads.scan(nx=512, rfov=128.0, sid=500.0, sdd=1000.0, n_cols=24, dcol_rad=0.02, n_views=2)
    plan = FanBeamPlan(p, a)
    n = 3070
    assert n * 74 * 74 > 2 ** 24
    batch = UnevenBatch([plan] * n)
    y = torch.randn((n,) + plan.sino_shape, generator=torch.Generator().manual_seed(1)).cuda()
    out = batch.fp_adjoint(y.reshape(-1))
    for s in (0, n // 2, n - 2, n - 1):
        assert torch.equal(batch.image(out, s), plan.fp_adjoint(y[s:s + 1])[0]), s


@pytest.mark.parametrize("views,dcol", [(70000, 0.02), (270000, 0.006)])  # a view a workgroup, four views
def test_bp_adjoint_of_many_views(views, dcol, oracle_mod):
    # more than 65536 view groups, in either split of the work
    p, a = workloads.scan(nx=4, rfov=2.0, sid=60.0, sdd=120.0, n_cols=8, dcol_rad=dcol, n_views=views)
    plan, o = FanBeamPlan(p, a), oracle_mod.Oracle(p, a)
    x = np.random.default_rng(views).normal(size=(2,) + plan.image_shape).astype(np.float32)
    for fn, weighted in ((plan.bp_adjoint, False), (plan.fbp_weighted_bp_adjoint, True)):
        got = fn(torch.from_numpy(x).cuda()).double().cpu().numpy()
        e = rel_l2(got, o.bp_adjoint(x, weighted=True) if weighted else o.bp_adjoint(x))
        print("%d views: %.2e" % (views, e), flush=True)
        assert e <= 1e-5
