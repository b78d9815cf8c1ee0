"""GPU: the ramp filter's tile shapes at their edges, against the FP64 oracle.

The filter picks its tile by the row and column counts: 32 x 64 (few tiles), 64 x 128 and
128 x 256 (many columns and rows).  Each is run with rows and columns that no tile divides
and from row bases that are no multiple of 16 bytes.  Tolerance: 1e-5 relative L2, the
three-way split's (tests/test_gpu_parity.py).
"""
import numpy as np
import pytest
import torch

from conftest import rel_l2
from fanbeamctrecon_tensorflowop_amd import workloads
from fanbeamctrecon_tensorflowop_amd.cone import ConePlan
from fanbeamctrecon_tensorflowop_amd.plan import FanBeamPlan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("views,cols,slices", [
    (1, 2, 1), (3, 97, 1), (33, 64, 1), (31, 65, 2), (16, 257, 4),  # 32 x 64
    (90, 130, 115), (97, 767, 36), (64, 128, 321),                  # 64 x 128
    (97, 1000, 127), (128, 768, 128),                               # 128 x 256
])
def test_ramp_tiles(views, cols, slices, oracle_mod):
    p, a = workloads.tiny_scan(nx=16, n_views=views, n_cols=cols)
    plan, o = FanBeamPlan(p, a), oracle_mod.Oracle(p, a)
    y = np.random.default_rng(cols).normal(size=(slices,) + plan.sino_shape).astype(np.float32)
    buf = torch.empty(y.size + 1, device="cuda")
    buf[1:] = torch.from_numpy(y).cuda().reshape(-1)  # rows off the 16-byte grid
    got = plan.ramp_filter(buf[1:].view(y.shape)).double().cpu().numpy()
    for s in sorted({0, slices // 2, slices - 1}):
        e = rel_l2(got[s], o.ramp_filter(y[s:s + 1])[0])
        print("ramp %d views x %d columns, slice %d of %d: %.2e" % (views, cols, s, slices, e), flush=True)
        assert e <= 1e-5


@pytest.mark.parametrize("cols", [61, 300, 301])
def test_bf16_rows_of_any_length(cols):
    # BF16 values widen exactly, so the FP32 input's split has only its first part and the
    # products are the same; 1e-6 leaves room for another tile's order of accumulation
    g, a = workloads.cone_scan(nx=32, nz=4, n_views=20, n_cols=cols, n_rows=7)
    plan = ConePlan(g, a)
    x = torch.randn((2,) + plan.proj_shape, device="cuda").to(torch.bfloat16)
    e = rel_l2(plan.filter(x).double().cpu().numpy(), plan.filter(x.float()).double().cpu().numpy())
    print("bf16 rows of %d columns: %.2e" % (cols, e), flush=True)
    assert e <= 1e-6
