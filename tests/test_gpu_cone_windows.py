"""GPU: the staged cone backprojection kernels where a tile's corners lie outside the FOV disk of a wide
fan, beyond the range that the polynomial of atan is fitted on (tests/test_cone_windows.py checks the
windows themselves), against the FP64 oracle.

Relative L2 <= 1e-5, as for every FP32 reconstruction of this suite."""
import math

import numpy as np
import pytest
import torch

from conftest import rel_l2
from fanbeamctrecon_tensorflowop_amd import workloads
from fanbeamctrecon_tensorflowop_amd.cone import ConePlan, cone_geom

pytestmark = pytest.mark.gpu


# side, rFOV / R, columns, fan / FOV fan, slices, views: 8 x 8 pixel tiles, then (more than 1024 tiles times
# chunks of sixteen slices) 16 x 16 pixel tiles
@pytest.mark.parametrize("side,ratio,cols,cover,nz,views", [
    (12, 0.605, 40, 1.2, 8, 30), (16, 0.63, 64, 1.2, 8, 30), (17, 0.63, 64, 1.2, 13, 30), (25, 0.62, 70, 1.2, 8, 24),
    (17, 0.645, 64, 0.9, 8, 30), (16, 0.8, 64, 1.1, 8, 30),
    (40, 0.62, 90, 1.2, 1840, 10), (24, 0.605, 70, 1.2, 4104, 10),
])
@pytest.mark.parametrize("detector", ["curved", "flat"])
def test_wide_fans(side, ratio, cols, cover, nz, views, detector, oracle_mod):
    R, D = 250.0, 470.0
    rfov, half, zhalf = ratio * R, cover * math.asin(ratio), 20.0
    d_col = 2.0 * half / cols if detector == "curved" else 2.0 * D * math.tan(half) / cols
    g = cone_geom(R=R, D=D, n_views=views, d_angle=2.0 * math.pi / views, detector=detector, n_cols=cols, n_rows=24,
                  d_col=d_col, d_row=5.0, nx=side, nz=nz, dx=2.0 * rfov / side, dz=2.0 * zhalf / nz)
    a = (np.arange(views) * (2.0 * math.pi / views) + 0.1).astype(np.float32)
    ells = workloads.random_ellipsoids(6, seed=side + nz, rfov=rfov, zhalf=zhalf)
    P = workloads.ellipsoid_projections(ells, g, a).numpy()
    P = (P + np.random.default_rng(nz).normal(0, 1e-3, size=P.shape)).astype(np.float32)
    got = ConePlan(g, a).fdk(torch.from_numpy(P[None]).cuda())
    e = rel_l2(got.double().cpu().numpy(), oracle_mod.ConeOracle(g, a).fdk(P[None].astype(np.float64)))
    print("%s %d px, rFOV/R %g, %d slices: %.2e" % (detector, side, ratio, nz, e), flush=True)
    assert e <= 1e-5
