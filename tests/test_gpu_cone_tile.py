"""GPU: the staged cone backprojection kernels where a view of a tile may be staged or not, against the FP64
oracle: short last z-chunks, detectors narrower than the FOV (the in-range decision of voxels at the fan's
edges), windows too tall (rows magnified near the source) or too wide (fine columns) for some tiles and views.

The plan's own windows say that a case has both staged and unstaged (tile, view) pairs.  Which kernel a volume
takes follows from its size: 16 x 16 pixel tiles from 16 slices on where there are more than 1024 tiles times
chunks of 16 slices and less than 2.2 detector rows between two slices, else 8 x 8 pixel tiles.

Every voxel is bounded by itself.  A column coordinate carries, in units of 2^-24 of half the detector, 4 for t, 4
for U, 2 for the reciprocal, 3 for products and the sum and 3 for the arc tangent: 16; a row coordinate 7 for the
magnification and 5 for products and sums: 12.  An error of a coordinate changes an update by that times the
difference of the taps on either side, which the oracle backprojects as it does the values; weights and
interpolation take 20 roundings of an update, the sum one for each view.
"""
import math

import numpy as np
import pytest
import torch

from conftest import rel_l2
from fanbeamctrecon_tensorflowop_amd import workloads
from fanbeamctrecon_tensorflowop_amd.cone import ConePlan, cone_geom

pytestmark = pytest.mark.gpu

R, D = 250.0, 470.0

# tile side, pixels, slices, pixel (mm), views, part of the FOV fan on the detector, column pitch, row pitch (mm),
# whether (nearly) every pair is staged
CASES = {
    "short_chunk": (16, 272, 50, 0.5, 9, 1.1, 1.2, 1.2, True),
    "one_slice_over": (16, 300, 33, 0.4, 7, 1.1, 1.1, 0.9, True),
    "narrow_detector": (16, 272, 50, 0.5, 11, 0.6, 1.0, 1.2, False),
    "tall_windows": (16, 272, 50, 0.5, 9, 1.1, 1.0, 0.44, False),
    "wide_windows": (16, 272, 50, 0.5, 9, 1.1, 0.3, 1.2, False),
    "wave_wide_windows": (8, 24, 16, 2.0, 30, 1.1, 1.0, 2.0, False),
    "wave_narrow_short": (8, 61, 21, 1.0, 24, 0.7, 1.3, 1.6, False),
}


def _check(plan, g, a, seed, what, oracle_mod):
    cols, rows, views, nz, dx = (g[k] for k in ("nCols", "nRows", "nViews", "nZ", "dx"))
    ells = workloads.random_ellipsoids(6, seed=seed, rfov=g["rFOV"], zhalf=0.5 * nz * dx)
    P = workloads.ellipsoid_projections(ells, g, a).numpy()
    P = (P + np.random.default_rng(nz).normal(0, 1e-3, size=P.shape)).astype(np.float32)
    q = plan.filter(torch.from_numpy(P[None]).cuda())
    got = plan.backproject(q)[0].double().cpu().numpy()
    q, o = q.double().cpu().numpy(), oracle_mod.ConeOracle(g, a)
    ref, eps = o.backproject(q)[0], 2.0 ** -24

    def steps(axis):  # the larger of a sample's differences to its neighbours
        d = np.abs(np.diff(q, axis=axis))
        pad = [(0, 0)] * q.ndim
        pad[axis] = (0, 1)
        low = np.pad(d, pad)
        pad[axis] = (1, 0)
        return np.maximum(low, np.pad(d, pad))

    bound = (8.0 * eps * cols * o.backproject(steps(3))[0] + 6.0 * eps * rows * o.backproject(steps(2))[0]
             + (20 + views) * eps * o.backproject(np.abs(q))[0])
    err = np.abs(got - ref)
    worst = float((err / np.maximum(bound, 1e-30)).max())
    print("%s, rel_l2 %.2e, worst voxel %.2f of its bound" % (what, rel_l2(got, ref), worst), flush=True)
    assert worst <= 1.0
    assert np.count_nonzero(bound) > 0.7 * bound.size


@pytest.mark.parametrize("detector", ["flat", "curved"])
@pytest.mark.parametrize("name", sorted(CASES))
def test_staged_and_not(name, detector, oracle_mod):
    side, nx, nz, dx, views, cover, d_col, d_row, whole = CASES[name]
    rfov = 0.5 * nx * dx
    half = cover * math.asin(rfov / R)
    cols = int(2.0 * D * math.tan(half) / d_col)
    rows = int(1.3 * nz * dx * D / R / d_row)
    pitch = 2.0 * half / cols if detector == "curved" else d_col
    chunk = side
    g = cone_geom(R=R, D=D, n_views=views, d_angle=2.0 * math.pi / views, detector=detector, n_cols=cols, n_rows=rows,
                  d_col=pitch, d_row=d_row, nx=nx, nz=nz, dx=dx, dz=dx)
    a = (np.arange(views) * (2.0 * math.pi / views) + 0.1).astype(np.float32)
    plan = ConePlan(g, a)
    step, tiles = dx * D / d_row / R, math.ceil(nx / 16) ** 2 * math.ceil(nz / 16)
    assert (side == 16) == (nz >= 16 and step < 2.2 and tiles > 1024)
    staged = [plan.windows(side, i, j, k)[:, 0] for i in range(0, nx, side) for j in range(0, nx, side)
              for k in range(0, nz, chunk)
              # tiles with a pixel inside the FOV disk
              if min(abs(c - 0.5 * nx) for c in (i + 0.5, min(i + side, nx) - 0.5)) ** 2
              + min(abs(c - 0.5 * nx) for c in (j + 0.5, min(j + side, nx) - 0.5)) ** 2 < (0.5 * nx) ** 2]
    share = float(np.mean(staged))
    assert share > 0.98 if whole else 0.1 < share < 0.95
    _check(plan, g, a, nx + nz, "%s %s: %.2f staged" % (name, detector, share), oracle_mod)


# few views: 16, 8 and 4 waves a tile (sums over the waves), of 8 slices (8 x 8 pixel tiles times chunks of 8 from
# 700 and 1500 on) and from global memory
@pytest.mark.parametrize("nx,nz,d_row,views", [
    (60, 56, 1.5, 9), (80, 56, 1.5, 9), (80, 56, 1.5, 40), (80, 56, 1.5, 64), (100, 72, 1.5, 1), (100, 72, 1.5, 9),
    (100, 72, 1.5, 57), (240, 4, 1.5, 3), (240, 4, 1.5, 33), (60, 4, 1.5, 17),
])
def test_few_views(nx, nz, d_row, views, oracle_mod):
    half = 1.1 * math.asin(0.5 * nx / R)
    cols, rows = int(2.0 * D * math.tan(half) / 1.4), int(1.3 * nz * D / R / d_row)
    g = cone_geom(R=R, D=D, n_views=views, d_angle=2.0 * math.pi / views, detector="flat", n_cols=cols, n_rows=rows,
                  d_col=1.4, d_row=d_row, nx=nx, nz=nz, dx=1.0, dz=1.0)
    a = (np.arange(views) * (2.0 * math.pi / views) + 0.1).astype(np.float32)
    _check(ConePlan(g, a), g, a, nx + nz, "%d x %d, %d views" % (nx, nz, views), oracle_mod)
