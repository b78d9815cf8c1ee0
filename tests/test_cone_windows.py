"""The detector windows of the staged cone backprojection kernels hold every tap of the voxels inside the
FOV disk, checked on the host against FP64 coordinates: fans from narrow to the widest whose atan is a
polynomial (tile corners outside the disk lie beyond the range that it is fitted on), flat detectors,
sources close to the volume, and detectors whose rows lie beyond the range that a window can start at."""
import math

import numpy as np
import pytest

from fanbeamctrecon_tensorflowop_amd.cone import ConePlan, cone_geom

KZ = {8: 8, 16: 16}


def _plan(detector, side, ratio, cols, cover, nz=8, rows=24, views=30, d_row=2.5, row_bottom=None):
    R, D = 250.0, 470.0
    rfov = ratio * R
    half = cover * math.asin(ratio)
    d_col = 2.0 * half / cols if detector == "curved" else 2.0 * D * math.tan(min(half, 1.4)) / cols
    g = cone_geom(R=R, D=D, n_views=views, d_angle=2.0 * math.pi / views, detector=detector, n_cols=cols, n_rows=rows,
                  d_col=d_col, d_row=d_row, row_bottom=row_bottom, nx=side, nz=nz, dx=2.0 * rfov / side, dz=1.0)
    return ConePlan(g, (np.arange(views) * (2.0 * math.pi / views) + 0.1).astype(np.float32))


def _check(plan, side):
    """Number of staged (tile, view) pairs; asserts that none of them misses a tap."""
    g = plan.geom
    staged = 0
    beta = plan.angles.astype(np.float64).reshape(-1, 1)
    for k0 in range(0, g["nZ"], KZ[side]):
        for j0 in range(0, g["nY"], side):
            for i0 in range(0, g["nX"], side):
                w = plan.windows(side, i0, j0, k0)
                i, j = np.meshgrid(np.arange(i0, min(i0 + side, g["nX"])), np.arange(j0, min(j0 + side, g["nY"])))
                x, y = (g["xmin"] + g["dx"] * (i.ravel() + 0.5)), (g["ymin"] + g["dy"] * (j.ravel() + 0.5))
                keep = x * x + y * y <= g["rFOV"] ** 2 * (1.0 - 1e-6)
                x, y = x[keep], y[keep]
                if x.size == 0:
                    continue
                U, t = g["R"] - x * np.cos(beta) - y * np.sin(beta), x * np.sin(beta) - y * np.cos(beta)
                a = np.arctan(t / U) if g["detector"] == 1 else g["D"] * t / U
                ct = (a - g["colLeft"]) / g["dCol"] + g["dShift"] - 0.5
                ends = []
                for k in (k0, min(k0 + KZ[side], g["nZ"]) - 1):
                    z = g["zmin"] + g["dz"] * (k + 0.5)
                    ends.append((z * g["D"] / U - g["rowBottom"]) / g["dRow"] - 0.5)
                for v in np.nonzero(w[:, 0])[0]:
                    staged += 1
                    rows = np.floor([e[v] for e in ends])
                    msg = "tile %d,%d,%d side %d view %d: %s" % (i0, j0, k0, side, v, w[v])
                    assert np.floor(ct[v]).min() >= w[v, 1] and np.floor(ct[v]).max() + 1 <= w[v, 2], msg
                    assert rows.min() >= w[v, 3] and rows.max() + 1 <= w[v, 4], msg
    return staged


@pytest.mark.parametrize("ratio", [0.2, 0.45, 0.55, 0.59, 0.605, 0.62, 0.63, 0.645, 0.66, 0.8])
@pytest.mark.parametrize("detector", ["curved", "flat"])
def test_taps_lie_in_staged_windows(detector, ratio):
    staged = 0
    for side, cols in ((12, 40), (16, 64), (17, 64), (25, 70), (40, 90)):
        for cover in (0.9, 1.2):
            plan = _plan(detector, side, ratio, cols, cover)
            staged += sum(_check(plan, s) for s in (8, 16))
    assert staged > 0


def test_source_close_to_the_disk():
    for ratio in (0.95, 0.99):
        for s in (8, 16):
            _check(_plan("curved", 30, ratio, 200, 1.05), s)


def test_rows_far_from_the_detector():
    # a volume whose shadow lies 2.3e6 rows from row 0, beyond the 1e6 at which a window's ends are cut
    for sign in (1.0, -1.0):
        plan = _plan("curved", 16, 0.3, 64, 1.2, d_row=1e-3, row_bottom=sign * 2300.0, rows=32)
        assert _check(plan, 8) == 0 and _check(plan, 16) == 0
