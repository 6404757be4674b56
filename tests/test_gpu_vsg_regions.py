"""VSG radius windows (dice_hip_vsg_strain) on subsets that are dense in a part of their bounds, against the oracle:
a region and a few subsets far from it, where the lanes deal out candidates instead of cell rows (cells as wide as
the radius, between half of it and it, and just below half), and a cell with more entries than the LDS tile holds.

Bar as in test_gpu_vsg_cells: MATCH identical, fields within one float ulp or 1e-12 of the sum that cancels."""
import numpy as np
import pytest

import dice_amd as dh
import oracle_py as o

pytestmark = pytest.mark.gpu

CASES = {
    # side of the region, step, extent of the whole, window: radius and cell side
    "as-the-radius": (100, 5, 2000, 41),       # 20, 20
    "above-half": (450, 5, 2000, 61),          # 30, 21
    "just-below-half": (450, 5, 1200, 61),     # 30, 13
    "rows": (450, 5, 600, 61),                 # 30, 7.5
    "crowded": (50, 1, 1500, 61),              # 30, 29: a cell of 870 subsets, ranges beyond the tile
    "alone": (6, 2, 1500, 21),                 # 10, 10: few subsets
}


@pytest.mark.parametrize("name", list(CASES))
def test_vsg_regions(name):
    side, step, extent, window = CASES[name]
    gx, gy = np.meshgrid(np.arange(0.0, side, step), np.arange(0.0, side, step))
    cx = np.concatenate([gx.ravel(), [extent, extent, extent - 4.0, 0.0]])
    cy = np.concatenate([gy.ravel(), [0.0, extent, extent - 3.0, extent]])
    rng = np.random.default_rng(len(name))
    order = rng.permutation(len(cx))
    cx, cy = cx[order], cy[order]
    f = dh.new_fields(cx, cy)
    f[dh.F["DISP_X"]] = (0.5 + 0.002 * cx + 0.2 * np.sin(cy / 80)).astype(np.float32)
    f[dh.F["DISP_Y"]] = (-0.3 + 0.001 * cy + 0.1 * np.cos(cx / 50)).astype(np.float32)
    f[dh.F["SIGMA"]] = 0.01
    f[dh.F["SIGMA"], rng.random(len(cx)) < 0.05] = -1.0
    fg, fo = f.copy(), f.copy()
    with dh.Context(0) as ctx:
        ctx.set_subsets(np.round(cx), np.round(cy), 21)
        vg = ctx.vsg_strain(fg, window)
    vo = o.vsg_strain(fo, window)
    assert np.array_equal(fg[dh.F["MATCH"]], fo[o.F["MATCH"]])
    assert np.all(np.abs(vg - vo) <= 1.2e-7 * np.abs(vo) + 1e-12), np.abs(vg - vo).max()
