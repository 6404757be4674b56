"""The cell-ordered list and the row extents behind the VSG radius windows (dice_hip_vsg_strain) against the
oracle, at the sizes where they can go wrong: windows below the step (no neighbour but the subset itself),
exactly at a neighbour's distance, cell counts around one scan group (1024) and far beyond it, more candidates
than the LDS tile holds, all subsets in one cell, and centres far from the origin.

Bar as in test_gpu_vsg: MATCH identical, fields within one float ulp or 1e-12 of the sum that cancels; the sums
are FP64 over the same neighbours in another order."""
import numpy as np
import pytest

import dice_amd as dh
import oracle_py as o

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = dh.Context(0)
    yield c
    c.close()


def square(nx, ny, step):
    return [g.ravel().astype(np.float64) for g in np.meshgrid(np.arange(nx) * step, np.arange(ny) * step)]


CASES = {
    "below-step": (square(40, 30, 9.0), 5, 0.0),
    "at-distance": (square(70, 33, 5.0), 40, 0.0),
    "row": (square(1100, 1, 4.0), 33, 0.0),
    "column": (square(1, 1025, 4.0), 33, 0.0),
    "many-cells": (square(110, 90, 6.0), 26, 0.0),
    "dense-tile": (square(90, 60, 1.0), 61, 0.0),
    "one-cell": (square(20, 20, 0.04), 400, 0.0),
    "far-away": (square(50, 40, 3.25), 31, 40000.0),
}


@pytest.mark.parametrize("name", list(CASES))
def test_vsg_cells(ctx, name):
    (cx, cy), window, offset = CASES[name]
    rng = np.random.default_rng(len(name))
    order = rng.permutation(len(cx))  # ids in no order of place
    cx, cy = cx[order] + offset, cy[order] + offset
    ctx.set_subsets(np.round(cx), np.round(cy), 21)
    f = dh.new_fields(cx, cy)
    f[dh.F["DISP_X"]] = (0.5 + 0.002 * (cx - offset) + 0.2 * np.sin((cy - offset) / 80)).astype(np.float32)
    f[dh.F["DISP_Y"]] = (-0.3 + 0.001 * (cy - offset) + 0.1 * np.cos((cx - offset) / 50)).astype(np.float32)
    f[dh.F["SIGMA"]] = 0.01
    f[dh.F["SIGMA"], rng.random(len(cx)) < 0.05] = -1.0
    fg, fo = f.copy(), f.copy()
    vg, vo = ctx.vsg_strain(fg, window), o.vsg_strain(fo, window)
    assert np.array_equal(fg[dh.F["MATCH"]], fo[o.F["MATCH"]])
    assert np.all(np.abs(vg - vo) <= 1.2e-7 * np.abs(vo) + 1e-12), np.abs(vg - vo).max()
