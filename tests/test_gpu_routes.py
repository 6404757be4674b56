"""Which kernel solved the subsets of a BATCHED correlation (read from the counts right after it), and the
workgroup-per-subset kernel against the oracle, on polygons, as the second pass of a combined optimization and
where it leaves a subset to the PLAIN kernel."""
import numpy as np
import pytest

import dice_amd as dh
from dice_amd import synth
from gpu_common import compare, run_oracle
from test_gpu_wide import H, W, check, params, scene  # noqa: F401 (scene: the fixture)

pytestmark = pytest.mark.gpu


def grid(S, step, margin):
    c = S // 2 + margin
    gx, gy = np.meshgrid(np.arange(c, W - c, step), np.arange(c, H - c, step))
    return gx.ravel().astype(float), gy.ravel().astype(float)


def batched(ctx, p, ref, de, f0):
    """The BATCHED result and its counts, then the PLAIN result."""
    ctx.set_params(p)
    ctx.set_ref_image(ref)
    ctx.set_def_image(de)
    fb = ctx.correlate(f0.copy())
    counts, left = ctx.pass_counts(), ctx.handover_counts()
    return fb, counts, left, ctx.correlate(f0.copy(), mode=dh.MODE_PLAIN)


@pytest.mark.parametrize("affine", [False, True], ids=["translation", "affine"])
@pytest.mark.parametrize("S,step", [(31, 8), (31, 40), (41, 8), (41, 40)])
def test_common_case_kernels_finish_the_subsets(scene, S, step, affine):
    ctx, ref, de = scene
    cx, cy = grid(S, step, 12)
    assert (len(cx) > 1024) == (step < 40)
    ctx.set_subsets(cx, cy, S)
    p = params(dh.GRADIENT_BASED, affine=affine)
    fb, counts, left, _ = batched(ctx, p, ref, de, dh.new_fields(cx, cy))
    assert counts == (0, 0, 0) and left == (0, 0, 0)


@pytest.mark.parametrize("affine", [False, True], ids=["translation", "affine"])
@pytest.mark.parametrize("S,step", [(47, 60), (75, 40), (125, 100)])
def test_wide_kernel_takes_large_subsets(scene, S, step, affine):
    ctx, ref, de = scene
    cx, cy = grid(S, step, 12)
    ctx.set_subsets(cx, cy, S)
    p = params(dh.GRADIENT_BASED, affine=affine)
    f0 = dh.new_fields(cx, cy)
    fb, counts, left, fp = batched(ctx, p, ref, de, f0)
    assert counts == (0, len(cx), 0)
    assert left[1:] == (0, 0)
    check(fb, fp)
    # (gamma of the translation-only fits is far from 0, so its bar holds without the float build)
    compare(fb, run_oracle(p, ref, de, cx, cy, S, fields=f0), ff=run_oracle(p, ref, de, cx, cy, S, fields=f0,
                                                                             precision="float"))


def test_wide_kernel_on_polygons(scene):
    ctx, ref, de = scene
    cx, cy, off, px, py, act = synth.conformal_subsets(60, W, H, area_lo=300, area_hi=3000, seed=9)
    conf = (off, px, py, act)
    ctx.set_subsets(cx, cy, 0, conformal=conf)
    p = params(dh.GRADIENT_BASED)
    f0 = dh.new_fields(cx, cy)
    fb, counts, left, fp = batched(ctx, p, ref, de, f0)
    assert 0 < counts[1] < len(cx)  # the small ones fit a wave's slot
    assert left[1:] == (0, 0)
    # the small ones: FP32 lane sums against PLAIN's FP64 ones, the parity bar; the others as in check()
    compare(fb, run_oracle(p, ref, de, cx, cy, 0, fields=f0, conformal=conf),
            ff=run_oracle(p, ref, de, cx, cy, 0, fields=f0, conformal=conf, precision="float"))
    big = np.diff(off) > 2500  # at least 57 px across: no slot holds them
    assert big.sum() >= 3
    check(fb[:, big], fp[:, big])


@pytest.mark.parametrize("opt,limit,value", [
    (dh.GRADIENT_BASED_THEN_SIMPLEX, "max_solver_iterations_fast", 2),
    (dh.SIMPLEX_THEN_GRADIENT_BASED, "max_solver_iterations_robust", 20),
], ids=["gradient-then-simplex", "simplex-then-gradient"])
@pytest.mark.parametrize("S,step", [(75, 60), (47, 16)], ids=["75px", "47px"])
def test_wide_kernel_as_the_second_pass(scene, S, step, opt, limit, value):
    """The first optimizer's limit stops it early, so its subsets go to the other one: the lists of the two
    passes change places."""
    ctx, ref, de = scene
    cx, cy = grid(S, step, 12)
    ctx.set_subsets(cx, cy, S)
    p = params(opt, affine=opt == dh.GRADIENT_BASED_THEN_SIMPLEX and S == 75)
    setattr(p, limit, value)
    fb, counts, left, fp = batched(ctx, p, ref, de, dh.new_fields(cx, cy))
    assert 0 < counts[0] <= len(cx)
    assert counts[1] == len(cx) and counts[2] == counts[0]
    assert left[1:] == (0, 0)
    check(fb, fp)


def test_wide_kernel_leaves_a_singular_system_to_plain(scene):
    """A single bright pixel on a ground of 0 at the subset's centre: gx is 0 off its row and gy off its column,
    so rotation and shear change nothing, their rows of the six-parameter system are exactly 0 and L D L^T is
    refused: the pivoted LU of the PLAIN kernel decides.  (The pixel is a place further on in the deformed image,
    or the solve would be skipped.)  The other subsets stay."""
    ctx, ref, de = scene
    S = 75
    cx, cy = grid(S, 80, 12)
    ref, de = ref.copy(), de.copy()
    k = len(cx) // 2
    x0, y0 = int(cx[k]), int(cy[k])
    for im in (ref, de):
        im[y0 - 44:y0 + 45, x0 - 44:x0 + 45] = 0.0
    ref[y0, x0] = de[y0, x0 + 1] = 0.01
    alone = np.maximum(np.abs(cx - x0), np.abs(cy - y0)) > 37 + 44 + 8  # subsets clear of the flat patch
    alone[k] = True
    cx, cy = cx[alone], cy[alone]
    k = int(alone[:k].sum())
    assert len(cx) > 3
    ctx.set_subsets(cx, cy, S)
    fb, counts, left, fp = batched(ctx, params(dh.GRADIENT_BASED), ref, de, dh.new_fields(cx, cy))
    assert counts == (0, len(cx), 0)
    assert left[1:] == (1, 0)
    assert np.array_equal(fb[:, k], fp[:, k], equal_nan=True)
    rest = np.arange(len(cx)) != k
    check(fb[:, rest], fp[:, rest])
