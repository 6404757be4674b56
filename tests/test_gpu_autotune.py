"""dice_hip_autotune: the default launch shape is among those that it times, and a tuned shape is kept for the
parameters that it was tuned with."""
import numpy as np
import pytest

import dice_amd as dh
from dice_amd import synth

pytestmark = pytest.mark.gpu

DEFAULT_SLOT = 2560


@pytest.fixture(scope="module")
def scene():
    w, h = 700, 560
    sp = synth.Speckle(w, h, seed=61)
    return w, h, sp.frame(None), sp.frame(synth.affine_field(0.4, -0.3, 0.0, 0.0, 0.0, 0.0), noise_sigma=1.0,
                                          noise_seed=62)


def setup(ctx, scene, p, S, step):
    w, h, ref, de = scene
    c = S // 2 + 8
    gx, gy = np.meshgrid(np.arange(c, w - c, step), np.arange(c, h - c, step))
    cx, cy = gx.ravel().astype(float), gy.ravel().astype(float)
    ctx.set_params(p)
    ctx.set_ref_image(ref)
    ctx.set_def_image(de)
    ctx.set_subsets(cx, cy, S)
    return dh.new_fields(cx, cy)


def params(affine):
    p = dh.default_params()
    p.optimization_method = dh.GRADIENT_BASED
    if affine:
        p.enable_rotation = p.enable_normal_strain = p.enable_shear_strain = 1
    return p


def device(f):
    import torch
    return torch.from_numpy(f).to("cuda:0")


def test_large_subsets_keep_the_default_slot():
    """At 91 px, default parameters, a workgroup per subset (the default slot) takes two thirds of the time of one
    wave per subset in the best slot that holds the windows (0.99 and 1.48 ms for 3,400 subsets), far more than a
    run's own spread."""
    w, h = 1000, 800
    sp = synth.Speckle(w, h, seed=63)
    scene = w, h, sp.frame(None), sp.frame(synth.affine_field(0.4, -0.3, 0.0, 0.0, 0.0, 0.0))
    with dh.Context(0) as ctx:
        f0 = setup(ctx, scene, params(False), 91, 14)
        ctx.autotune(device(f0).data_ptr())
        assert ctx.launch_shape()[2] == DEFAULT_SLOT
        ctx.correlate(f0.copy())
        assert ctx.pass_counts() == (0, f0.shape[1], 0)


def test_a_shape_of_ones_own_is_timed_too(scene):
    """The shape that is set when the tuner is called can win; whichever does is a legal one and is set after it."""
    with dh.Context(0) as ctx:
        f0 = setup(ctx, scene, params(True), 31, 9)
        ctx.set_launch_shape(3, 4, 2600)
        ctx.autotune(device(f0).data_ptr())
        waves, per_cu, slot = ctx.launch_shape()
        assert waves in (1, 2, 3, 4) and slot >= DEFAULT_SLOT
        fb = ctx.correlate(f0.copy())
        assert np.isin(fb[dh.F["STATUS"]], dh.CONVERGED_STATUSES).mean() > 0.99


def test_a_tuned_shape_belongs_to_its_parameters(scene):
    """Translation-only and six-parameter frames run different kernels.  Whether the tuner ran is read from the
    counts of the last launch: the frame before starts 3,000 px off, so all of its subsets are handed over, and the
    tuner's own runs hand over none."""
    with dh.Context(0) as ctx:
        f0 = setup(ctx, scene, params(True), 31, 9)
        d = device(f0)
        off = f0.copy()
        off[dh.F["DISP_X"]] = -3000.0

        def tuned():
            ctx.correlate(off.copy(), first_frame=False)
            assert ctx.handover_counts()[0] == f0.shape[1]
            ctx.autotune(d.data_ptr())
            return ctx.handover_counts()[0] == 0

        assert tuned()
        assert not tuned()  # kept
        ctx.set_params(params(False))
        assert tuned()
        assert not tuned()
        ctx.set_params(params(True))
        assert not tuned()  # the first one's again
