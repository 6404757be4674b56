"""correlate_wide_kernel (one workgroup per subset with the deformed window in LDS) against the PLAIN
kernel on the same inputs: both add the same float terms in FP64, so statuses and iteration counts agree
and the results differ by float rounding only.  Sizes: windows just above a wave's slot, one near the
kernel's own LDS window, one beyond it (taps from the image), few subsets (1024 threads each) and many
(256), subsets that run into the image border (handed on to the PLAIN kernel)."""
import numpy as np
import pytest

import dice_amd as dh
from dice_amd import synth

pytestmark = pytest.mark.gpu

W, H = 420, 404


@pytest.fixture(scope="module")
def scene():
    sp = synth.Speckle(W, H, seed=21)
    ref = sp.frame(None)
    de = sp.frame(synth.affine_field(0.7, -0.4, 0.004, 0.002, -0.003, 0.005), noise_sigma=2.0, noise_seed=22)
    ctx = dh.Context(0)
    yield ctx, ref, de
    ctx.close()


def both_modes(ctx, p, ref, de, f0):
    ctx.set_params(p)
    ctx.set_ref_image(ref)
    ctx.set_def_image(de)
    return [ctx.correlate(f0.copy(), mode=m) for m in (dh.MODE_BATCHED, dh.MODE_PLAIN)]


def check(fb, fp):
    for name in ("STATUS", "ITERATIONS", "ACTIVE_PIXELS", "MATCH"):
        assert np.array_equal(fb[dh.F[name]], fp[dh.F[name]]), name
    ok = np.isin(fp[dh.F["STATUS"]], dh.CONVERGED_STATUSES)
    assert ok.any()
    # a rounding of the update by one ulp of a parameter below 2 px
    for name in ("DISP_X", "DISP_Y", "ROT_Z", "NS_XX", "NS_YY", "SS_XY"):
        assert np.abs(fb[dh.F[name]] - fp[dh.F[name]]).max() <= 1e-6, name
    for name in ("GAMMA", "SIGMA", "NOISE", "CONTRAST", "CONDITION") + tuple("FIELD_%d" % k for k in range(1, 8)):
        a, b = fb[dh.F[name]], fp[dh.F[name]]
        assert np.abs(a - b).max() <= 2e-5 * max(np.abs(b).max(), 1e-3), name


def params(opt, interp=dh.KEYS_FOURTH, affine=True):
    p = dh.default_params()
    p.optimization_method = opt
    p.interpolation_method = interp
    if affine:
        p.enable_rotation = p.enable_normal_strain = p.enable_shear_strain = 1
    return p


@pytest.mark.parametrize("S,step,interp,affine,dtype", [
    (45, 60, dh.KEYS_FOURTH, True, np.float32),   # the smallest windows above the slot: through the list
    (57, 12, dh.KEYS_FOURTH, True, np.float32),   # many subsets: 256 threads each
    (75, 40, dh.KEYS_FOURTH, False, np.uint16),
    (91, 60, dh.BILINEAR, True, np.uint16),
    (125, 50, dh.KEYS_FOURTH, True, np.float32),  # beyond the LDS window
])
def test_gauss_newton(scene, S, step, interp, affine, dtype):
    ctx, ref, de = scene
    if dtype == np.uint16:
        ref, de = [np.clip(np.round(np.maximum(i, 0) * 16), 0, 4095).astype(np.uint16) for i in (ref, de)]
    # centres up to the border: some warped subsets lose pixels to the guard
    c = S // 2 + 3
    gx, gy = np.meshgrid(np.arange(c, W - c, step), np.arange(c, H - c, step))
    cx, cy = gx.ravel().astype(float), gy.ravel().astype(float)
    ctx.set_subsets(cx, cy, S)
    p = params(dh.GRADIENT_BASED, interp, affine)
    fb, fp = both_modes(ctx, p, ref, de, dh.new_fields(cx, cy))
    assert ctx.pass_counts() == (0, 0, 0)  # the PLAIN run's
    check(fb, fp)


@pytest.mark.parametrize("S,n,interp", [(61, 5, dh.KEYS_FOURTH), (49, 9, dh.BILINEAR), (125, 2, dh.KEYS_FOURTH),
                                        (47, 300, dh.KEYS_FOURTH)])
def test_simplex(scene, S, n, interp):
    ctx, ref, de = scene
    rng = np.random.default_rng(S)
    cx = rng.integers(S // 2 + 4, W - S // 2 - 4, n).astype(float)
    cy = rng.integers(S // 2 + 4, H - S // 2 - 4, n).astype(float)
    ctx.set_subsets(cx, cy, S)
    p = params(dh.SIMPLEX, interp, False)
    p.enable_rotation = 1
    check(*both_modes(ctx, p, ref, de, dh.new_fields(cx, cy)))
