"""The common-case Gauss-Newton kernels against each other on one set of square subsets: the
translation-only kernel against the general kernel (taken with an initial-gamma threshold that no subset
exceeds), and the crews of four waves (at most 1024 subsets) against one wave per subset.  They add the
same FP32 terms in the same order, so parameters, statuses and iteration counts are equal bit for bit;
the other fields (sums in another order) agree to float rounding."""
import numpy as np
import pytest

import dice_amd as dh
from dice_amd import synth

pytestmark = pytest.mark.gpu

W, H = 390, 371
EXACT = ("DISP_X", "DISP_Y", "ROT_Z", "NS_XX", "NS_YY", "SS_XY", "STATUS", "ITERATIONS", "ACTIVE_PIXELS", "MATCH",
         "CONDITION")
CLOSE = ("SIGMA", "GAMMA", "NOISE", "CONTRAST") + tuple("FIELD_%d" % k for k in range(1, 8))


@pytest.fixture(scope="module")
def scene():
    sp = synth.Speckle(W, H, seed=31)
    ref = sp.frame(None)
    de = sp.frame(synth.affine_field(0.6, -0.7, 0.002, 0.001, -0.001, 0.002), noise_sigma=2.0, noise_seed=32)
    ctx = dh.Context(0)
    yield ctx, ref, de
    ctx.close()


def run(ctx, p, ref, de, cx, cy, S):
    ctx.set_params(p)
    ctx.set_ref_image(ref)
    ctx.set_def_image(de)
    ctx.set_subsets(cx, cy, S)
    f0 = dh.new_fields(cx, cy)
    # a whole-pixel start among them: v + dy then rounds across integers
    f0[dh.F["DISP_X"]] = np.where(np.arange(len(cx)) % 3 == 0, -1e-8, 0.25)
    f0[dh.F["DISP_Y"]] = np.where(np.arange(len(cx)) % 5 == 0, -1e-8, 0.0)
    first = ctx.correlate(f0.copy(), first_frame=False)
    again = ctx.correlate(f0.copy(), first_frame=False)  # from the cached per-subset constants
    for name in EXACT:
        assert np.array_equal(first[dh.F[name]], again[dh.F[name]]), name
    return first


def same(a, b):
    assert np.isin(a[dh.F["STATUS"]], dh.CONVERGED_STATUSES).mean() > 0.5
    for name in EXACT:
        assert np.array_equal(a[dh.F[name]], b[dh.F[name]]), name
    for name in CLOSE:
        x, y = a[dh.F[name]], b[dh.F[name]]
        assert np.abs(x - y).max() <= 2e-5 * max(np.abs(y).max(), 1e-3), name


@pytest.mark.parametrize("affine", [False, True], ids=["translation", "affine"])
@pytest.mark.parametrize("S,interp,dtype", [(5, dh.KEYS_FOURTH, np.float32), (31, dh.KEYS_FOURTH, np.uint16),
                                            (33, dh.BILINEAR, np.float32), (37, dh.KEYS_FOURTH, np.float32),
                                            (43, dh.KEYS_FOURTH, np.float32), (43, dh.BILINEAR, np.uint16)])
def test_same_results(scene, S, interp, dtype, affine):
    ctx, ref, de = scene
    if dtype == np.uint16:
        ref, de = [np.clip(np.round(np.maximum(i, 0) * 16), 0, 4095).astype(np.uint16) for i in (ref, de)]
    c = S // 2  # up to the border: subsets that the common case hands over
    gx, gy = np.meshgrid(np.arange(c, W - c, 9), np.arange(c, H - c, 9))
    cx, cy = gx.ravel().astype(float), gy.ravel().astype(float)
    assert len(cx) > 1024
    p = dh.default_params()
    p.optimization_method = dh.GRADIENT_BASED
    p.interpolation_method = interp
    if affine:
        p.enable_rotation = p.enable_normal_strain = p.enable_shear_strain = 1
    wave = run(ctx, p, ref, de, cx, cy, S)
    few = np.arange(0, len(cx), 7)
    crew = run(ctx, p, ref, de, cx[few], cy[few], S)
    # (the start values depend on the index)
    keep = (np.arange(len(few)) % 3 == 0) == (few % 3 == 0)
    keep &= (np.arange(len(few)) % 5 == 0) == (few % 5 == 0)
    same(wave[:, few][:, keep], crew[:, keep])
    if not affine:
        q = dh.default_params()
        for name, _ in dh.Params._fields_:
            setattr(q, name, getattr(p, name))
        q.initial_gamma_threshold = 1e9
        general = run(ctx, q, ref, de, cx, cy, S)
        ok = general[dh.F["STATUS"]] != 5  # flat or empty subsets fail the threshold
        same(wave[:, ok], general[:, ok])


@pytest.mark.parametrize("step", [6, 55], ids=["wave", "crew"])
def test_bilinear_uncertainty_far_from_the_origin(step):
    """With bilinear images the uncertainty fields take each pixel's weights from the float sum x + u, which
    rounds by 2^-13 px at x = 1100: the translation kernels follow the general one in that.  The terms are
    positive and at most 64 pixels go to an FP32 lane sum in each kernel, in another order: 64 * 2^-24 on r_tot2
    and the other sums, half of that after the root, twice for the two kernels: 4e-6."""
    w, h, S = 1300, 200, 35
    sp = synth.Speckle(w, h, seed=33)
    ref = sp.frame(None)
    de = sp.frame(synth.affine_field(0.37, -0.21, 0.0, 0.0, 0.0, 0.0), noise_sigma=1.0, noise_seed=34)
    gx, gy = np.meshgrid(np.arange(22, w - 22, step), np.arange(22, h - 22, step))
    cx, cy = gx.ravel().astype(float), gy.ravel().astype(float)
    assert (len(cx) > 1024) == (step == 6)
    p = dh.default_params()
    p.optimization_method = dh.GRADIENT_BASED
    p.interpolation_method = dh.BILINEAR
    ctx = dh.Context(0)
    a = run(ctx, p, ref, de, cx, cy, S)
    p.initial_gamma_threshold = 1e9
    b = run(ctx, p, ref, de, cx, cy, S)
    ctx.close()
    for name in EXACT:
        assert np.array_equal(a[dh.F[name]], b[dh.F[name]]), name
    ok = np.isin(a[dh.F["STATUS"]], dh.CONVERGED_STATUSES)
    assert ok.mean() > 0.9
    for k in (1, 3, 4, 5, 6, 7):
        x, y = a[dh.F["FIELD_%d" % k]][ok], b[dh.F["FIELD_%d" % k]][ok]
        assert np.all(np.abs(x - y) <= 4e-6 * np.abs(y)), k
