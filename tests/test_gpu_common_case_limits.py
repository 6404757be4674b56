"""The common-case Gauss-Newton kernels (see test_gpu_common_case.py) at the edges of what they take."""
import numpy as np
import pytest

import dice_amd as dh
from dice_amd import synth
from test_gpu_common_case import CLOSE, EXACT

pytestmark = pytest.mark.gpu


def images(w, h, u, v, seed):
    sp = synth.Speckle(w, h, seed=seed)
    return sp.frame(None), sp.frame(synth.affine_field(u, v, 0.0, 0.0, 0.0, 0.0), noise_sigma=1.0, noise_seed=seed + 1)


def params(interp=dh.KEYS_FOURTH):
    p = dh.default_params()
    p.optimization_method = dh.GRADIENT_BASED
    p.interpolation_method = interp
    return p


def run(ctx, p, ref, de, cx, cy, S, f0, mode=dh.MODE_BATCHED):
    ctx.set_params(p)
    ctx.set_ref_image(ref)
    ctx.set_def_image(de)
    ctx.set_subsets(cx, cy, S)
    return ctx.correlate(f0.copy(), mode=mode, first_frame=False)


def check(a, general):
    """Against the general kernel: equal bit for bit, sums in another order to float rounding."""
    assert np.isin(a[dh.F["STATUS"]], dh.CONVERGED_STATUSES).mean() > 0.9
    for name in EXACT:
        assert np.array_equal(a[dh.F[name]], general[dh.F[name]]), name
    for name in CLOSE:
        x, y = a[dh.F[name]], general[dh.F[name]]
        assert np.abs(x - y).max() <= 2e-5 * max(np.abs(y).max(), 1e-3), name


@pytest.mark.parametrize("interp", [dh.KEYS_FOURTH, dh.BILINEAR], ids=["keys", "bilinear"])
@pytest.mark.parametrize("S", [62, 63, 64])
def test_widest_subsets(S, interp):
    """With a slot that holds their window: 63 columns fill the wave (sizes 62 and 63), size 64 has 65 columns."""
    ref, de = images(420, 300, 0.37, -0.21, 51)
    gx, gy = np.meshgrid(np.arange(40, 380, 9), np.arange(40, 260, 7))
    cx, cy = gx.ravel().astype(float), gy.ravel().astype(float)
    assert len(cx) > 1024
    f0 = dh.new_fields(cx, cy)
    p, q = params(interp), params(interp)
    q.initial_gamma_threshold = 1e9  # the general kernel
    with dh.Context(0) as ctx:
        ctx.set_launch_shape(1, 8, 6400)
        a = run(ctx, p, ref, de, cx, cy, S, f0)
        b = run(ctx, q, ref, de, cx, cy, S, f0)
    check(a, b)


@pytest.mark.parametrize("step", [6, 45], ids=["wave", "crew"])
@pytest.mark.parametrize("interp", [dh.KEYS_FOURTH, dh.BILINEAR], ids=["keys", "bilinear"])
@pytest.mark.parametrize("u,v", [(7.3, -3.6), (-9.4, 12.2), (0.2, -6.7)])
def test_large_motion(u, v, interp, step):
    """A translation of more than 5 px: the unshifted subset lies outside the window that the uncertainty fields
    are formed from (in places in the image's last columns and rows, which count as 0 there), and the kernels
    still finish every subset themselves."""
    w, h, S = 340, 320, 35
    ref, de = images(w, h, u, v, 53)

    def centres(size, d):  # up to the border that the motion leads away from
        return np.arange(S // 2 + max(0, int(7 - d)), size - S // 2 - max(0, int(d + 7)), step)

    gx, gy = np.meshgrid(centres(w, u), centres(h, v)[::-1])
    gx[:, -1] = w - 1 - S // 2 - max(0, int(u + 7))
    gy[0] = h - 1 - S // 2 - max(0, int(v + 7))
    cx, cy = gx.ravel().astype(float), gy.ravel().astype(float)
    assert (len(cx) > 1024) == (step == 6)
    f0 = dh.new_fields(cx, cy)
    f0[dh.F["DISP_X"]], f0[dh.F["DISP_Y"]] = round(u), round(v)
    p, q = params(interp), params(interp)
    q.initial_gamma_threshold = 1e9  # the general kernel
    with dh.Context(0) as ctx:
        a = run(ctx, p, ref, de, cx, cy, S, f0)
        assert ctx.pass_counts()[1] == 0 and ctx.handover_counts() == (0, 0, 0)
        b = run(ctx, q, ref, de, cx, cy, S, f0)
    check(a, b)
