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
