"""The common-case Gauss-Newton kernels (see test_gpu_common_case.py) at the edges of what they take."""
import numpy as np
import pytest

import dice_amd as dh
from dice_amd import synth
import test_gpu_common_case as common
from test_gpu_common_case import CLOSE, EXACT, scene  # noqa: F401 (scene: the fixture)

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


@pytest.mark.parametrize("S,interp,dtype", [(5, dh.KEYS_FOURTH, np.float32), (31, dh.KEYS_FOURTH, np.uint16),
                                            (33, dh.BILINEAR, np.float32), (37, dh.KEYS_FOURTH, np.float32),
                                            (41, dh.KEYS_FOURTH, np.float32), (41, dh.BILINEAR, np.uint16)])
def test_inside(scene, S, interp, dtype):
    """Translation only, all subsets inside the image: one wave per subset, crews and the general kernel."""
    ctx, ref, de = scene
    if dtype == np.uint16:
        ref, de = [np.clip(np.round(np.maximum(i, 0) * 16), 0, 4095).astype(np.uint16) for i in (ref, de)]
    c = S // 2 + 6
    gx, gy = np.meshgrid(np.arange(c, common.W - c, 9), np.arange(c, common.H - c, 9))
    cx, cy = gx.ravel().astype(float), gy.ravel().astype(float)
    assert len(cx) > 1024
    p, q = params(interp), params(interp)
    q.initial_gamma_threshold = 1e9  # the general kernel
    wave = common.run(ctx, p, ref, de, cx, cy, S)
    finished = ctx.handover_counts()[0] < 0.05 * len(cx)
    few = np.arange(0, len(cx), 15)  # 15: the start values, which depend on the index, are those of the whole set
    crew = common.run(ctx, p, ref, de, cx[few], cy[few], S)
    general = common.run(ctx, q, ref, de, cx, cy, S)
    keep = (np.arange(len(few)) % 3 == 0) & (np.arange(len(few)) % 5 == 0)
    common.same(wave[:, few][:, keep], crew[:, keep])
    ok = general[dh.F["STATUS"]] != 5
    common.same(wave[:, ok], general[:, ok])
    assert finished


@pytest.mark.parametrize("S,interp,step", [(21, dh.KEYS_FOURTH, 4), (35, dh.KEYS_FOURTH, 4), (35, dh.BILINEAR, 3)])
def test_border_of_a_large_frame(scene, S, interp, step):
    """Enough subsets for the translation kernel although some reach the border, which it hands over."""
    ctx, ref, de = scene
    c = S // 2
    gx, gy = np.meshgrid(np.arange(c, common.W - c, step), np.arange(c, common.H - c, step))
    cx, cy = gx.ravel().astype(float), gy.ravel().astype(float)
    assert len(cx) > (5120 if interp == dh.KEYS_FOURTH else 10240)
    p, q = params(interp), params(interp)
    q.initial_gamma_threshold = 1e9
    a = common.run(ctx, p, ref, de, cx, cy, S)
    assert 0 < ctx.handover_counts()[0] < 0.2 * len(cx)
    general = common.run(ctx, q, ref, de, cx, cy, S)
    ok = general[dh.F["STATUS"]] != 5
    common.same(a[:, ok], general[:, ok])


def test_border_of_a_small_frame(scene):
    """Few subsets, some at the border: the general kernel takes them all."""
    ctx, ref, de = scene
    S = 21
    gx, gy = np.meshgrid(np.arange(10, common.W - 10, 23), np.arange(10, common.H - 10, 23))
    cx, cy = gx.ravel().astype(float), gy.ravel().astype(float)
    p, q = params(), params()
    q.initial_gamma_threshold = 1e9
    a = common.run(ctx, p, ref, de, cx, cy, S)
    assert ctx.handover_counts() == (0, 0, 0)
    general = common.run(ctx, q, ref, de, cx, cy, S)
    ok = general[dh.F["STATUS"]] != 5
    for name in EXACT + CLOSE:
        assert np.array_equal(a[dh.F[name]][ok], general[dh.F[name]][ok]), name


@pytest.mark.parametrize("step", [3, 45], ids=["wave", "crew"])
@pytest.mark.parametrize("interp", [dh.KEYS_FOURTH, dh.BILINEAR], ids=["keys", "bilinear"])
@pytest.mark.parametrize("u,v", [(7.3, -3.6), (-9.4, 12.2), (0.2, -6.7)])
def test_large_motion(u, v, interp, step):
    """A translation of more than 5 px: the unshifted subset lies outside the window that the uncertainty fields
    are formed from (in places in the image's last columns and rows, which count as 0 there), and the kernels
    still finish every subset themselves."""
    w, h, S = (340, 320, 35) if interp == dh.KEYS_FOURTH else (420, 400, 35)
    ref, de = images(w, h, u, v, 53)

    edge = 0 if step == 3 else 4  # crews: clear of the border before the motion too

    def centres(size, d):  # up to the border that the motion leads away from
        lo, hi = S // 2 + max(edge, int(7 - d)), size - 1 - S // 2 - max(edge, int(d + 7))
        return np.append(np.arange(lo, hi, step), hi)

    gx, gy = np.meshgrid(centres(w, u), centres(h, v))
    cx, cy = gx.ravel().astype(float), gy.ravel().astype(float)
    assert len(cx) > 5120 if step == 3 else len(cx) <= 1024
    f0 = dh.new_fields(cx, cy)
    f0[dh.F["DISP_X"]], f0[dh.F["DISP_Y"]] = round(u), round(v)
    p, q = params(interp), params(interp)
    q.initial_gamma_threshold = 1e9  # the general kernel
    with dh.Context(0) as ctx:
        a = run(ctx, p, ref, de, cx, cy, S, f0)
        assert ctx.pass_counts()[1] == 0 and ctx.handover_counts() == (0, 0, 0)
        # (the rule sends a border frame of this size to the translation kernel; crews have none here)
        assert len(cx) > (5120 if interp == dh.KEYS_FOURTH else 10240) or step == 45
        b = run(ctx, q, ref, de, cx, cy, S, f0)
    check(a, b)


@pytest.mark.parametrize("step", [6, 45], ids=["wave", "crew"])
@pytest.mark.parametrize("interp", [dh.KEYS_FOURTH, dh.BILINEAR], ids=["keys", "bilinear"])
def test_sub_images_at_offsets(interp, step):
    """Reference and deformed images cut out at different places, so that the unshifted pixel lies 11 and 7 px from
    where the subset is found."""
    w, h, S = 360, 340, 31
    full_ref, full_def = images(w, h, 0.4, -0.3, 57)
    ref, de = full_ref[9:, 20:], full_def[16:330, 31:350]
    gx, gy = np.meshgrid(np.arange(60, 300, step), np.arange(50, 290, step))
    cx, cy = gx.ravel().astype(float), gy.ravel().astype(float)
    f0 = dh.new_fields(cx, cy)
    p, q = params(interp), params(interp)
    q.initial_gamma_threshold = 1e9  # the general kernel
    with dh.Context(0) as ctx:
        out = []
        for k in (p, q):
            ctx.set_params(k)
            ctx.set_ref_image(np.ascontiguousarray(ref))
            ctx.set_def_image(np.ascontiguousarray(de))
            ctx.set_image_offsets(20, 9, 31, 16)
            ctx.set_subsets(cx, cy, S)
            out.append(ctx.correlate(f0.copy(), first_frame=False))
            if k is p:
                assert ctx.handover_counts() == (0, 0, 0)
    check(*out)
