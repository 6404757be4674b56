"""The rule that picks a common-case Gauss-Newton kernel (dice_amd/csrc/dice_dispatch.h), compiled for the host
and swept over subset sizes, counts and LDS slots, and the cell size of VSG radius windows there."""
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
NONE, LEAN, TRANS, CREW = range(4)


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("dispatch") / "dispatch")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-o", exe,
                           os.path.join(ROOT, "tests", "cpp", "dispatch.cpp")])

    def ask(rows):
        text = "\n".join(" ".join(str(int(v)) for v in r) for r in rows)
        out = subprocess.run([exe], input=text, capture_output=True, text=True, timeout=60, check=True).stdout
        return np.array(out.split(), dtype=np.int64).reshape(len(rows), -1)

    ask.exe = exe
    return ask


def sweep(ns=(1, 255, 1024, 1025, 5000), sizes=range(1, 100), slots=(2560, 2704, 2812, 5184, 6400, 16000)):
    return [(n, S, affine, slot, keys, unc, listed, 0) for n in ns for S in sizes for affine in (0, 1) for slot in slots
            for keys in (0, 1) for unc in (0, 1) for listed in (0, 1)]


def test_the_translation_kernels_have_a_lane_per_column(rule):
    """A subset of even size S is S + 1 pixels wide: size 64 has 65 columns, one more than a wave has lanes."""
    rows = sweep()
    for (n, S, affine, slot, *_), (kernel, wave_lds, crew_lds) in zip(rows, rule(rows)):
        if kernel in (TRANS, CREW):
            assert S // 2 * 2 + 1 <= 64, (n, S, affine, slot)
            assert (crew_lds if kernel == CREW else wave_lds) <= 62 * 1024, (n, S, affine, slot)
        assert kernel != TRANS or not affine, (n, S, affine, slot)
        assert kernel != LEAN or affine, (n, S, affine, slot)


def test_no_launch_whose_subsets_are_all_handed_over(rule):
    """The window of a subset at a translation of (0.5, 0.5) px and, with uncertainty fields, the general kernel's
    window of them (3 px before and 4 px after the box), counted pixel by pixel, against the slot less the
    per-subset constants (104 floats)."""
    rows = sweep()
    for (n, S, affine, slot, keys, unc, *_), (kernel, _, _) in zip(rows, rule(rows)):
        h = S // 2
        need = np.floor(h + 0.5) + (3 if keys else 1) - (np.floor(-h + 0.5) - (2 if keys else 0)) + 1
        if unc:
            need = max(need, 2 * h + (6 if affine else 8))
        fits = need ** 2 <= slot - 104
        if kernel in (TRANS, CREW):
            assert fits, (n, S, affine, slot, keys, unc)
        if not affine and fits and S <= 41 and n > 1024:
            assert kernel == TRANS, (n, S, affine, slot, keys, unc)


@pytest.mark.parametrize("S,affine,listed,most", [(8, 1, 0, 256), (9, 1, 0, 256), (10, 1, 0, 768), (31, 1, 0, 768),
                                                  (41, 1, 0, 768), (9, 1, 1, 1024), (31, 1, 1, 1024),
                                                  (9, 0, 0, 1024), (41, 0, 0, 1024), (31, 0, 1, 1024)])
def test_number_of_subsets_that_crews_take(rule, S, affine, listed, most):
    """One crew per CU (of 256) for small six-parameter subsets, three for larger ones, four for translation only
    and for lists."""
    rows = [(n, S, affine, 2560, 1, 1, listed, 0) for n in (1, most, most + 1, 1 << 17)]
    many = LEAN if affine else TRANS
    assert rule(rows)[:, 0].tolist() == [CREW, CREW, many, many]


LEFT, RIGHT, TOP, BOTTOM = 1, 2, 4, 8


@pytest.mark.parametrize("keys,most", [(1, 5120), (0, 10240)])
def test_border_subsets_of_small_frames_stay_with_the_others(rule, keys, most):
    """Translation only with a subset at the border: the general kernel takes the whole frame up to a size;
    six-parameter frames (whose lean kernel there always was) as without one."""
    for S in (9, 35, 41):
        for border in range(1, 16):
            rows = [(n, S, 0, 2560, keys, 1, 0, border) for n in (1, 1024, 1025, most, most + 1)]
            assert rule(rows)[:, 0].tolist() == [NONE] * 4 + [TRANS]
            for listed in (0, 1):
                rows = [[(n, S, 1, 2560, keys, 1, listed, b) for n in (1, 300, 5000)] for b in (0, border)]
                assert np.array_equal(rule(rows[0]), rule(rows[1])) and (rule(rows[1])[:, 0] != NONE).all()


def test_border_of_a_chain(rule):
    """Rounds of neighbour initialization, translation only: the general kernel where the chain's columns reach the
    border at both ends or three sides do, crews elsewhere."""
    for border in range(16):
        ends = border & (TOP | BOTTOM) == TOP | BOTTOM
        three = bin(border).count("1") >= 3
        got = rule([(n, 27, 0, 2560, 1, 1, 1, border) for n in (1, 361, 1024)])[:, 0].tolist()
        assert got == [NONE if ends or three else CREW] * 3, border


@pytest.mark.parametrize("radius", [1.0, 7.0, 20.0, 60.0, 300.0])
@pytest.mark.parametrize("extent,n", [(60.0, 30000), (445.0, 8000), (1900.0, 445), (1900.0, 155236), (4096.0, 7)])
def test_vsg_cells_between_a_quarter_of_the_radius_and_the_radius(rule, radius, extent, n):
    """Four rings of cells reach the radius, and no cell is wider than it however few subsets there are for their
    bounds (the one subset per cell on average in between)."""
    slack = 0.05
    cell = float(subprocess.check_output([rule.exe, str(radius), str(slack), str(extent ** 2), str(n)]))
    assert 4.0 * cell >= radius + 4.0 * slack - 1e-9
    assert cell <= max(radius, (radius + 4.0 * slack) / 4.0)
    if radius / 2 < extent / n ** 0.5 < radius:
        assert abs(cell - extent / n ** 0.5) < 1e-9
