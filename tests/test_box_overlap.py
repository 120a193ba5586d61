"""How many instance boxes a point of the scene lies in (box_overlap.h), which decides whether rays over
instances are sorted: against closed forms, whatever the number, flatness and distance of the boxes."""
import os
import subprocess

import numpy as np
import pytest

from luisacompute_amd import build

PROGRAM = r"""
#include "box_overlap.h"
#include <cstdio>
#include <vector>
int main() {
    std::vector<float> b;
    float v;
    while (std::scanf("%f", &v) == 1) b.push_back(v);
    std::printf("%.9g\n", lchip::box_overlap(b.data(), (uint32_t)(b.size() / 8)));
}
"""
FAR = 3e38  # where instances without geometry are put


@pytest.fixture(scope="module")
def overlap(tmp_path_factory):
    at = tmp_path_factory.mktemp("overlap")
    (at / "overlap.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "-I", build.CSRC, str(at / "overlap.cpp"), "-o",
                    str(at / "overlap")], check=True)

    def run(lo, hi):
        b = np.zeros((len(lo), 8), np.float32)
        b[:, :3], b[:, 4:7] = lo, hi
        text = " ".join("%.9g" % x for x in b.reshape(-1))
        return float(subprocess.run([str(at / "overlap")], input=text, check=True, capture_output=True, text=True).stdout)

    return run


def _cubes(centres, half):
    c, h = np.asarray(centres, float), np.broadcast_to(np.asarray(half, float).reshape(-1, 1), (len(centres), 3))
    return c - h, c + h


@pytest.mark.parametrize("far", (0, 1, 20))
@pytest.mark.parametrize("copies", (2, 3, 8))
def test_overlapping_scenes_with_distant_instances(overlap, copies, far):
    """Copies of one box overlap `copies` times; small instances far away do not change that."""
    centres = [[50.0, 50.0, 50.0]] * copies + [[1000.0 + 10 * k, -500.0, 2000.0] for k in range(far)]
    assert overlap(*_cubes(centres, [50.0] * copies + [1.0] * far)) == pytest.approx(copies)


@pytest.mark.parametrize("side", (2, 4, 10))
def test_instances_side_by_side(overlap, side):
    grid = np.stack(np.meshgrid(*[np.arange(side)] * 3), -1).reshape(-1, 3) * 10.0
    around = (10.0 * (side - 1) + 9.8) ** 3
    assert overlap(*_cubes(grid, 4.9)) == pytest.approx(side ** 3 * 9.8 ** 3 / around, rel=1e-5)


def test_partial_overlap(overlap):
    """Two boxes that share half of each: 2 volumes over 1.5."""
    assert overlap(*_cubes([[0, 0, 0], [5, 0, 0]], 5.0)) == pytest.approx(2 / 1.5)


def test_scattered_groups(overlap):
    """Groups of overlapping boxes that lie apart are no overlapping scene, also when there are only two."""
    rng = np.random.default_rng(5)
    for groups in (2, 100):
        at = np.concatenate([[[0, 0, 0], [100, 100, 100]], rng.uniform(0, 100, (groups - 2, 3))]).repeat(3, axis=0)
        want = 3 * groups * 6.0 ** 3 / 106.0 ** 3
        assert overlap(*_cubes(at, 3.0)) == pytest.approx(want, rel=1e-5)


def test_flat_boxes(overlap):
    """Boxes flat but for the padding every instance box has: as their other extents overlap."""
    pad = np.array([0, 0, 1e-5])
    lo, hi = np.zeros((3, 3)), np.array([[10, 10, 0]] * 3, float)
    assert overlap(lo - pad, hi + pad) == pytest.approx(3.0)
    apart = np.array([[0, 0, 0], [20, 0, 0], [40, 0, 0]], float)
    assert overlap(lo + apart - pad, hi + apart + pad) == pytest.approx(0.6)


def test_boxes_without_a_volume(overlap):
    """No geometry, or no finite size: such boxes count nothing, and alone they give no overlap."""
    none = np.full((2, 3), FAR)
    assert overlap(none, none) == 0.0
    lo, hi = _cubes([[0, 0, 0]] * 2, 1.0)
    assert overlap(np.concatenate([lo, none]), np.concatenate([hi, none])) == pytest.approx(2.0)
    for bad in (np.nan, np.inf):
        odd = np.full((1, 3), bad)
        assert overlap(np.concatenate([odd, lo]), np.concatenate([odd, hi])) == pytest.approx(2.0)
