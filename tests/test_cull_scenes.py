"""CPU: the rule of contour3d_amd/csrc/c3d_cull.h on whole scenes moved away
from the origin, scaled and stretched, and on images of extreme proportions
(tests/cull/check_cull_scenes.cpp): no fragment of a cell that the rule calls
regular may leave its brick's pixel box or come nearer than its bound, down
to lattice spacings of a unit in the last place of the coordinates."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = tmp_path_factory.mktemp("cull") / "check_cull_scenes"
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-I", os.path.join(ROOT, "contour3d_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cull", "check_cull_scenes.cpp"), "-o", str(exe)], check=True)

    def run(*scenes):
        r = subprocess.run([str(exe), "1", "20000", *scenes], capture_output=True, text=True, timeout=300)
        print(r.stdout)
        assert r.returncode == 0, r.stdout
        return {m[1]: (int(m[2]), int(m[3]))
                for m in re.finditer(r"^(\S+): .* (\d+) cut cells, (\d+) regular", r.stdout, re.M)}

    return run


def test_scenes_far_from_the_origin(check):
    got = check("shift:0", "shift:6", "shift:8", "shift:10", "shift:11", "shift:11.3", "shift:11.6", "shift:12",
                "shift:13", "shift:14", "shift:15")
    # of use near the origin (the smallest cells of these scenes fall below
    # the bound there, too)
    assert got["shift:0"][1] > 0.4 * got["shift:0"][0] > 0


def test_images_of_extreme_proportions(check):
    check("wide:8", "wide:14")


def test_scenes_of_any_length_scale(check):
    """A power of two changes no rounding, so the same cells are regular at
    every scale; past the ends of the range that the rule takes, none are."""
    got = check("scale:0", "scale:20", "scale:40", "scale:54", "scale:62", "scale:90", "scale:120", "scale:200",
                "scale:-60")
    assert got["scale:0"][1] > 0
    for s in ("scale:20", "scale:40", "scale:54", "scale:62", "scale:90"):
        assert got[s] == got["scale:0"], s
    assert got["scale:120"][1] == got["scale:200"][1] == got["scale:-60"][1] == 0


def test_cells_of_extreme_proportions(check):
    check("stretch:-10", "stretch:-40", "stretch:-80", "stretch:-120", "stretch:-149", "stretch:2")
