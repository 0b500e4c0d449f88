"""CPU: the arithmetic that stands in for divisions by view constants and for
the reference's pixel box (contour3d_amd/csrc/c3d_geom.h, the header the
device kernels use).  tests/view_math/check_view_math.cpp compares pixel
centres and FP32 quotients with the divisions bit for bit, over whole small
images, random columns of images up to 2^31 wide, any bit patterns, values
near the subnormals, and checks that the box of pixel_box lies in the
reference's and holds every pixel that the coverage test accepts."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "contour3d_amd", "csrc")
SRC = os.path.join(ROOT, "tests", "view_math", "check_view_math.cpp")


def build(out, include):
    exe = out / "check_view_math"
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-I", str(include), "-I", CSRC, SRC, "-o",
                    str(exe)], check=True)
    return str(exe)


@pytest.mark.parametrize("seed", [1, 2])
def test_view_math_equals_the_divisions_and_boxes(tmp_path, seed):
    r = subprocess.run([build(tmp_path, CSRC), str(seed), "200000"], capture_output=True, text=True, timeout=300)
    print(r.stdout)
    assert r.returncode == 0, r.stdout


@pytest.mark.parametrize("line, wrong", [
    ("return __builtin_fma(__builtin_fma(-extent, q, a), rb, q);", "return q;"),
    ("float q = float(double(a) * rb);", "float q = a * float(rb);"),
    ("const R M = (R(5.8e-8) * emax + R(12) * g * D * e2 * fabs(ainv)) * R(1.00000095367431640625) + "
     "R(16) * eps * qmax;", "const R M = R(0);"),
])
def test_check_sees_a_planted_mistake(tmp_path, line, wrong):
    hdr = open(os.path.join(CSRC, "c3d_geom.h")).read()
    assert hdr.count(line) == 1
    inc = tmp_path / "inc"
    inc.mkdir()
    (inc / "c3d_geom.h").write_text(hdr.replace(line, wrong))
    r = subprocess.run([build(tmp_path, inc), "1", "100000"], capture_output=True, text=True, timeout=300)
    assert r.returncode == 1, r.stdout
