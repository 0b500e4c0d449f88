"""CPU: the bricks a frame's tessellation walks (contour3d_amd/csrc/c3d_bricks.h,
the header the device kernels use): tests/bricks/check_bricks.cpp visits
every cell of a lattice through the XCD lists, groups, bricks and lanes, for
lattices around the brick and group sizes, flat and one-cell axes, long rows,
the row and plane knobs, and bricks of 8, 4 and 2 columns a side."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

LATTICES = [
    (1, 1, 1, 0, 8, 1), (1, 1, 300, 0, 8, 2), (500, 1, 1, 0, 4, 1), (1, 700, 2, 0, 1, 1), (8, 8, 8, 0, 8, 1),
    (9, 7, 17, 0, 8, 1), (31, 33, 32, 0, 8, 2), (63, 65, 64, 0, 2, 1), (300, 186, 22, 0, 8, 2), (127, 127, 127, 0, 4, 2),
    (40, 41, 42, 1, 1, 1), (17, 90, 5, 3, 100, 1), (2500, 3, 4, 0, 8, 1), (7, 2500, 3, 0, 5, 2),
]


def test_bricks_visit_every_cell_once(tmp_path):
    exe = tmp_path / "check_bricks"
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", os.path.join(ROOT, "contour3d_amd", "csrc"),
                    os.path.join(ROOT, "tests", "bricks", "check_bricks.cpp"), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)] + [str(v) for lat in LATTICES for v in lat], capture_output=True, text=True,
                       timeout=300)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
    assert r.stdout.count("ok ") == 3 * len(LATTICES)
