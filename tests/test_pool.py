"""CPU: the bounded pool of freed meshes' device blocks
(contour3d_amd/csrc/c3d_pool.h) against a model (tests/pool/check_pool.cpp)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_pool_holds_what_it_should(tmp_path):
    exe = tmp_path / "check_pool"
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", os.path.join(ROOT, "contour3d_amd", "csrc"),
                    os.path.join(ROOT, "tests", "pool", "check_pool.cpp"), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.startswith("ok"), r.stdout
