"""GPU: the divisions by constants of a view as frames make them, with the
reciprocals that the host rounds once (set_recips), equal the compiler's
divisions bit for bit in both forms: tests/div_check/check_div_view, built by
__graft_entry__.build()."""
import os
import subprocess

import pytest

pytestmark = pytest.mark.gpu

EXE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "div_check", "check_div_view")


def test_divisions_by_view_constants():
    assert os.path.exists(EXE), "build first: python -c 'import __graft_entry__ as g; g.build()'"
    r = subprocess.run([EXE], capture_output=True, text=True, timeout=120)
    print(r.stdout)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "fp64: " in r.stdout and "fp32: " in r.stdout and r.stdout.count("mismatches 0") == 2
