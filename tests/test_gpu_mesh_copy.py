"""GPU: a mesh's triangles in host arrays, unpacked on the device in parts of
2^18 triangles: below, at several parts with a remainder, and any subset of
the arrays.  FP64 arrays equal the oracle's bit for bit; an FP32 mesh has the
same cells and edges, its positions and weights are floats, and subsets equal
the full copy."""
import ctypes as C

import numpy as np
import pytest

from contour3d_amd import api, fields

pytestmark = pytest.mark.gpu

NAMES = ("pos", "wfn", "vn", "cell", "edges")


def copy(mesh, want):
    n = mesh.count(0)
    room = dict(pos=np.full((n, 9), 7.0), wfn=np.full((n, 3), 7.0), vn=np.full((n, 9), 7.0),
                cell=np.full(n, 7, np.uint32), edges=np.full(n, 7, np.uint32))
    ptr = [room[k].ctypes.data if k in want else None for k in NAMES]
    assert api.lib().contour3d_amd_mesh_copy(mesh.handle, C.c_size_t(0), *ptr) == 0
    return {k: room[k] for k in want}


@pytest.mark.parametrize("shape, parts", [((14, 13, 12), 1), ((118, 112, 121), 2)])
def test_copy_in_parts(orc, shape, parts):
    f = fields.turbulence(shape, kmax=shape[0] // 4, seed=3)
    cont = [dict(field=f, threshold=0.1, color=(1, 2, 3))]
    ref = orc.mesh(f, 0.1)
    for precision in (api.FP64, api.FP32):
        m = api.Mesh(cont, precision=precision)
        try:
            n = m.count(0)
            assert parts == 1 or n > (parts - 1) * 2 ** 18 and n % 2 ** 18
            full = copy(m, NAMES)
            assert np.array_equal(full["cell"].astype(np.int64), np.asarray(ref["cell"]))
            if precision == api.FP64:
                assert np.array_equal(full["pos"].reshape(-1).view(np.uint64),
                                      np.ascontiguousarray(ref["pos"]).reshape(-1).view(np.uint64))
            else:
                for k in ("pos", "wfn"):
                    assert np.array_equal(full[k], full[k].astype(np.float32).astype(np.float64))
            inner = (full["edges"] >> 15) & 1 == 1
            assert inner.any() and not inner.all()
            length = np.linalg.norm(full["vn"].reshape(n, 3, 3)[inner], axis=2)
            assert np.nanmax(np.abs(length - 1)) < 1e-6
            for want in (("vn",), ("wfn", "edges"), ("pos", "cell"), ("cell",), ("pos", "vn")):
                part = copy(m, want)
                for k in want:
                    assert np.array_equal(part[k], full[k], equal_nan=k == "vn"), (precision, want, k)
        finally:
            m.free()
