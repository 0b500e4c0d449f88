"""GPU: every array of a mesh copied to the host in parts (2^18 triangles each
and a remainder).  FP64: positions, weights, cells, edge ids, interior bits and
interior vertex normals equal the oracle's bit for bit.  FP32: cells and edges
equal the FP64 mesh's, vertex normals are mesh_normals' floats, positions and
weights are the FP64 ones within rounding.  A copy also works after the
library was finalized."""
import numpy as np
import pytest

from contour3d_amd import api, fields

from test_gpu_mesh_copy import NAMES, copy
from test_gpu_parity import same_bits

pytestmark = pytest.mark.gpu

SHAPE, THR = (118, 112, 121), 0.1
PART = 2 ** 18


@pytest.fixture(scope="module")
def contours():
    f = fields.turbulence(SHAPE, kmax=29, seed=3)
    return [dict(field=f, threshold=THR, color=(1, 2, 3))]


def unpack_edges(e):
    return np.stack([e & 31, (e >> 5) & 31, (e >> 10) & 31], axis=1), ((e >> 15) & 1).astype(bool)


def test_fp64_arrays_equal_the_oracle(orc, contours):
    ref = orc.mesh(contours[0]["field"], THR)
    m = api.Mesh(contours)
    got = copy(m, NAMES)
    n = m.count(0)
    assert n > 2 * PART and n % PART
    edge, interior = unpack_edges(got["edges"])
    assert np.array_equal(got["cell"].astype(np.int64), ref["cell"])
    assert np.array_equal(edge, ref["edge"])
    assert np.array_equal(interior, ref["interior"].astype(bool))
    assert same_bits(got["pos"].reshape(-1), np.asarray(ref["pos"]).reshape(-1))
    assert same_bits(got["wfn"].reshape(n, 3), ref["area"][:, None] * ref["fn"])
    vn = got["vn"].reshape(n, 9)
    assert same_bits(vn[interior], np.asarray(ref["vn"]).reshape(n, 9)[interior])
    assert np.isnan(vn[~interior]).all()
    # the library finalized between build and copy
    api.finalize()
    again = copy(m, NAMES)
    m.free()
    for k in NAMES:
        assert np.array_equal(again[k], got[k], equal_nan=k == "vn"), k


def test_fp32_arrays_against_the_fp64_mesh(contours):
    import torch

    m64, m32 = api.Mesh(contours), api.Mesh(contours, precision=api.FP32)
    a, b = copy(m64, NAMES), copy(m32, NAMES)
    n = m32.count(0)
    assert np.array_equal(a["cell"], b["cell"])
    assert np.array_equal(a["edges"], b["edges"])
    out = torch.zeros((n, 9), dtype=torch.float32, device="cuda")
    m32.normals(0, out=out)
    assert same_bits(b["vn"], out.cpu().numpy().astype(np.float64))
    # positions lie in [-0.5, 0.5]: two coordinates, a quotient, a product and
    # a sum, each rounded once in FP32
    assert np.abs(a["pos"] - b["pos"]).max() <= 8 * 2.0 ** -24
    # a weight is the cross product of two edges of at most a cell's diagonal,
    # each off by two such errors per component
    diagonal = np.sqrt(3.0) / min(SHAPE)
    assert np.abs(a["wfn"] - b["wfn"]).max() <= 4 * diagonal * 16 * 2.0 ** -24
    m64.free()
    m32.free()
