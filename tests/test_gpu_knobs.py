"""GPU: the brick knobs (rows of cells and planes of every brick of a frame, of
every tile of a mesh) and the workgroups that draw change no bit, below, at and
beyond the sizes of a brick, alone and together, eager and captured."""
import numpy as np
import pytest

from contour3d_amd import api, fields

from test_gpu_batch import uneven_batch
from test_gpu_parity import same_bits, view_for

pytestmark = pytest.mark.gpu

# rows, planes, workgroups
SETTINGS = [(1, 0, 0), (3, 0, 0), (8, 0, 0), (9, 0, 0), (0, 1, 0), (0, 3, 0), (0, 8, 0), (0, 9, 0), (0, 16, 8),
            (1, 1, 0), (2, 5, 8), (7, 2, 1024), (4096, 4096, 1)]


def set_knobs(rows, planes, grid):
    api.tune(api.TUNE_TESS_ROWS, rows)
    api.tune(api.TUNE_TESS_ZPLANES, planes)
    api.tune(api.TUNE_TESS_GRID, grid)


def images():
    # beside the small images: a long row, a close-up, and two images of a pass
    out = [dict(im, want_depth=True) for im in uneven_batch()]
    f = fields.turbulence((37, 35, 150), kmax=9, seed=12)
    cont = [dict(field=f, threshold=t, color=(90, 200, 40 * q)) for q, t in enumerate((-0.8, -0.2, 0.1, 0.5, 1.0))]
    for zoom in (1.0, 0.2):
        v = view_for(110, 90)
        v["local"] = tuple(tuple(zoom * c for c in w) for w in v["local"])
        out.append(dict(v, contours=cont, want_depth=True))
    return out


@pytest.mark.parametrize("precision", [api.FP64, api.FP32], ids=["fp64", "fp32"])
def test_knobs_change_no_frame(precision):
    batch = images()
    ref = api.execute_batch(batch, precision=precision)
    assert all((d > -1e300).any() for _, d in ref)
    try:
        for graphs in (0, 1):
            for setting in SETTINGS:
                set_knobs(*setting)
                api.tune(api.TUNE_GRAPHS, graphs)
                for _ in range(1 + graphs):
                    for q, (rgb, depth) in enumerate(api.execute_batch(batch, precision=precision)):
                        assert np.array_equal(rgb, ref[q][0]), (setting, graphs, q)
                        assert same_bits(depth, ref[q][1]), (setting, graphs, q)
    finally:
        api.tune(api.TUNE_GRAPHS, 0)
        set_knobs(0, 0, 0)


@pytest.mark.parametrize("precision", [api.FP64, api.FP32], ids=["fp64", "fp32"])
def test_knobs_change_no_mesh(precision):
    cont = images()[-1]["contours"][:2]

    def arrays():
        m = api.Mesh(cont, precision=precision)
        got = [m.copy(o) for o in range(len(cont))]
        m.free()
        return got

    ref = arrays()
    try:
        for setting in SETTINGS:
            set_knobs(*setting)
            for a, b in zip(arrays(), ref):
                for k in b:
                    assert np.array_equal(a[k], b[k], equal_nan=b[k].dtype.kind == "f"), (setting, k)
    finally:
        set_knobs(0, 0, 0)
