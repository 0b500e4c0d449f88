"""The resolve's pixel tiles (32 x 8) at their edges: images of one pixel, one
row, one column, one pixel more and less than a tile, and a batch of them, on
a far view (every pixel its own triangle) and a close-up (one triangle over
many tiles), against the oracle bit for bit in FP64 and, in FP32, equal to the
stored mesh's render (an independent raster path)."""
import numpy as np
import pytest

from contour3d_amd import api, fields

pytestmark = pytest.mark.gpu

SIZES = [(1, 1), (32, 8), (33, 9), (31, 7), (1, 70), (257, 1), (200, 130)]


def scene(n, zoom):
    f = fields.turbulence((n, n + 3, n - 2), kmax=5, seed=3)
    contours = [dict(field=f, threshold=t, color=c) for t, c in
                ((-0.7, (250, 40, 10)), (0.0, (30, 200, 90)), (0.8, (60, 90, 255)))]
    return contours, zoom


def view_at(W, H, zoom):
    v = fields.sphere_view(0.4, 0.9, W, H)
    v["local"] = tuple(tuple(zoom * c for c in w) for w in v["local"])
    return v


@pytest.mark.parametrize("n, zoom", [(40, 1.0), (14, 0.08)])
def test_tile_edges_match_the_oracle(orc, n, zoom):
    contours, zoom = scene(n, zoom)
    images, refs = [], []
    for W, H in SIZES:
        v = view_at(W, H, zoom)
        ref, dep = orc.execute(v["camera"], v["light"], v["size"], v["center"], v["local"], v["bg"], contours)[:2]
        rgb, d = api.execute_rgb(v["camera"], v["light"], v["size"], v["center"], v["local"], v["bg"], contours,
                                 want_depth=True)
        assert np.array_equal(rgb, ref), (W, H)
        assert np.array_equal(d.view(np.uint64), dep.view(np.uint64)), (W, H)
        images.append(dict(camera=v["camera"], light=v["light"], size=v["size"], center=v["center"],
                           local=v["local"], bg=v["bg"], contours=contours))
        refs.append(ref)
    for (rgb, _), ref in zip(api.execute_batch(images), refs):
        assert np.array_equal(rgb, ref)


@pytest.mark.parametrize("precision", [api.FP64, api.FP32])
@pytest.mark.parametrize("n, zoom", [(40, 1.0), (14, 0.08)])
def test_tile_edges_match_the_stored_mesh(n, zoom, precision):
    contours, zoom = scene(n, zoom)
    mesh = api.Mesh(contours, precision=precision)
    for W, H in SIZES:
        v = view_at(W, H, zoom)
        a = api.execute_rgb(v["camera"], v["light"], v["size"], v["center"], v["local"], v["bg"], contours,
                            precision=precision, want_depth=True)
        b = mesh.render(v["camera"], v["light"], v["size"], v["center"], v["local"], v["bg"], want_depth=True)
        assert np.array_equal(a[0], b[0]) and np.array_equal(a[1].view(np.uint64), b[1].view(np.uint64)), (W, H)
    mesh.free()
