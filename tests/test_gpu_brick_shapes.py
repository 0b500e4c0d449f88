"""GPU: a frame chooses the shape of its bricks by the work of its view, so the
same field is drawn with bricks of 8 x 8 x 8 down to 2 x 2 x 1 cells as the
camera closes in.  Image and depths must stay the oracle's, bit for bit, from
far away to deep inside, for one field and for a batch of fields of uneven
sizes that share one launch."""
import numpy as np
import pytest

from contour3d_amd import api, fields

pytestmark = pytest.mark.gpu


def scene(n, nthr=2, shift=0.0):
    gx, gy, gz = [(np.arange(m) - (m - 1) / 2) / max(n) for m in n]
    z, y, x = np.meshgrid(gz, gy, gx, indexing="ij")
    f = np.ascontiguousarray(np.sin(19 * x + shift) * np.cos(17 * y) + np.sin(23 * z + x))
    thr = (-0.4, 0.1, 0.3, 0.6, 0.9)[:nthr]
    return [dict(field=f, grids=(gx, gy, gz), threshold=t, color=(250 - 40 * q, 60 + 30 * q, 90)) for q, t in enumerate(thr)]


def view(zoom, W, H, azimuth=0.7):
    v = fields.sphere_view(0.4, azimuth, W, H)
    v["local"] = tuple(tuple(zoom * c for c in w) for w in v["local"])
    return v


def args(v):
    return v["camera"], v["light"], v["size"], v["center"], v["local"], v["bg"]


@pytest.mark.parametrize("zoom", [3.0, 1.0, 0.3, 0.05])
@pytest.mark.parametrize("n, nthr", [((20, 17, 23), 1), ((49, 65, 33), 5), ((130, 31, 66), 2)])
def test_every_zoom_is_the_oracles(orc, n, nthr, zoom):
    contours, v = scene(n, nthr), view(zoom, 97, 71)
    ref, dep = orc.execute(*args(v), contours)[:2]
    rgb, d = api.execute_rgb(*args(v), contours, want_depth=True)
    assert np.array_equal(d.view(np.uint64), dep.view(np.uint64))
    assert np.array_equal(rgb, ref)


def test_uneven_fields_share_a_launch(orc):
    sizes = [(9, 9, 9), (33, 40, 21), (70, 64, 66)]
    images = []
    for q, n in enumerate(sizes):
        v = view((1.0, 0.2, 0.5)[q], 64 + 9 * q, 48, 0.3 + q)
        images.append((v, scene(n, 1 + q, 0.2 * q)))
    ims = []
    for v, contours in images:
        W, H = v["size"]
        ims.append(dict(camera=v["camera"], light=v["light"], size=v["size"], center=v["center"], local=v["local"],
                        bg=v["bg"], contours=contours, rgb=np.zeros((H, W, 3), np.uint8)))
    api.execute_batch(ims)
    for (v, contours), im in zip(images, ims):
        assert np.array_equal(im["rgb"], orc.execute(*args(v), contours)[0])
