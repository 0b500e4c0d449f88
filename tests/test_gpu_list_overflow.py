"""GPU: a frame whose fragment list overflows finds its ids by a pass over the
geometry instead (k_frame's id mode).  The list is made one entry long right
before each frame, eager and replayed from a graph, in both forms: waves
reserve 64 entries at a time, so every frame that draws anything overflows it.
The allocation-free frame's list of 3 * 2^20 entries overflows when several
objects of one surface cover enough pixels: each of them puts at least one
fragment per covered pixel into the list, since equal depths all pass the
z-test."""
import numpy as np
import pytest

from contour3d_amd import api, fields

from test_gpu_batch import uneven_batch
from test_gpu_parity import same_bits, view_for
from test_zz_no_alloc import noalloc

pytestmark = pytest.mark.gpu

FORMS = pytest.mark.parametrize("precision", [api.FP64, api.FP32], ids=["fp64", "fp32"])
SCRATCH_LIST = 3 << 20  # entries of the allocation-free frame's list


def batch():
    """A batch with depths, lines, shared and tied surfaces."""
    images = [dict(im, want_depth=True) for im in uneven_batch()]
    f = fields.blobs((9, 9, 9), seed=5)
    tied = [dict(field=f, threshold=0.45, color=(10 * q, 200 - 10 * q, 40)) for q in range(6)]
    images.append(dict(view_for(120, 90), contours=tied, want_depth=True))
    return images


def same(got, ref):
    for q, (g, r) in enumerate(zip(got, ref)):
        assert np.array_equal(g[0], r[0]), q
        assert same_bits(g[1], r[1]), q


@FORMS
def test_eager_frames(orc, precision):
    images = batch()
    ref = api.execute_batch(images, precision=precision)
    try:
        for _ in range(2):
            api.tune(api.TUNE_FRAG_CAPACITY, 1)
            same(api.execute_batch(images, precision=precision), ref)
        # the list has grown: the same frame through it
        same(api.execute_batch(images, precision=precision), ref)
    finally:
        api.tune(api.TUNE_FRAG_CAPACITY, 0)
    if precision == api.FP64:
        im = images[-1]
        rgb, depth = orc.execute(im["camera"], im["light"], im["size"], im["center"], im["local"], im["bg"],
                                 im["contours"])
        assert (depth > -1e300).any()
        same(ref[-1:], [(rgb, depth)])


@FORMS
def test_captured_frames(precision):
    import torch

    images = batch()
    ref = api.execute_batch(images, precision=precision)
    try:
        api.tune(api.TUNE_GRAPHS, 1)
        api.execute_batch(images, precision=precision)
        for _ in range(3):
            # a list of one entry: the next call captures with it, and its
            # replay takes the id pass; the call after replays the grown one
            api.tune(api.TUNE_FRAG_CAPACITY, 1)
            same(api.execute_batch(images, precision=precision), ref)
            torch.cuda.synchronize()
            same(api.execute_batch(images, precision=precision), ref)
            same(api.execute_batch(images, precision=precision), ref)
    finally:
        api.tune(api.TUNE_FRAG_CAPACITY, 0)
        api.tune(api.TUNE_GRAPHS, 0)


@FORMS
def test_allocation_free_frames(precision):
    import torch

    assert api.lib().contour3d_amd_init(0) == 0
    # a sphere around the camera's axis that fills most of the image
    n = 40
    g = fields.uniform_grid(n)
    z, y, x = np.meshgrid(g, g, g, indexing="ij")
    f = torch.from_numpy(np.sqrt(x * x + y * y + z * z)).cuda()
    contours = [dict(field=f, grids=(g, g, g), threshold=0.45, color=(40 * q, 250 - 40 * q, 90)) for q in range(6)]
    v = fields.sphere_view(0.3, 0.7, 1900, 1080)
    v["local"] = tuple(tuple(0.5 * c for c in w) for w in v["local"])
    args = (v["camera"], v["light"], v["size"], v["center"], v["local"], v["bg"], contours)
    ref_rgb, ref_depth = api.execute_rgb(*args, precision=precision, want_depth=True)
    assert int((ref_depth > -1e300).sum()) * len(contours) > SCRATCH_LIST
    rgb = torch.zeros((1080, 1900, 3), dtype=torch.uint8, device="cuda")
    depth = torch.zeros((1080, 1900), dtype=torch.float64, device="cuda")
    for _ in range(2):
        rgb.zero_()
        depth.zero_()
        torch.cuda.synchronize()
        assert noalloc(v, contours, [], precision, rgb, depth) == 0
        torch.cuda.synchronize()
        assert np.array_equal(rgb.cpu().numpy(), ref_rgb)
        assert same_bits(depth.cpu().numpy(), ref_depth)
