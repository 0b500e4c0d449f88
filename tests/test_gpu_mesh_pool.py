"""Meshes freed and built again take the freed ones' device blocks: meshes of
changing size and form, alive together and freed out of order, hold the same
triangles and normals as the first build of each, and finalize gives the
blocks back."""
import numpy as np
import pytest

from contour3d_amd import api, fields

pytestmark = pytest.mark.gpu


def test_reused_blocks_hold_the_same_meshes():
    import torch

    shapes = [(20, 24, 28), (40, 33, 37), (9, 60, 14)]
    contours = [[dict(field=fields.turbulence(s, kmax=4, seed=q), threshold=t, color=(9, 9, 9)) for t in (-0.3, 0.4)]
                for q, s in enumerate(shapes)]
    jobs = [(c, p) for c in contours for p in (api.FP64, api.FP32)]
    api.finalize()
    first = []
    for c, p in jobs:
        m = api.Mesh(c, precision=p)
        first.append([m.copy(o) for o in range(2)])
        m.free()
    order = np.random.default_rng(5)
    for _ in range(3):
        meshes = [api.Mesh(c, precision=p) for c, p in jobs]
        for q in order.permutation(len(meshes)):
            for o in range(2):
                got = meshes[q].copy(o)
                for k, a in first[q][o].items():
                    assert np.array_equal(a, got[k], equal_nan=a.dtype.kind == "f"), (q, o, k)
            meshes[q].free()
    api.finalize()
    torch.cuda.synchronize()
    m = api.Mesh(*jobs[0])
    assert np.array_equal(m.copy(0)["pos"], first[0][0]["pos"])
    m.free()
