"""GPU: the pool of freed meshes' device blocks gives its memory back: a mesh
freed after finalize does not enter it (nothing would take it out again), and
a device allocation that fails empties it before it is tried again."""
import numpy as np
import pytest

from contour3d_amd import api, fields

pytestmark = pytest.mark.gpu

FLOOR = 64 << 20  # other buffers and the driver's own granularity


def free_bytes():
    import torch

    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def build():
    """A mesh of about 800 MB."""
    f = fields.turbulence((200, 200, 200), kmax=50, seed=11)
    cont = [dict(field=f, threshold=t, color=(1, 2, 3)) for t in (-0.5, 0.0, 0.5)]
    return api.Mesh(cont)


def test_mesh_freed_after_finalize_returns_its_memory():
    # what the process loads once (code, the static array) comes first
    build().free()
    api.finalize()
    before = free_bytes()
    m = build()
    n = m.count(0)
    api.finalize()
    held = before - free_bytes()
    assert held > (400 << 20), held
    m.free()
    assert before - free_bytes() < FLOOR
    # and the library still builds the same mesh, and pools it while it is up
    m = build()
    assert m.count(0) == n
    m.free()
    assert before - free_bytes() > (400 << 20)
    api.finalize()
    assert before - free_bytes() < FLOOR


def test_failing_allocation_empties_the_pool(capfd):
    api.finalize()
    m = build()
    first = m.copy(1)
    m.free()
    pooled = free_bytes()
    f = fields.blobs((20, 20, 20), seed=4)
    v = fields.example_view(700, 500)
    args = (v["camera"], v["light"], v["size"], v["center"], v["local"], v["bg"],
            [dict(field=f, threshold=0.5, color=(0, 255, 255))])
    # the frame's first allocations, pinned or on the device, fail one by one
    # (none of them is large)
    emptied = False
    for n in (1, 2, 3, 4):
        api.tune(api.TUNE_FAIL_ALLOC, n)
        try:
            with pytest.raises(RuntimeError):
                api.execute_rgb(*args)
        finally:
            api.tune(api.TUNE_FAIL_ALLOC, 0)
        assert "[CONTOUR3D ERROR] " in capfd.readouterr().err
        emptied = emptied or free_bytes() - pooled > (300 << 20)
    assert emptied
    api.execute_rgb(*args)
    m = build()
    again = m.copy(1)
    m.free()
    assert all(np.array_equal(first[k], again[k], equal_nan=first[k].dtype.kind == "f") for k in first)
