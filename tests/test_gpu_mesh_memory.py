"""GPU: what rendering a stored mesh allocates.  The fragment list (2^24 entries
at first, and a quarter of headroom) has 16-byte entries in FP64, and an FP32
render, which keeps no list, allocates none."""
import numpy as np
import pytest

from contour3d_amd import api, fields

from test_gpu_parity import same_bits, view_for
from test_gpu_pool_release import free_bytes

pytestmark = pytest.mark.gpu

LIST = (1 << 24) * 16 * 5 // 4


@pytest.mark.parametrize("precision, limit", [(api.FP64, LIST), (api.FP32, 0)], ids=["fp64", "fp32"])
def test_render_allocates_the_list_it_uses(precision, limit):
    cont = [dict(field=fields.blobs((24, 24, 24), seed=9), threshold=0.5, color=(9, 90, 200))]
    v = view_for(96, 72)
    args = (v["camera"], v["light"], v["size"], v["center"], v["local"], v["bg"])
    m = api.Mesh(cont, precision=precision)
    m.render(*args)  # (what the process loads once)
    m.free()
    api.finalize()
    m = api.Mesh(cont, precision=precision)
    before = free_bytes()
    rgb, depth = m.render(*args, want_depth=True)
    used = before - free_bytes()
    m.free()
    assert used < limit + (32 << 20), used
    # a frame after it takes the longer entries
    ref = api.execute_rgb(*args, cont, precision=precision, want_depth=True)
    assert np.array_equal(rgb, ref[0]) and same_bits(depth, ref[1])
