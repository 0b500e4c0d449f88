"""GPU: a frame whose grown fragment list finds no memory is drawn with the
first list and the id pass, in both forms; of a call's allocations only that
one may fail so."""
import numpy as np
import pytest

from contour3d_amd import api, fields

from test_gpu_parity import same_bits, view_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [api.FP64, api.FP32], ids=["fp64", "fp32"])
def test_no_memory_for_a_grown_list(precision, capfd):
    f = fields.turbulence((24, 26, 22), kmax=6, seed=3)
    v = view_for(96, 72)
    cont = [dict(field=f, threshold=t, color=c) for t, c in ((-0.4, (250, 60, 30)), (0.4, (30, 60, 250)))]
    args = (v["camera"], v["light"], v["size"], v["center"], v["local"], v["bg"], cont)
    ref = api.execute_rgb(*args, precision=precision, want_depth=True)

    def failures(capacity):
        """Calls that fail when the n-th allocation does, over n."""
        ok = []
        while ok[-3:] != [True] * 3 and len(ok) < 60:
            api.finalize()
            api.lib().contour3d_amd_init(0)
            api.tune(api.TUNE_FRAG_CAPACITY, capacity)
            api.tune(api.TUNE_FAIL_ALLOC, len(ok) + 1)
            try:
                rgb, depth = api.execute_rgb(*args, precision=precision, want_depth=True)
                assert np.array_equal(rgb, ref[0]) and same_bits(depth, ref[1])
                ok.append(True)
            except RuntimeError:
                ok.append(False)
            finally:
                api.tune(api.TUNE_FAIL_ALLOC, 0)
            rgb, depth = api.execute_rgb(*args, precision=precision, want_depth=True)
            assert np.array_equal(rgb, ref[0]) and same_bits(depth, ref[1])
        return ok.count(False)

    try:
        first, grown = failures(1 << 24), failures((1 << 24) + 4096)
    finally:
        api.tune(api.TUNE_FRAG_CAPACITY, 0)
    capfd.readouterr()
    assert first > 8 and grown == first - 1
