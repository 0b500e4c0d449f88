"""CPU: what api.autotune sweeps and leaves set (the knobs recorded instead of
passed to the library).  The defaults are among the settings, and they stay
unless another setting is clearly faster: a brick shape that is set holds for
every later view."""
import time

import pytest

from contour3d_amd import api


class Knobs(dict):
    clock = 0.0

    def spend(self, s):
        self.clock += s


@pytest.fixture
def knobs(monkeypatch):
    """The knobs as they are set; spend() is what a run takes."""
    import torch

    now = Knobs({p: 0 for p in api.AUTOTUNE_KNOBS})
    monkeypatch.setattr(api, "tune", lambda p, v: now.__setitem__(p, v))
    monkeypatch.setattr(torch.cuda, "synchronize", lambda: None)
    monkeypatch.setattr(time, "perf_counter", lambda: now.clock)
    return now


def test_the_defaults_are_swept_and_stay(knobs):
    for values in api.AUTOTUNE_KNOBS.values():
        assert values[0] == 0 and len(set(values)) == len(values)
    # a frame's bricks have at most 8 rows and planes, its grid 6 workgroups on each of 256 CUs
    assert max(api.AUTOTUNE_KNOBS[api.TUNE_TESS_ZPLANES]) <= 8
    assert max(api.AUTOTUNE_KNOBS[api.TUNE_TESS_ROWS]) <= 8
    assert max(api.AUTOTUNE_KNOBS[api.TUNE_TESS_GRID]) < 6 * 256

    def run():  # the defaults are 1 % slower than the rest
        knobs.spend(0.02 if any(knobs.values()) else 0.0202)

    kept, ms, sweep = api.autotune(run, reps=1)
    assert set(knobs.values()) == {0} and set(kept.values()) == {0}
    assert len(sweep) == 16 and ms == dict((tuple(k.values()), m) for k, m in sweep)[(0, 0, 0)]


def test_a_clearly_faster_setting_is_kept(knobs):
    def run():
        knobs.spend(0.002 if knobs[api.TUNE_TESS_ZPLANES] == 2 and knobs[api.TUNE_TESS_ROWS] == 0 else 0.01)

    kept, _, _ = api.autotune(run, reps=1)
    assert kept["tess_zplanes"] == 2 and kept["tess_rows"] == 0
    assert {api.KNOB_NAMES[p]: v for p, v in knobs.items()} == kept


def test_a_sweep_without_the_defaults_keeps_the_fastest(knobs):
    kept, _, _ = api.autotune(lambda: knobs.spend(0.001 * knobs[api.TUNE_TESS_ZPLANES]),
                              knobs={api.TUNE_TESS_ZPLANES: (8, 2, 4)}, reps=1)
    assert kept == {"tess_zplanes": 2} and knobs[api.TUNE_TESS_ZPLANES] == 2
