"""The autotuner against a plan whose runs take times from a table: the
automatic shape is measured and kept where it is the fastest, and shapes
measured on another engine are not applied."""
import os

import numpy as np
import pytest

from fwiflow import models, tune


class FakePlan:
    """Runs of (tile, shots forward, shots backward) take cost(...) seconds;
    the automatic shape is tile `auto` (0: every step one launch), 3 / 2 shots."""
    auto, now = 2, 0.0
    ran = []

    def __init__(self, *a):
        self.shape = (-1, -1, -1)

    def __enter__(self):
        return self

    def __exit__(self, *a):
        pass

    def set_model(self, *a):
        pass

    set_stf = set_obs = set_model

    def data(self):
        return np.zeros(1)

    def set_launch(self, *a):
        self.shape = a

    def shots_per_launch(self):
        return 3, 2

    def tile_width(self):
        return self.auto

    def run(self, calc):
        t, f, b = self.shape
        shape = (self.auto if t == -1 else t, 3 if f == -1 else f, 2 if b == -1 else b)
        type(self).ran.append(shape)
        type(self).now += self.cost(*shape)

    def cost(self, t, f, b):
        return 1.0 + abs(t - self.auto) + abs(f - 3) + abs(b - 2)


def _tune(ws, monkeypatch, auto):
    c = models.case_small(nz=40, nx=60, nSteps=100, nshots=5)
    para, stf = models.write_case(c, ws)
    FakePlan.auto, FakePlan.now, FakePlan.ran = auto, 0.0, []
    monkeypatch.setattr(tune, "Plan", FakePlan)
    monkeypatch.setattr(tune.time, "perf_counter", lambda: FakePlan.now)
    path = os.path.join(ws, "tune", "launch.json")
    return tune.autotune(para, range(5), *models.moduli(c, "true"), stf, path=path), para, path


@pytest.mark.parametrize("auto", [1, 2, 3])
def test_automatic_shape_is_measured_and_kept_if_fastest(workspace, monkeypatch, auto):
    e, para, path = _tune(workspace, monkeypatch, auto)
    assert (e["tile_x"], e["shots_fwd"], e["shots_bwd"]) == (auto, 3, 2)
    assert e["automatic"] == [auto, 3, 2] and e["automatic_seconds"] == e["seconds"] == 1.0
    assert {1, 2, 4} <= {s[0] for s in FakePlan.ran[2:]}
    assert tune.lookup(para, 5, path) == e


def test_tiles_are_not_varied_where_steps_have_none(workspace, monkeypatch):
    e, para, path = _tune(workspace, monkeypatch, 0)
    assert {s[0] for s in FakePlan.ran[2:]} == {2}
    assert len(e["candidates"]) > 1 and e["automatic_seconds"] is not None


def test_shapes_of_another_engine_are_not_applied(workspace, monkeypatch):
    e, para, path = _tune(workspace, monkeypatch, 2)
    fake = FakePlan()
    assert tune.apply_tuned(fake, para, 5, path) == e and fake.shape == (2, 3, 2)
    for old in ({k: v for k, v in e.items() if k != "engine"}, dict(e, engine=tune.ENGINE - 1)):
        tune.store(tune.cache_key(para, 5), old, path)
        fake = FakePlan()
        assert tune.apply_tuned(fake, para, 5, path) is None
        assert fake.shape == (-1, -1, -1)
