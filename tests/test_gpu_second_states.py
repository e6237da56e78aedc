"""Steps of one launch keep a second copy of the state.  Where a plan has no
room for it (FWIFLOW_PLAN_BYTES), its run takes two launches a step, holds
nothing for the other form and gives the same numbers, bit for bit; only where
the two-launch form does not fit either is the run refused."""
import os

import numpy as np
import pytest

import fwiflow
from fwiflow import models
from test_gpu import env

pytestmark = pytest.mark.gpu


def _case(ws, nz, nx, shots, steps=60):
    c = models.case_small(nz=nz, nx=nx, nSteps=steps, nshots=shots)
    para, stf = models.write_case(c, ws)
    ids = list(range(shots))
    fwiflow.fwi_obs_op(*models.moduli(c, "true"), stf, 0, ids, para)
    return para, stf, ids, models.moduli(c, "start")


def _plan(case, limit=0):
    para, stf, ids, m = case
    with env(FWIFLOW_PLAN_BYTES=str(int(limit))):
        P = fwiflow.Plan(para, ids)
    P.set_model(*m)
    P.set_stf(stf)
    P.load_obs()
    return P


def _run(P, every):
    P.set_checkpoint(every)
    P.set_illumination(True)
    P.run(1)
    held = P.device_bytes()
    return held, [P.data(), P.illumination(), *P.gradients()]


def _same(a, b):
    return all(np.array_equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("shots,every", [(2, 0), (2, 17), (5, 0)])
def test_run_without_room_for_second_states(workspace, shots, every):
    case = _case(workspace, 41, 61, shots)
    with _plan(case) as P:
        most, want = _run(P, every)
        tile = P.tile_width()
    with _plan(case, most - 4) as P:
        held, got = _run(P, every)
        assert P.tile_width() > 0 and _same(got, want)
        # a run that needs less finds the room
        P.run(2)
        assert P.tile_width() in (0, 2) and np.array_equal(P.data(), want[0])
    assert held < most and tile == (0 if shots == 2 else 2)
    for limit in np.linspace(held, most - 4, 7).astype(int):
        with _plan(case, limit) as P:
            h, got = _run(P, every)
            assert h == held and P.tile_width() > 0 and _same(got, want), limit
    with _plan(case, held - 4) as P, pytest.raises(fwiflow.FwiflowError) as e:
        _run(P, every)
    assert e.value.status == "FWIFLOW_ERR_MEMORY"


def test_job_whose_second_plan_has_no_room(workspace):
    cases = [_case(os.path.join(workspace, str(k)), *g, 2) for k, g in enumerate([(41, 61), (50, 80)])]
    want, half = [], []
    for c in cases:
        with _plan(c) as P:
            most, w = _run(P, 0)
        with _plan(c, most - 4) as P:
            half.append(_run(P, 0)[0])
        want.append(w)
    plans = [_plan(cases[0]), _plan(cases[1], half[1])]
    try:
        for P in plans:
            P.set_illumination(True)
        with fwiflow.Job(plans) as J:
            J.run(1)
            assert J.fused()
        for P, h, w in zip(plans, half, want):
            assert P.device_bytes() == h and P.tile_width() == 2
            assert _same([P.data(), P.illumination(), *P.gradients()], w)
    finally:
        for P in plans:
            P.close()


def test_second_states_are_sized_for_the_launches_that_have_them(workspace):
    """24 shots forward in one launch of half steps, backward alone: the second
    state holds one shot (13 + 5 arrays)."""
    case = _case(workspace, 41, 331, 24, 20)
    with _plan(case) as P:
        P.set_launch(2, 0, 1)
        most, want = _run(P, 0)
        cells = P.nz * P.nx
    with _plan(case, most - 4) as P:
        P.set_launch(2, 0, 1)
        held, got = _run(P, 0)
    assert _same(got, want)
    assert most - held == 18 * 4 * cells


@pytest.mark.parametrize("shots,every", [(2, 0), (3, 17), (5, 0)])
def test_second_states_of_earlier_runs_give_way(workspace, shots, every):
    """A modelling run takes one launch a step and keeps its second state; what
    the plan asks for afterwards (observed data, a gradient's buffers,
    illumination) has to find the room that it would have found without."""
    para, stf, ids, m = case = _case(workspace, 41, 61, shots)
    with _plan(case) as P:
        most, want = _run(P, every)
        obs = np.concatenate([np.fromfile(f"{workspace}/Data/Shot{i}.bin", np.float32) for i in ids])
    with _plan(case, most - 4) as P:
        held, _ = _run(P, every)
    with env(FWIFLOW_PLAN_BYTES=str(held)):
        P = fwiflow.Plan(para, ids)
    with P:
        P.set_model(*m)
        P.set_stf(stf)
        P.run(2)
        assert P.tile_width() == 0
        assert np.array_equal(P.data(), want[0])
        P.set_obs(obs)
        P.run(0)
        h, got = _run(P, every)
        assert h <= held and _same(got, want)
        P.run(2)
        assert np.array_equal(P.data(), want[0])
        assert _same(_run(P, every)[1], want)
