"""Gradients and illumination of small grids are turned on the host, of others on
the device: both sides of the line (20480 cells, padding included) against the
CPU oracle in FP32 (contract tolerances), and the time that the former take."""
import time

import numpy as np
import pytest

import fwiflow
from fwiflow import models
from test_gpu import GRAD_TOL, SEIS_TOL, rel

pytestmark = pytest.mark.gpu


# NZ = 160, NX = 127, 128 (the line), 129; and a small ragged one
@pytest.mark.parametrize("nz,nx,cells", [(104, 103, 20320), (104, 104, 20480), (104, 105, 20640), (41, 61, 8160)])
def test_turned_on_host_or_device(oracle_mod, workspace, nz, nx, cells):
    c = models.case_small(nz=nz, nx=nx, nSteps=150, nshots=2)
    para, stf = models.write_case(c, workspace)
    ids = [0, 1]
    fwiflow.fwi_obs_op(*models.moduli(c, "true"), stf, 0, ids, para)
    m = models.moduli(c, "start")
    with fwiflow.Plan(para, ids) as P:
        assert P.nz * P.nx == cells
        P.set_model(*m)
        P.set_stf(stf)
        P.load_obs()
        P.set_illumination(True)
        P.run(1)
        got = [P.illumination(), *P.gradients()]
        again = [P.illumination(), *P.gradients()]
        J = P.misfit()
        P.run(0)  # the arrays that the turn uses are cleared by a run
        assert P.misfit() == J
    assert all(np.array_equal(a, b) for a, b in zip(got, again))
    o = oracle_mod.cufd(*m, stf, 1, ids, para, precision=32)
    f = oracle_mod.cufd(*m, stf, 2, ids, para, precision=32, illumination=True)[5]
    assert rel(got[0], f["illum"]) <= SEIS_TOL
    for a, b in zip(got[1:], o[1:5]):
        assert rel(a, np.asarray(b)[:len(a)]) <= GRAD_TOL
    # (single precision, as it is on the device)
    assert all(np.array_equal(a, a.astype(np.float32)) for a in got)


def test_gradients_of_a_small_grid_take_one_copy(workspace):
    """On 96 x 84 cells: against the time of data(), which is a kernel, a copy and
    a wait.  Two copies (the source gradient's the second) and the turn: 1.5 times
    it; with a kernel and a copy an array 2.4."""
    c = models.case_small(nz=40, nx=60, nSteps=60, nshots=1)
    para, stf = models.write_case(c, workspace)
    with fwiflow.Plan(para, [0]) as P:
        P.set_model(*models.moduli(c, "true"))
        P.set_stf(stf)
        P.run(2)
        P.set_obs(P.data())
        P.run(1)
        best = [np.inf, np.inf]
        for _ in range(200):
            for k, f in enumerate((P.gradients, P.data)):
                t = time.perf_counter()
                f()
                best[k] = min(best[k], time.perf_counter() - t)
    print("gradients, data:", [1e6 * b for b in best])
    assert best[0] < 2.0 * best[1]
