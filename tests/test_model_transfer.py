"""Models to the device and gradients back, at grid sizes around the 32 x 32
tiles that turn them: what the device ends up with is compared bit for bit
between the two layouts the entry points take, and the Courant check between
the host's and the device's pass over the model."""
import numpy as np
import pytest

import fwiflow
from fwiflow import models
from test_gpu import _run_plan


def _setup(ws, nz, nx):
    c = models.case_small(nz=nz, nx=nx, nSteps=120, nshots=2)
    para, stf = models.write_case(c, ws)
    return c, para, stf, models.moduli(c, "true")


def _refused(call):
    with pytest.raises(fwiflow.FwiflowError) as e:
        call()
    return e.value.status == "FWIFLOW_ERR_COURANT"


def _bad_models(m):
    """(model, refused): a fast cell last, a first cell without a speed, and
    another cell without one, which the maximum passes over."""
    lam, mu, den = m
    fast, first, other = lam.copy(), lam.copy(), lam.copy()
    fast[-1, -1] *= 100.0
    first[0, 0] = np.nan
    other[3, 5] = np.nan
    return [((fast, mu, den), True), ((first, mu, den), True), ((other, mu, den), False),
            ((-lam, -mu, den), True), (m, False)]


def test_courant_check_of_models_without_a_speed(workspace):
    c, para, stf, m = _setup(workspace, 40, 60)
    for bad, refused in _bad_models(m):
        if refused:
            assert _refused(lambda: fwiflow.check_call(2, [0], para, *bad))
        else:
            fwiflow.check_call(2, [0], para, *bad)


@pytest.mark.gpu
@pytest.mark.parametrize("nz,nx", [(40, 40), (40, 73), (41, 72), (104, 103)])
def test_layouts_and_refusals(workspace, nz, nx):
    c, para, stf, m = _setup(workspace, nz, nx)
    fwiflow.fwi_obs_op(m[0] * 1.02, m[1], m[2], stf, 0, [0, 1], para)
    d, g, J, _ = _run_plan(para, [0, 1], *m, stf)
    with fwiflow.Plan(para, [0, 1]) as P:
        P.set_model(*(a.ravel(order="F") for a in m), zfast=True)
        P.set_stf(stf)
        P.load_obs()
        for bad, refused in _bad_models(m):
            if refused:  # the model in place stays
                assert _refused(lambda: P.set_model(*bad))
        P.run(1)
        assert np.array_equal(P.data(), d)
        g2 = P.gradients()
        assert all(np.array_equal(a, b) for a, b in zip(g2, g))
        assert np.any(g2[0])
        P.run(0)
        assert P.misfit() == J
