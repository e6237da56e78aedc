"""Launch shapes that a caller chooses: the automatic one can be asked for, and
every tile of the two-launch steps gives the automatic one's numbers, bit for
bit (a cell's arithmetic and the order of the sums do not depend on the tile).
"""
import numpy as np
import pytest

import fwiflow
from fwiflow import models

pytestmark = pytest.mark.gpu


def _case(ws, nz, nx, shots, steps):
    c = models.case_small(nz=nz, nx=nx, nSteps=steps, nshots=shots)
    para, stf = models.write_case(c, ws)
    ids = list(range(shots))
    fwiflow.fwi_obs_op(*models.moduli(c, "true"), stf, 0, ids, para)
    return para, stf, ids, models.moduli(c, "start")


def _ready(P, m, stf):
    P.set_model(*m)
    P.set_stf(stf)
    P.load_obs()


def _grad(P):
    P.run(1)
    return [P.data(), *P.gradients()]


def _same(a, b):
    return all(np.array_equal(x, y) for x, y in zip(a, b))


# shots: tile of a gradient run's half steps (0: whole steps, 2, and 1 where
# four threads share a cell)
@pytest.mark.parametrize("shots,width", [(2, 0), (5, 2), (9, 1)])
def test_automatic_tile_can_be_asked_for(workspace, shots, width):
    para, stf, ids, m = _case(workspace, 41, 61, shots, 60)
    with fwiflow.Plan(para, ids) as P:
        assert P.tile_width() == 0
        _ready(P, m, stf)
        assert P.launch() == (-1, -1, -1)
        want = _grad(P)
        assert P.tile_width() == width
        P.set_launch(*P.launch())
        assert _same(_grad(P), want) and P.tile_width() == width
        P.set_launch(4, -1, -1)
        assert P.launch() == (4, -1, -1)
        assert _same(_grad(P), want) and P.tile_width() == (4 if width else 0)
        P.set_launch(-1)
        assert P.launch() == (-1, -1, -1)
        assert _same(_grad(P), want) and P.tile_width() == width
        for tile in (-2, 0, 5):
            with pytest.raises(fwiflow.FwiflowError) as e:
                P.set_launch(tile)
            assert e.value.status == "FWIFLOW_ERR_ARG"
        assert P.launch() == (-1, -1, -1)
