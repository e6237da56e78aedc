"""The two-launch steps in every tile width and in captured graphs: where the
launches are so large that both directions take them (24 shots of 65 x 357 cells,
17136 columns of whole-step tiles, four threads a cell backward; the update
region's 353 columns are a multiple of no tile width), and with five shots of a
small grid (half steps backward alone, two threads a cell).

Against the CPU oracle in FP32 (contract tolerances: data 1e-4, gradients 1e-3
relative L2) and, bit for bit, against each other: a cell's arithmetic and the
order of the sums over shots do not depend on the launch.
"""
import numpy as np
import pytest

import fwiflow
from fwiflow import models
from test_gpu import GRAD_TOL, SEIS_TOL, env, rel, say

pytestmark = pytest.mark.gpu

CASES = {"four_threads": (41, 333, 24, 60), "two_threads": (41, 62, 5, 150)}
SEPARATE = {"FWIFLOW_FOLD_INJECT": "0"}
GRAPHS = {"FWIFLOW_GRAPHS": "1"}


def _case(ws, name):
    nz, nx, shots, steps = CASES[name]
    c = models.case_small(nz=nz, nx=nx, nSteps=steps, nshots=shots)
    para, stf = models.write_case(c, ws)
    ids = list(range(shots))
    fwiflow.fwi_obs_op(*models.moduli(c, "true"), stf, 0, ids, para)
    return para, stf, ids, models.moduli(c, "start")


def _plan(case, **settings):
    para, stf, ids, m = case
    with env(**settings):
        P = fwiflow.Plan(para, ids)
    P.set_model(*m)
    P.set_stf(stf)
    P.load_obs()
    P.set_illumination(True)
    return P


def _outputs(P, calc):
    P.run(calc)
    out = [P.data(), P.illumination()]
    if calc < 2:
        out.append(np.array([P.misfit()]))
    return out + list(P.gradients()) if calc == 1 else out


def _same(a, b):
    return len(a) == len(b) and all(np.array_equal(x, y) for x, y in zip(a, b))


def test_modelling_in_pairs_of_columns_matches_oracle(oracle_mod, workspace):
    """The default tile of a forward run (two columns), then the others."""
    case = _case(workspace, "four_threads")
    para, stf, ids, m = case
    with _plan(case) as P:
        want = _outputs(P, 2)
        assert P.tile_width() == 2
        J = _outputs(P, 0)[2]
        for tile in (1, 2, 3, 4):
            P.set_launch(tile)
            assert _same(_outputs(P, 2), want) and P.tile_width() == tile
            assert _outputs(P, 0)[2] == J
    f = oracle_mod.cufd(*m, stf, 2, ids, para, precision=32, illumination=True)[5]
    for a, b in zip(want, (np.concatenate(f["syn"]), f["illum"])):
        e = rel(a.ravel(), b.ravel())
        say("modelling", f"{e:.2e}")
        assert e <= SEIS_TOL


@pytest.mark.parametrize("mode", ["reference", "exact"])
@pytest.mark.parametrize("name", list(CASES))
def test_gradients_in_every_tile_match_oracle_and_each_other(oracle_mod, workspace, name, mode):
    case = _case(workspace, name)
    para, stf, ids, m = case
    with _plan(case) as P:
        P.set_adjoint(mode)
        want = _outputs(P, 1)
        assert P.tile_width() == (1 if name == "four_threads" else 2)
        P.set_checkpoint(17)
        segments = _outputs(P, 1)
        for tile in (1, 2, 3, 4):
            P.set_launch(tile)
            P.set_checkpoint(0)
            assert _same(_outputs(P, 1), want) and P.tile_width() == tile
            P.set_checkpoint(17)
            assert _same(_outputs(P, 1), segments)
    with _plan(case, **SEPARATE) as P:  # residuals injected by a launch of their own
        P.set_adjoint(mode)
        for tile in (-1, 3):
            P.set_launch(tile)
            assert _same(_outputs(P, 1), want)
    scheme = dict(scheme=3, ckpt_every=50) if mode == "exact" else {}
    o = oracle_mod.cufd(*m, stf, 1, ids, para, precision=32, **scheme)
    for a, b in zip(want[3:], o[1:5]):
        b = np.asarray(b)[:len(a)]
        e = rel(a.ravel(), b.ravel())
        say(name, mode, f"{e:.2e}")
        assert e <= GRAD_TOL


@pytest.mark.parametrize("mode", ["reference", "exact"])
@pytest.mark.parametrize("name", list(CASES))
def test_replayed_graphs_match_eager_runs(workspace, name, mode):
    """Captured on the first run of a kind and launch shape, replayed on the
    others, with runs of other kinds and an eager plan's work between them."""
    case = _case(workspace, name)
    with _plan(case) as E, _plan(case, **GRAPHS) as G:
        E.set_adjoint(mode)
        G.set_adjoint(mode)
        want = {c: _outputs(E, c) for c in (0, 1, 2)}
        for calc in (2, 1, 1, 0, 2, 1, 2, 0, 1):
            assert _same(_outputs(G, calc), want[calc]), calc
            E.run(0)
        G.set_launch(3)
        for calc in (1, 2, 1):
            assert _same(_outputs(G, calc), want[calc]), calc
            assert G.tile_width() in (0, 3)
