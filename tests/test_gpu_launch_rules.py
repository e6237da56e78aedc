"""The launch shapes that the engine picks by size, at the edges of their
tiles, against the CPU oracle in FP32 (contract tolerances: data 1e-4,
gradients 1e-3 relative L2) and, bit for bit, against each other: a cell's
arithmetic and the order of the sums over shots do not depend on the launch.

``cases`` names (nz, nx, shots, steps): grid edges around the 60 x 4 core of a
whole step and the 64 x 2 tile of a half step (12 C-PML cells a side), one
to four shots (whole backward steps), five and nine shots (two and four
threads a cell, the last round of eight ragged), and a launch of more than
16384 waves (two launches a forward step, shots in slices).
"""
import numpy as np
import pytest

import fwiflow
from fwiflow import models
from test_gpu import GRAD_TOL, SEIS_TOL, env, rel, say

pytestmark = pytest.mark.gpu

CASES = {
    "core_exact_1_shot": (40, 60, 1, 120),
    "core_plus_one_2_shots": (41, 61, 2, 121),
    "two_strips_4_shots": (100, 62, 4, 90),
    "two_strips_long_4_shots": (100, 62, 4, 300),
    "core_plus_one_4_shots": (41, 63, 4, 150),
    "core_plus_one_5_shots": (41, 60, 5, 150),
    "strip_plus_one_9_shots": (105, 63, 9, 61),
    "whole_steps_in_pairs_25_shots": (41, 61, 25, 60),
    "sliced_forward": (41, 331, 24, 60),
}


def _run(P, m, stf, mode, every):
    P.set_adjoint(mode)
    P.set_model(*m)
    P.set_stf(stf)
    P.load_obs()
    P.set_checkpoint(every)
    P.set_illumination(True)
    P.run(1)
    return [P.data(), P.illumination(), *P.gradients()]


def _differing(a, b):
    """{output: (values that differ, span of the rows, of the columns)}"""
    out = {}
    for k, (x, y) in enumerate(zip(a, b)):
        w = np.nonzero(np.atleast_2d(x) != np.atleast_2d(y))
        if len(w[0]):
            out[k] = (len(w[0]), (w[0].min(), w[0].max()), (w[-1].min(), w[-1].max()))
    return out


@pytest.mark.parametrize("mode", ["reference", "exact"])
@pytest.mark.parametrize("name", list(CASES))
def test_launch_rules_match_oracle_and_each_other(oracle_mod, workspace, name, mode):
    nz, nx, shots, steps = CASES[name]
    c = models.case_small(nz=nz, nx=nx, nSteps=steps, nshots=shots)
    para, stf = models.write_case(c, workspace)
    ids = list(range(shots))
    fwiflow.fwi_obs_op(*models.moduli(c, "true"), stf, 0, ids, para)
    m = models.moduli(c, "start")
    say(name, mode, "grid", c.NZ, c.NX, "shots", shots)
    with fwiflow.Plan(para, ids) as P:
        auto = _run(P, m, stf, mode, 0)
        again = _run(P, m, stf, mode, 0)
    assert not _differing(auto, again)
    # one column a workgroup; recomputed segments of 17 steps keep the data
    with env(FWIFLOW_TILE_X="1"), fwiflow.Plan(para, ids) as P:
        assert not _differing(_run(P, m, stf, mode, 0), auto)
        assert not _differing(_run(P, m, stf, mode, 17)[:2], auto)
    scheme = dict(scheme=3, ckpt_every=50) if mode == "exact" else {}
    o = oracle_mod.cufd(*m, stf, 1, ids, para, precision=32, **scheme)
    # (writes its data over the observed files)
    f = oracle_mod.cufd(*m, stf, 2, ids, para, precision=32, illumination=True)[5]
    want = [np.concatenate(f["syn"]), f["illum"], *o[1:5]]
    for k, (a, b) in enumerate(zip(auto, want)):
        n = shots if k == 5 else None  # rows of the source gradient
        a, b = np.ravel(np.asarray(a)[:n]), np.ravel(np.asarray(b)[:n])
        # (90 steps do not reach the anomaly: no residual, gradients that underflow)
        e = rel(a, b) if np.abs(b).max() > 1e-30 else float(np.abs(a).max())
        say(name, mode, k, f"{e:.2e}")
        assert e <= (SEIS_TOL if k < 2 else GRAD_TOL), (k, e)


@pytest.mark.parametrize("groups", [(1, 3), (2, 5), (3, 5), (5, 2)])
def test_recomputed_groups_may_exceed_forward_groups(workspace, groups):
    """Backward launches recompute their own shots from the checkpoints, also
    more of them than a forward launch holds: the same gradients as with one
    launch for all shots, bit for bit where the backward launches are alike."""
    c = models.case_small(nz=41, nx=60, nSteps=150, nshots=5)
    para, stf = models.write_case(c, workspace)
    ids = list(range(5))
    fwiflow.fwi_obs_op(*models.moduli(c, "true"), stf, 0, ids, para)
    m = models.moduli(c, "start")
    fwd, bwd = groups
    with fwiflow.Plan(para, ids) as P:
        P.set_launch(2, 5, bwd)
        want = _run(P, m, stf, "reference", 17)
        P.set_launch(2, fwd, bwd)
        got = _run(P, m, stf, "reference", 17)
    # (the illumination adds up another way over other forward launches)
    assert not _differing(got[:1] + got[2:], want[:1] + want[2:])
