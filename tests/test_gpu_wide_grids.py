"""Grids of many columns: the two-launch steps walk them in chunks of 16 columns
an XCD, several slices of the shots side by side."""
import time

import numpy as np
import pytest

import fwiflow
from fwiflow import models

pytestmark = pytest.mark.gpu


def _plan(ws, nz, nx, shots, steps):
    c = models.case_small(nz=nz, nx=nx, nSteps=steps, nshots=shots)
    para, stf = models.write_case(c, ws)
    P = fwiflow.Plan(para, list(range(shots)))
    P.set_model(*models.moduli(c, "true"))
    P.set_stf(stf)
    P.run(2)
    P.set_obs(P.data())
    P.set_model(*models.moduli(c, "start"))
    return P


# 24 and 117 chunks, of three slices and of one; the last chunk ragged
@pytest.mark.parametrize("nx,shots", [(3003, 6), (14977, 2)])
@pytest.mark.parametrize("mode", ["reference", "exact"])
def test_chunks_and_slices_cover_a_wide_grid(workspace, nx, shots, mode):
    """The same numbers, bit for bit, for every tile (each cuts other chunks)
    and with single shots in launches of their own; gradients up to the order
    of the sums over the launches there."""
    P = _plan(workspace, 24, nx, shots, 40)
    with P:
        P.set_adjoint(mode)
        got = {}
        for shape in ((-1, -1, -1), (1, -1, -1), (2, -1, -1), (3, -1, -1), (4, -1, -1), (2, 1, 1)):
            P.set_launch(*shape)
            P.run(1)
            got[shape] = [P.data(), *P.gradients()]
    want = got.pop((-1, -1, -1))
    single = got.pop((2, 1, 1))
    for shape, g in got.items():
        assert all(np.array_equal(a, b) for a, b in zip(g, want)), shape
    assert np.array_equal(single[0], want[0])
    for a, b in zip(single[1:], want[1:]):
        assert np.linalg.norm(a - b) <= 1e-5 * np.linalg.norm(b)


def test_time_follows_the_cells_not_the_columns(workspace):
    """3.8 million cells in 64 rows and in 1024: the first have four times as
    many C-PML rows (2.1 times the traffic a cell at most) and the same number
    of waves.  2.5 leaves room for noise; a loop over the 469 chunks took 5.1 (now 1.4)."""
    ms = []
    for k, (nz, nx) in enumerate([(40, 60000), (1000, 3700)]):
        with _plan(f"{workspace}/{k}", nz, nx, 1, 60) as P:
            best = np.inf
            for _ in range(6):
                t = time.perf_counter()
                P.run(2)
                best = min(best, time.perf_counter() - t)
        ms.append(best * 1e3)
    print("wide / deep:", ms)
    assert ms[0] < 2.5 * ms[1]
