"""The network on a map of more than 524288 rows: its tiles, 8 rows each, are more
than 65536, which is as many workgroups as a grid holds along y."""
import numpy as np
import pytest

from fwiflow.precond import CNN

pytestmark = pytest.mark.gpu

TAIL = 8201      # rows of the short map: 16 x 512 and a ragged rest
H = 516096 + TAIL  # 524297, 16 x 32256 rows above it


def test_last_rows_of_a_tall_map():
    """An output depends on 4 rows above it, a gradient of a loss that sees the
    last rows alone on no more: both equal a short map's bit for bit (tiles and
    the order of their sums start at the same rows)."""
    rng = np.random.default_rng(0)
    x = rng.standard_normal((4, H, 1)).astype(np.float32)
    t = rng.standard_normal((3, H, 1)).astype(np.float32)
    m = np.zeros((H, 1), np.float32)
    m[-64:] = 1.0
    with CNN(H, 1, seed=5) as tall, CNN(TAIL, 1, seed=5) as short:
        out = tall.forward(x)
        L, g = tall.gradients(x, t, m)
        tail = [np.ascontiguousarray(a[..., -TAIL:, :]) for a in (x, t, m)]
        ref = short.forward(tail[0])
        Ls, gs = short.gradients(*tail)
    assert np.any(ref[:, -1]) and np.any(gs)
    assert np.array_equal(out[:, -TAIL + 4:], ref[:, 4:])
    assert L == pytest.approx(Ls, rel=1e-12) and np.array_equal(g, gs)
