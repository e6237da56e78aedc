"""The network's kernels at the edges of their tiles (32 x 8 pixels of a
convolution, 16 x 16 of a weight gradient; 256 partials of one reduction
pass) against the numpy reference, which rounds the same values to BF16.

Tolerances as for the ragged map of test_gpu_cnn.py: what remains is the order
of FP32 sums and the few values on the other side of a BF16 rounding, 2^-8 of
a value each: 5e-3 relative L2 for outputs, 2e-2 for gradients, 3e-2 a layer.
"""
import numpy as np
import pytest

import cnn_ref as R
from fwiflow.precond import CNN
from test_gpu_cnn import _data, rel, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,W", [(1, 1), (8, 32), (9, 33), (7, 31), (16, 64), (17, 65), (288, 240)])
def test_tile_edges(H, W):
    x, t, m = _data(H, W, 2)
    if H * W == 1:
        m[:] = 1.0
    with CNN(H, W, seed=5) as net:
        p = net.get_params()
        p += 0.05 * np.random.default_rng(3).normal(size=p.size).astype(np.float32)  # biases too
        net.set_params(p)
        out = net.forward(x)
        L, g = net.gradients(x, t, m)
        again = net.gradients(x, t, m)
    assert L == again[0] and np.array_equal(g, again[1])
    p = p.astype(np.float64)
    ref, _ = R.forward(p, x, bf16=True)
    Lr, gr = R.loss_and_grad(p, x, t, m, bf16=True)
    say("tiles", H, W, rel(out, ref), rel(g, gr))
    assert rel(out, ref) < 5e-3
    assert L == pytest.approx(Lr, rel=5e-3)
    assert rel(g, gr) < 2e-2
    o = 0
    for ci, co in R.LAYERS:
        n = co * ci * 9 + co
        assert rel(g[o:o + n], gr[o:o + n]) < 3e-2, (ci, co)
        o += n
