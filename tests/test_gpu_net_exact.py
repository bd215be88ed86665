"""Network kernels on whole numbers: outputs and gradients must be exact.

Weights of -1, 0 and 1 with few entries per output channel (and parity, where
a layer doubles the grid), inputs and output gradients of -1, 0 and 1: every
activation and gradient is a whole number of at most 256, which bf16 holds, and
every FP32 sum stays below 2^24.  So the device has to give the oracle's
(oracle/cnn_oracle.py) numbers, at the faces of the grid and in every layer,
with no tolerance.
"""
import numpy as np
import pytest

from oracle import cnn_oracle as N
from pigfem_assignment_amd.api import GuessNet

pytestmark = pytest.mark.gpu


def sparse_case(seed, G=64):
    rng = np.random.RandomState(seed)
    layers = []
    for l, (m, ci, co) in enumerate(N.SPECS):
        T = N.taps(m)
        per = 5 if l == 7 else 2  # three of layer 7's outputs are used
        W = np.zeros((T, ci, co))
        for n in range(co):
            for t in (range(T) if m == N.UP else rng.randint(T, size=per)):
                W[t, rng.randint(ci, size=per), n] = rng.choice([1, -1])
        layers.append((W, rng.randint(0, 2, co).astype(np.float64)))
    x = rng.choice([-1, 0, 0, 1], (G, G, G, 8)).astype(np.float32)
    dy = rng.choice([-1, 0, 0, 0, 0, 0, 0, 1], (G, G, G, 3)).astype(np.float32)
    return N.flatten(layers), x, dy


@pytest.mark.parametrize("seed", [0, 1])
def test_whole_numbers_are_exact(seed):
    p, x, dy = sparse_case(seed)
    dy16 = np.zeros(dy.shape[:3] + (16,))
    dy16[..., :3] = dy
    yo = N.forward(p, x)[0][..., :3]
    go = N.backward(p, x, dy16)
    assert np.abs(go).max() < 2 ** 24
    # what is rounded to bf16 is a whole number that bf16 holds
    assert np.array_equal(go, N.backward(p, x, dy16, rounding=False))
    assert np.array_equal(yo, N.forward(p, x, rounding=False)[0][..., :3])
    net = GuessNet(seed=1)
    net.set_params(p.astype(np.float32))
    assert np.array_equal(net.forward(x), yo.astype(np.float32))
    g = net.backward(x, dy)
    o = 0
    for l, (m, ci, co) in enumerate(N.SPECS):
        for k in (N.taps(m) * ci * co, co):
            bad = np.flatnonzero(g[o:o + k] != go[o:o + k])
            assert bad.size == 0, "layer %d: %d of %d differ, first %d" % (l, bad.size, k, bad[0])
            o += k
