"""The matrix-core loss gradient at the edges of its split: 32 samples per
wavefront, one chunk per block up to 256 blocks (8 192 samples), then 8
wavefronts per block (65 536 samples), then chunks in turn.

Tolerance: a gradient entry is a sum of per-sample terms, each the result of
at most 64 + 64 + 9 + 10 rounded operations in a row and the activations'
3 ulp, so each term is off by at most 160 x 2^-24 = 1e-5 of its size; terms of
one block of parameters cancel by less than a factor of ten on these inputs.
"""
import numpy as np
import pytest

from oracle import oracle as O
from simuverse_amd import lbm as L

pytestmark = pytest.mark.gpu

BLOCKS = ((0, 576), (576, 640), (640, 4736), (4736, 4800), (4800, 5376), (5376, 5385))


@pytest.mark.parametrize("n", [1, 31, 32, 33, 8192, 8193, 65537, 70001])
def test_gradient_at_split_edges(n):
    assert L.device_count() >= 1, "no gfx950 device visible"
    print(f"case: loss gradient n={n}", flush=True)
    rng = np.random.default_rng(n)
    p = (rng.standard_normal(5385) * 0.3).astype(np.float32)
    x = rng.standard_normal((n, 9)).astype(np.float32)
    t = rng.standard_normal((n, 9)).astype(np.float32)
    net = L.Network(seed=1)
    net.set_params(p)
    loss, g = net.loss_grad(x, t)
    lref, gref = O.mlp_loss_grad(p.astype(np.float64), x.astype(np.float64), t.astype(np.float64))
    assert abs(loss - lref) < 1e-5 * lref
    for a, b in BLOCKS:
        assert np.linalg.norm(g[a:b] - gref[a:b]) <= 1e-4 * np.linalg.norm(gref[a:b])
    # the same bits again
    loss2, g2 = net.loss_grad(x, t)
    assert loss2 == loss and np.array_equal(g2, g)
    net.close()


def test_gradient_large_activations():
    """Pre-activations far outside GELU's bend, both signs: finite, and the
    derivative is 0 or 1 there."""
    print("case: loss gradient, large activations", flush=True)
    rng = np.random.default_rng(7)
    p = (rng.standard_normal(5385) * 0.3).astype(np.float32)
    x = (rng.standard_normal((257, 9)) * 300.0).astype(np.float32)
    t = rng.standard_normal((257, 9)).astype(np.float32)
    net = L.Network(seed=1)
    net.set_params(p)
    loss, g = net.loss_grad(x, t)
    lref, gref = O.mlp_loss_grad(p.astype(np.float64), x.astype(np.float64), t.astype(np.float64))
    assert np.all(np.isfinite(g))
    assert abs(loss - lref) < 1e-5 * lref
    for a, b in BLOCKS:
        assert np.linalg.norm(g[a:b] - gref[a:b]) <= 1e-4 * np.linalg.norm(gref[a:b])
    net.close()
