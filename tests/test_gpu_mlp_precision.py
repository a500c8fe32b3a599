"""How exact the matrix-core loss gradient is: its GELU and the derivative at
single points, and whole gradients beside a plain binary32 evaluation."""
import math

import numpy as np
import pytest
import torch

from simuverse_amd import lbm as L

pytestmark = pytest.mark.gpu

W1, B1, W2, B2, W3, B3, END = 0, 576, 640, 4736, 4800, 5376, 5385
U = 2.0**-24


def gelu_at(net, a):
    """GELU and GELU' of 64 binary32 points as the gradient kernel forms them.

    One sample; unit k of the first layer has weights 0 and bias a[k], the
    second layer's unit 0 has weights 2^-30 and bias 30, where GELU is the
    identity, and feeds output 0.  Then dL/dW2[0][k] = D2 GELU(a[k]) and
    dL/db1[k] = 2^-30 D2 GELU'(a[k]) with D2 = dL/db2[0], each one product: the
    factors come out by a division in binary64."""
    p = np.zeros(END, np.float32)
    p[B1:W2] = a
    p[W2:W2 + 64] = 2.0**-30
    p[B2] = 30.0
    p[W3] = 1.0
    net.set_params(p)
    t = np.zeros((1, 9), np.float32)
    t[0, 0] = 25.5
    _, g = net.loss_grad(np.zeros((1, 9), np.float32), t)
    g = g.astype(np.float64)
    return g[W2:W2 + 64] / g[B2], g[B1:W2] / (g[B2] * 2.0**-30)


def test_gelu_and_its_derivative():
    """Bounds: with q = 1 - Phi(|x|), the fit is off by 8.3e-9 at most; q carries
    the roundings of a reciprocal, seven polynomial steps, two products and an
    exponential (14 units of 2^-24) and x^2 units from the exponent's argument;
    1 - q rounds once; then x Phi, or the product x phi(x) and its sum, and the
    readout here, each round once."""
    print("case: GELU of 1280 points", flush=True)
    net = L.Network(seed=1)
    x = np.concatenate([np.linspace(-9.0, 9.0, 1216), np.geomspace(1e-6, 0.5, 32), -np.geomspace(1e-6, 0.5, 32)])
    x = x.astype(np.float32)
    y, d = (np.concatenate(v) for v in zip(*(gelu_at(net, x[k:k + 64]) for k in range(0, x.size, 64))))
    net.close()
    X = x.astype(np.float64)
    erfc = np.array([math.erfc(abs(v) / math.sqrt(2.0)) for v in X])
    q = 0.5 * erfc
    Phi = np.where(X >= 0, 1.0 - q, q)
    dens = np.exp(-0.5 * X * X) / math.sqrt(2.0 * math.pi)
    dPhi = 8.3e-9 + q * (14 + X * X) * U + U
    ey, ed = np.abs(y - X * Phi), np.abs(d - (Phi + X * dens))
    print(f"  GELU error: largest {ey.max():.2e}, rms {np.sqrt((ey**2).mean()):.2e}; derivative: largest {ed.max():.2e}, "
          f"rms {np.sqrt((ed**2).mean()):.2e}", flush=True)
    assert np.all(ey <= np.abs(X) * dPhi + 3 * U * np.abs(X * Phi))
    assert np.all(ed <= dPhi + np.abs(X) * dens * (6 + X * X) * U + 4 * U)


def plain(p, x, t, dtype):
    """The same loss's gradient by torch on the CPU."""
    p = torch.tensor(p, dtype=dtype, requires_grad=True)
    x, t = torch.tensor(x, dtype=dtype), torch.tensor(t, dtype=dtype)
    gelu = torch.nn.functional.gelu
    h = gelu(x @ p[W1:B1].view(64, 9).T + p[B1:W2])
    h = gelu(h @ p[W2:B2].view(64, 64).T + p[B2:W3])
    y = h @ p[W3:B3].view(9, 64).T + p[B3:]
    ((y - t) ** 2).mean().backward()
    return p.grad.numpy().astype(np.float64)


@pytest.mark.parametrize("n", [1, 31, 33, 4096, 8193, 65537])
def test_gradient_beside_plain_binary32(n):
    """Each block of parameters at most four times as far from binary64 as
    torch's binary32 evaluation is, whose sums have as many terms (its error
    itself scatters by about that from one order of summation to another)."""
    print(f"case: gradient precision n={n}", flush=True)
    rng = np.random.default_rng(n + 5)
    p = (rng.standard_normal(END) * 0.3).astype(np.float32)
    x = rng.standard_normal((n, 9)).astype(np.float32)
    t = rng.standard_normal((n, 9)).astype(np.float32)
    net = L.Network(seed=1)
    net.set_params(p)
    _, g = net.loss_grad(x, t)
    net.close()
    exact, single = plain(p, x, t, torch.float64), plain(p, x, t, torch.float32)
    for a, b in ((W1, B1), (B1, W2), (W2, B2), (B2, W3), (W3, B3), (B3, END)):
        ours, torchs = np.linalg.norm(g[a:b] - exact[a:b]), np.linalg.norm(single[a:b] - exact[a:b])
        size = np.linalg.norm(exact[a:b])
        print(f"  {a}..{b}: {ours / size:.2e}, torch {torchs / size:.2e}", flush=True)
        assert ours <= 4 * torchs + 2 * U * size
