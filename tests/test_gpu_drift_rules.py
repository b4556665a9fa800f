"""The folded drift kernels' rules at their edge: real circulants that are odd, or
equal on both axes, only to 9e-13 of their largest entry.  FP64 gateway calls must
apply them as they are given, not their odd part or the first axis': the step then
differs by 6e-13 to 1.5e-12 (computed with the oracle, a step of size 1e3 that leaves the
derivative alone).

Tolerance: a derivative sums at most 6 N + 30 products: 270 * 1.1e-16 = 3e-14."""
import numpy as np
import pytest

import hpup
import oracle as O
from helpers import density, omega_grid, operators, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [20, 40])
@pytest.mark.parametrize("kind", ["even part", "axes"])
def test_circulants_at_the_edge(kind, N):
    print("case edge", kind, N, flush=True)
    B, L, dt = 3, 8.0, 1e3
    b, G = np.array([0.2, 0.3]), np.array([[0.1, 0.03], [0.02, 0.15]])
    f = density(B, 2, N, L, (8, 4, 2), seed=N, Sigma=np.eye(2) * 1.2)
    _, _, _, w = O.grid(B)
    F = O.fft_forward(B, f, O.wigner_table(B), w, 2, N)
    X, _, MR, u, cells = operators(B, 2, N, L)
    x = omega_grid(2, N, L)
    Xg = X.copy()
    if kind == "axes":
        Xg[..., 1] *= 1 + 0.9e-12
    else:
        mx = np.abs(np.fft.fft(x[0][:, 0]) / N).max()
        for p in range(2):
            Xg[..., p] = np.fft.fftn(x[p] + 0.9e-12j * mx * np.cos(2 * np.pi * x[p] / L))
    ref = O.integrate(B, 2, N, F, Xg, None, MR, b, G, dt, L, u, cells, "euler")
    plain = O.integrate(B, 2, N, F, X, None, MR, b, G, dt, L, u, cells, "euler")
    assert rel_l2(plain, ref) > 3e-13  # the difference that the call must not lose
    out = hpup.pendulum_propagate_reduced(F, Xg, MR, b, G, dt, L, u, cells, "euler")
    e = rel_l2(out, ref)
    print("  %.2e" % e, flush=True)
    assert e < 3e-14
