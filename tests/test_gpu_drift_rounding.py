"""The rounding of the FP32 drift operators.

Entries of the folded kernel (N = 18 to 30): B = 1 without noise leaves the damping
operators alone; on a unit impulse the derivative is a column of b_p c_p T_p, whose
entries reach the output through products with 1 and sums with 0.  Against the
FP64 plan's columns, relative in the Frobenius norm over all columns.  An entry is
the sum of an even and an odd part; each part rounded once and their sum rounded, in
that order on the host, gives 2.96e-8 to 3.76e-8 for these circulants (a device that
multiplies and adds rounded factors 4.4e-8 to 6.4e-8); bound 1.1 * 3.76e-8.  Such an
error is fixed, and grows with the steps.

One-tile kernel (N <= 16): the derivative's error against the FP64 plan's is that of
the unfolded kernel, which a plan that keeps its rounding runs: the same sums of the
same entries, each in an accumulator of its own, in another order; a geometric mean
over boxes and densities within 15 % of it."""
import numpy as np
import pytest

import hpup
from helpers import density

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [18, 20, 22, 24, 26, 28, 30])
def test_damping_entries(N):
    import torch
    print("case entries", N, flush=True)
    d, m = (hpup.Plan(1, 2, N, 10.0, b=(0.2, 0.2, 0.0), dt=0.004, method="rk4", precision=p) for p in ("fp64", "fp32"))
    num = den = 0.0
    for a in range(N * N):
        e = torch.zeros(N * N, dtype=torch.complex128, device="cuda")
        e[a] = 1.0
        x, y = d.derivative(e), m.derivative(e.to(torch.complex64)).to(torch.complex128)
        num += float((x - y).abs().pow(2).sum())
        den += float(x.abs().pow(2).sum())
    r = (num / den) ** 0.5
    print("  %.3e" % r, flush=True)
    assert r < 1.1 * 3.76e-8


@pytest.mark.parametrize("N", [8, 14, 16])
def test_one_tile_derivative(N):
    import torch
    print("case one tile", N, flush=True)
    ratio = []
    for L in (9.0, 10.0, 11.3):
        kw = dict(b=(0.2, 0.2, 0.0), G=np.eye(2) * 0.1, dt=0.004, method="rk4")
        d, m, k = (hpup.Plan(4, 2, N, L, precision=p, **kw) for p in ("fp64", "fp32", "fp32"))
        k.keep_rounding()
        for seed in range(2):
            f = density(4, 2, N, L, (6, 4, 1), seed=seed, Sigma=np.eye(2) * (0.8 + 0.3 * seed),
                        mu=np.arange(2) * 0.3 * (seed + 1))
            F = d.forward(torch.from_numpy(np.ascontiguousarray(f.ravel(order="F"))).cuda()).to(torch.complex64)
            x = d.derivative(F.to(torch.complex128))
            e = [float((p.derivative(F).to(torch.complex128) - x).norm()) for p in (m, k)]
            ratio.append(np.log(e[0] / e[1]))
    r = float(np.exp(np.mean(ratio)))
    print("  %.3f" % r, flush=True)
    assert r < 1.15
