"""The parity-folded drift kernels (odd real circulants on even and odd parts) and
the one-wave kernel of grids up to 16 points, against the oracle at the edges of
their ranges: the smallest grids, 14 and 16 (a partial and a whole tile), 18, 20, 22 |
24, 30 (the folded kernel's tile depths and slab groups), the reduced model's FP64
kernel for 34 to 62 points at 34, 38 | 40, 42 | 44, 46 | 48 | 62 (one and two quartets a
thread), full diffusion matrices, inertias with and without gyroscopic terms,
several slabs per workgroup, a coordinate whose real circulant is not odd, which the
folding must not take, and axes of different circulants.

Tolerances: relative L2 1e-10 (FP64) and 2e-5 (FP32), as the other drift kernels'
tests: a derivative is sums of at most 6 N + 30 products, so FP32 rounding stays
below 210 * 6e-8 = 1.3e-5."""
import numpy as np
import pytest

import hpup
import oracle as O
from helpers import density, omega_grid, operators, rel_l2

pytestmark = pytest.mark.gpu

G2 = np.array([[0.1, 0.03], [0.02, 0.15]])
G3 = np.array([[0.1, 0.02, 0.01], [0.03, 0.2, -0.02], [0.015, 0.025, 0.05]])
BT = (0.2, 0.3, 0.25)
JT = {"gyro": np.diag([1.0, 0.93539, 0.24935]), "iso": np.eye(3)}


def _full(B, dim, N, L, seed):
    f = density(B, dim, N, L, (8, 4, 2), seed=seed, Sigma=np.eye(dim) * 1.2)
    _, _, _, w = O.grid(B)
    return O.fft_forward(B, f, O.wigner_table(B), w, dim, N)


CASES = [(2, N, "") for N in (2, 4, 6, 12, 14, 16, 18, 22, 24, 30)] + \
        [(3, N, "gyro") for N in (2, 4, 6, 8, 10, 14, 16, 18, 20, 22, 24, 30)] + [(3, 10, "iso"), (3, 24, "iso")]


@pytest.mark.parametrize("dim,N,inertia", CASES)
@pytest.mark.parametrize("precision,tol", [("fp64", 1e-10), ("fp32", 2e-5)])
def test_derivative_and_step(dim, N, inertia, precision, tol):
    """dF (the derivative-only epilogue) and two midpoint steps (both update
    epilogues)."""
    import torch
    print("case fold", dim, N, inertia, precision, flush=True)
    B, L, dt = (3 if dim == 2 else 2 if N > 14 else 8), 8.0, 0.004
    Jt = JT[inertia] if dim == 3 else None
    G, b = (G3 if dim == 3 else G2), np.array(BT[:dim])
    Ffull = _full(B, dim, N, L, 10 * N + dim)
    X, OJO, MR, u, cells = operators(B, dim, N, L, Jt)
    kw = {} if Jt is None else {"Jt": Jt}
    p = hpup.Plan(B, dim, N, L, b=BT if dim == 3 else (BT[0], BT[1], 0.0), G=G, dt=dt, method="midpoint",
                  precision=precision, **kw)
    F = p.upload_full(Ffull)
    dF = p.derivative(F)
    torch.cuda.synchronize()

    def dense(y):
        return O.derivative(B, dim, N, y, X, OJO, MR, b, G, L, u, cells)

    def structured(y, h, method):
        return O.integrate_structured(B, dim, N, y, X, Jt, MR, b, G, h, L, u, cells, method)

    big = dim == 3  # the dense oracle takes minutes there
    ref = (structured(Ffull, 1.0, "euler") - Ffull) if big else dense(Ffull)
    e = rel_l2(p.download_full(dF), ref)
    print("  derivative rel err %.2e" % e, flush=True)
    assert e < tol
    p.step(F, 2)
    torch.cuda.synchronize()
    y = Ffull
    for _ in range(2):
        y = structured(y, dt, "midpoint") if big else y + dt * dense(y + dt / 2 * dense(y))
    e = rel_l2(p.download_full(F), y)
    print("  two steps rel err %.2e" % e, flush=True)
    assert e < tol


@pytest.mark.parametrize("N", [34, 38, 40, 42, 44, 46, 48, 62])
def test_derivative_and_step_64(N):
    test_derivative_and_step(2, N, "", "fp64", 1e-10)


@pytest.mark.parametrize("N", [20, 40])
def test_axes_of_different_ramps(N):
    """X_2 of a ramp twice as steep: odd real circulants that differ by axis, which
    the 34 to 62 point kernel's shared matrices must not take."""
    print("case fold axes", N, flush=True)
    B, L, dt = 3, 8.0, 0.01
    Ffull = _full(B, 2, N, L, 60 + N)
    X, _, MR, u, cells = operators(B, 2, N, L)
    Xg = X.copy()
    Xg[..., 1] *= 2.0
    b = np.array(BT[:2])
    ref = O.integrate(B, 2, N, Ffull, Xg, None, MR, b, G2, dt, L, u, cells, "RK2")
    out = hpup.pendulum_propagate_reduced(Ffull, Xg, MR, b, G2, dt, L, u, cells, "RK2")
    e = rel_l2(out, ref)
    print("  rel err %.2e" % e, flush=True)
    assert e < 1e-10


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-10), ("fp32", 2e-5)])
def test_many_rows(precision, tol):
    """B = 12 (2300 rows): every workgroup walks several rows, which the walk's
    order permutes."""
    import torch
    print("case fold rows", precision, flush=True)
    B, N, L, dt = 12, 18, 8.0, 0.004
    Ffull = _full(B, 2, N, L, 7)
    X, _, MR, u, cells = operators(B, 2, N, L)
    ref = O.integrate_structured(B, 2, N, Ffull, X, None, MR, np.array(BT[:2]), G2, dt, L, u, cells, "RK4")
    p = hpup.Plan(B, 2, N, L, b=(BT[0], BT[1], 0.0), G=G2, dt=dt, method="RK4", precision=precision)
    F = p.upload_full(Ffull)
    p.step(F, 1)
    torch.cuda.synchronize()
    e = rel_l2(p.download_full(F), ref)
    print("  rel err %.2e" % e, flush=True)
    assert e < tol


@pytest.mark.parametrize("N", [14, 30])
def test_circulant_not_odd(N):
    """x + 0.3 i cos(2 pi x / L): the circulant's real part stays constant but
    its imaginary part is not odd."""
    print("case fold not odd", N, flush=True)
    B, L, dt = 3, 8.0, 0.01
    Ffull = _full(B, 2, N, L, 40 + N)
    X, _, MR, u, cells = operators(B, 2, N, L)
    x = omega_grid(2, N, L)
    Xg = np.zeros_like(X)
    for p in range(2):
        Xg[..., p] = np.fft.fftn(x[p] + 0.3j * np.cos(2 * np.pi * x[p] / L))
    b = np.array(BT[:2])
    ref = O.integrate(B, 2, N, Ffull, Xg, None, MR, b, G2, dt, L, u, cells, "RK2")
    out = hpup.pendulum_propagate_reduced(Ffull, Xg, MR, b, G2, dt, L, u, cells, "RK2")
    e = rel_l2(out, ref)
    print("  rel err %.2e" % e, flush=True)
    assert e < 1e-10


@pytest.mark.parametrize("dim,N,inertia", [(2, 2, ""), (2, 10, ""), (2, 14, ""), (2, 16, ""), (3, 2, "gyro"),
                                           (3, 8, "gyro"), (3, 14, "iso"), (3, 16, "gyro"), (3, 16, "iso")])
@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("fp32", 2e-5)])
def test_adjoint_one_wave(dim, N, inertia, precision, tol):
    """<A x, y> = <x, A^H y> for the operator and <P x, y> = <x, P^H y> for two midpoint
    steps, on grids of the one-wave kernel's adjoint form; relative to |A x| |y|, the
    bounds of the adjoint operators' own tests."""
    import torch
    print("case adjoint one wave", dim, N, inertia, precision, flush=True)
    kw = {} if dim == 2 else {"Jt": JT[inertia]}

    def plan(op):
        return hpup.Plan(4, dim, N, 8.0, b=BT if dim == 3 else (BT[0], BT[1], 0.0), G=G3 if dim == 3 else G2, dt=0.004,
                         method="midpoint", precision=precision, operator=op, **kw)

    A, AH = plan(0), plan(1)
    g = torch.Generator().manual_seed(10 * N + dim)

    def rand():
        v = torch.randn(2, A.ncoef, generator=g, dtype=torch.float64)
        return torch.complex(v[0], v[1]).to(A.cdtype).cuda()

    x, y = rand(), rand()
    for Ax, AHy in ((A.derivative(x), AH.derivative(y)), (A.step(x.clone(), 2), AH.step(y.clone(), 2))):
        lhs, rhs = complex(torch.vdot(Ax, y).item()), complex(torch.vdot(x, AHy).item())
        e = abs(lhs - rhs) / float(Ax.abs().pow(2).sum().sqrt() * y.abs().pow(2).sum().sqrt())
        print("  %.2e" % e, flush=True)
        assert e <= tol, (lhs, rhs)
