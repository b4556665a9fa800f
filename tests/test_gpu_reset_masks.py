"""The row-group reset kernels where their short form of the pull-back (s . y in
body coordinates) decides a mask at rounding level: walls and grids on which
many omega points lie on the switching plane (omega . t = 0) or, in dim 2, map
onto an edge of the interpolation box; against the oracle's law, which decides
them in its own chain of operations.  Tolerances as the other reset tests: the
jump term to 1e-12 (FP64 rounding of a few dozen operations), FP32 to 2e-6."""
import math

import numpy as np
import pytest

import hpup
import oracle as O
from helpers import rel_l2

pytestmark = pytest.mark.gpu
WALL = dict(d=0.12, h=0.2, r=0.025, theta_t=5 * math.pi / 180, lambda_max=11.73)


def _omega(dim, N, L):
    ax = -L / 2 + L / N * np.arange(N)
    return np.stack(np.meshgrid(*([ax] * dim), indexing="ij"))


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("fp32", 2e-6)])
@pytest.mark.parametrize("B,dim,N,L,eps,tilt", [(6, 3, 8, 12.0, 0.8, 0.0), (6, 3, 10, 4.0, 1.0, 0.2), (4, 3, 2, 3.0, 0.5, 0.0),
                                                (6, 2, 12, 3.4, 1.0, 0.0), (8, 2, 16, 4.0, 0.8, 0.0), (5, 2, 34, 3.4, 0.5, 0.0)])
def test_reset_masks(B, dim, N, L, eps, tilt, precision, tol):
    import torch
    print("case", B, dim, N, eps, precision, flush=True)
    rng = np.random.default_rng(B * N)
    real = np.float64 if precision == "fp64" else np.float32
    n2 = 2 * B
    f = np.asfortranarray(rng.random((n2,) * 3 + (N,) * dim).astype(real).astype(np.float64))
    R = O.rotations(B)
    if dim == 3:
        lam, PC, t = O.reset3_tables(B, R, WALL["d"], WALL["h"], WALL["r"], WALL["theta_t"], WALL["lambda_max"], tilt)
        df = O.reset3_df(B, N, L, R, f, lam, PC, t, eps, tilt, True)
    else:
        x = _omega(2, N, L)
        lc, ind, lists, PC = O.getLambda_compact(B, N, R, x, *(WALL[k] for k in ("d", "h", "r", "theta_t", "lambda_max")))[:4]
        Om = O.getOmega(B, N, R, x, ind, eps, PC, "old")
        ii, co = O.getIndRule(N, x, Om)
        df = O.discrete_nonoise(B, N, f, lc, ind, lists, ii, co)
    p = hpup.Plan(B, dim, N, L, precision=precision)
    p.set_reset(**WALL, epsilon=eps, **(dict(tilt=tilt, jacobian=True) if dim == 3 else {}))
    assert len(p.reset_rows) > 0
    fd = torch.from_numpy(f.ravel(order="F").astype(real)).cuda()
    out = p.reset(fd, mode=1)
    torch.cuda.synchronize()
    assert rel_l2(out.cpu().numpy().astype(np.float64), np.asarray(df).ravel(order="F")) < tol
    # the transpose has the same masks: <R f, g> = <f, R^H g>
    g = torch.from_numpy(rng.random(f.size).astype(real)).cuda()
    rhg = p.reset_adjoint(g, scale=1.0) - g
    torch.cuda.synchronize()
    a, b = torch.dot(out.double(), g.double()).item(), torch.dot(fd.double(), rhg.double()).item()
    scale = torch.dot(out.double().abs(), g.double()).item()
    assert abs(a - b) < tol * scale


@pytest.mark.parametrize("dim,N,L,tilt", [(3, 8, 12.0, 0.0), (3, 10, 4.0, 0.2), (2, 12, 3.4, 0.0)])
def test_restitution_derivative_on_cell_faces(dim, N, L, tilt):
    """dR/d eps at eps = 1 and 0.5, where the pull-back takes many omega points to
    cell faces (the interpolant's derivative jumps there): the row-group kernel
    picks the cells the per-point kernel picks.  FP64, 1e-11 of the sum of the
    terms' magnitudes (both sum the same terms in other orders)."""
    import torch
    B = 6
    rng = np.random.default_rng(N)
    for eps in (1.0, 0.5):
        kw = dict(WALL, epsilon=eps, **(dict(tilt=tilt, jacobian=True) if dim == 3 else {}))
        p = hpup.Plan(B, dim, N, L, precision="fp64")
        p.set_reset(**kw)
        f, g = (torch.from_numpy(rng.random(p.ngrid)).cuda() for _ in range(2))
        acc = torch.zeros(1, dtype=torch.float64, device="cuda")
        p.reset_eps_grad(f, g, acc)
        torch.cuda.synchronize()
        ref, mag = _deps_reference(B, dim, N, L, eps, tilt, f.cpu().numpy(), g.cpu().numpy(), p.reset_rows)
        assert abs(acc.item() - ref) < 1e-11 * mag, (eps, acc.item(), ref)


def _deps_reference(B, dim, N, L, eps, tilt, f, g, rows):
    """<g, (dR/d eps) f> in the law's chain of operations (numpy, FP64)."""
    n2, nx = 2 * B, N ** dim
    R = O.rotations(B).reshape(9, -1, order="F")
    f, g = f.reshape(nx, -1), g.reshape(nx, -1)
    d, h, r, tt, lm = (WALL[k] for k in ("d", "h", "r", "theta_t", "lambda_max"))
    ew = (math.cos(tilt), 0.0, math.sin(tilt)) if dim == 3 else (1.0, 0.0, 0.0)
    th0 = math.asin(d / math.sqrt(h * h + r * r)) - math.asin(r / math.sqrt(h * h + r * r))
    hx, x0 = L / N, -L / 2
    ix = np.arange(nx)
    xg = -L / 2 + L / N * np.arange(N)
    Lg = xg[-1] - xg[0] + (xg[1] - xg[0])  # getIndRule's box length (dim 2)
    Om = [xg[(ix // N ** a) % N] for a in range(dim)] + [np.zeros(nx)] * (3 - dim)
    J, dJ = (1 / eps, -1 / eps ** 2) if dim == 3 else (1.0, 0.0)
    tot, mag = 0.0, 0.0
    for k in rows:
        Rk = R[:, k]
        th = math.asin(Rk[6] * ew[0] + Rk[7] * ew[1] + Rk[8] * ew[2]) if dim == 3 else math.asin(Rk[6])
        lam = lm if th > th0 + tt else lm / 2 * math.sin(math.pi / (2 * tt) * (th - th0)) + lm / 2
        PC = [(h - r * math.tan(th)) * Rk[6 + a] + r / math.cos(th) * ew[a] for a in range(3)]
        c = [Rk[7] * ew[2] - Rk[8] * ew[1], Rk[8] * ew[0] - Rk[6] * ew[2], Rk[6] * ew[1] - Rk[7] * ew[0]]
        nc = math.sqrt(c[0] * c[0] + c[1] * c[1] + c[2] * c[2])
        t = [v / nc for v in c]
        w = [Rk[a] * Om[0] + Rk[a + 3] * Om[1] + Rk[a + 6] * Om[2] for a in range(3)]
        if dim == 2:
            w = [Rk[a] * Om[0] + Rk[a + 3] * Om[1] for a in range(3)]
        kf = (1 + eps) / eps
        if dim == 3:
            P = [PC[1] * ew[2] - PC[2] * ew[1], PC[2] * ew[0] - PC[0] * ew[2], PC[0] * ew[1] - PC[1] * ew[0]]
            sigma = P[0] * t[0] + P[1] * t[1] + P[2] * t[2]
            dot = w[0] * t[0] + w[1] * t[1] + w[2] * t[2]
            on = sigma * dot < 0
            fac = kf * dot
            w = [w[a] - fac * t[a] for a in range(3)]
        else:
            dot = w[1] * t[1] + w[2] * t[2]
            fac = kf * dot
            w = [w[0], w[1] - fac * t[1], w[2] - fac * t[2]]
            on = ~(w[1] * PC[2] - w[2] * PC[1] < 0)
        Oo = [Rk[3 * a] * w[0] + Rk[3 * a + 1] * w[1] + Rk[3 * a + 2] * w[2] for a in range(dim)]
        cell, s, ds = [], [], []
        for a in range(dim):
            if dim == 3:
                cf = np.floor((Oo[a] - x0) * (1.0 / hx))
                on = on & (cf >= -1) & (cf <= N - 1)
                rt = Rk[3 * a] * t[0] + Rk[3 * a + 1] * t[1] + Rk[3 * a + 2] * t[2]
            else:
                lo, hi = xg[0] + 1e-10, xg[-1] - 1e-10
                on = on & ~((Oo[a] < lo) | (Oo[a] > hi))
                cf = np.floor((Oo[a] / Lg + 0.5) * N)
                on = on & (cf >= 0) & (cf <= N - 2)
                rt = Rk[3 * a + 1] * t[1] + Rk[3 * a + 2] * t[2]
            cf = np.clip(cf, -1, N - 1)
            cell.append(cf.astype(int))
            s.append((Oo[a] - (x0 + hx * cf)) / hx)
            ds.append(dot * rt / hx / eps ** 2)
        I, dI = np.zeros(nx), np.zeros(nx)
        for q in range(2 ** dim):
            j, inside = np.zeros(nx, int), on.copy()
            u, du = [], []
            for a in range(dim):
                b = (q >> a) & 1
                ja = cell[a] + b
                inside &= (ja >= 0) & (ja < N)
                j += np.clip(ja, 0, N - 1) * N ** a
                u.append(s[a] if b else 1 - s[a])
                du.append(ds[a] if b else -ds[a])
            fq = np.where(inside, f[j, k], 0.0)
            I += np.prod(u, axis=0) * fq
            for a in range(dim):
                dI += np.prod([du[b] if b == a else u[b] for b in range(dim)], axis=0) * fq
        term = g[:, k] * lam * np.where(on, dJ * I + J * dI, 0.0)
        tot += term.sum()
        mag += np.abs(term).sum()
    return tot, mag
