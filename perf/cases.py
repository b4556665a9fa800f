"""The work a user of this framework has it do, as measurable cases.

Every case goes through the public entry points (hpup.Plan, the gateway
functions, hpup.adjoint) on a density of the kind the drivers start from: a
mixture of matrix-Fisher x Gaussian components with seeded rotations, widths
and means.  Inputs are built from the seed with plain torch/numpy and have the
plan's own precision; exact() evaluates the same path from the same inputs in
64 bits, also with plain torch/numpy.

A case is a dict: kind, dim (omega dimension), B (bandlimit), N (omega points
per axis), precision, and for the gradient kinds the number of steps.
"""
import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hybridpendulum-up_amd"))
import hpup  # noqa: E402
from hpup.adjoint import Gradient, HybridGradient  # noqa: E402

DEV = "cuda" if torch.cuda.is_available() else "cpu"
C128, F64 = torch.complex128, torch.float64
JT = (1.0, 0.93539, 0.24935)  # scaled inertia of the 3-D pendulum
DAMP, NOISE = 0.2, 0.1
WALL = dict(d=0.12, h=0.2, r=0.025, theta_t=5 * math.pi / 180, lambda_max=100.0 * 0.1173)
EPS, TILT = 0.8, 0.2  # restitution coefficient; the 3-D law's wall tilt


# ------------------------------------------------------------------ cases --

def listed():
    def c(name, kind, dim, B, N, precision, **kw):
        return dict(name=name, kind=kind, dim=dim, B=B, N=N, precision=precision, **kw)
    return [
        # pure attitude densities (no omega grid), inverse then forward: the
        # smallest calls, a handful of short launches
        c("so3_b10_f64", "roundtrip", 0, 10, 1, "fp64"),
        # one RK4 step of the reduced model at the gradient workload's size,
        # as a filter's time loop calls it between its outputs
        c("step2_b10_n32_f64", "step", 2, 10, 32, "fp64"),
        # the same model through the MEX-style gateway: host arrays in and out
        # on every call, as the original drivers call it
        c("gateway2_b10_n32_f64", "gateway", 2, 10, 32, "fp64"),
        # parameter and initial-state gradients of the reduced model through
        # ten RK4 steps, checkpoint every five (measurement likelihoods)
        c("gradient2_b15_n30_f32", "gradient", 2, 15, 30, "fp32", steps=10, checkpoint=5),
        # one RK4 step of the 3-D pendulum, the propagation benchmark, in the
        # mixed-precision and the FP64 plan
        c("step3_b15_n30_f32", "step", 3, 15, 30, "fp32"),
        c("step3_b15_n30_f64", "step", 3, 15, 30, "fp64"),
        # its transforms: density output of the FP64 run, and the initial
        # density's coefficients in FP32
        c("inverse3_b15_n30_f64", "inverse", 3, 15, 30, "fp64"),
        c("forward3_b15_n30_f32", "forward", 3, 15, 30, "fp32"),
        # a bandlimit and omega grid between the drivers' own, both directions
        c("roundtrip3_b20_n18_f32", "roundtrip", 3, 20, 18, "fp32"),
        # one step of the large hybrid workload: RK4 step, inverse transform,
        # reflection reset on the grid, forward transform
        c("hybrid3_b30_n20_f32", "hybrid", 3, 30, 20, "fp32"),
        # one step of the reduced hybrid driver on its own grid, with the
        # statistics it stores after every step
        c("hybrid2_b30_n60_f64", "hybrid", 2, 30, 60, "fp64"),
        # restitution gradient through two hybrid steps of the 3-D pendulum
        # (3-D adjoint, transform adjoints, reset adjoint)
        c("hgrad3_b10_n16_f64", "hgrad", 3, 10, 16, "fp64", steps=2, checkpoint=1),
    ]


# per kind: omega dimensions, bandlimits, omega points per axis (dim 2, dim 3),
# precisions, and the largest grid (rotations x omega points) of a drawn case
_RANGES = {
    "roundtrip": ((0, 2, 3), (4, 30), (64, 30), ("fp64", "fp32"), 2.0e8),
    "inverse": ((2, 3), (4, 30), (64, 30), ("fp64", "fp32"), 4.0e8),
    "forward": ((2, 3), (4, 30), (64, 30), ("fp64", "fp32"), 4.0e8),
    "step": ((2, 3), (4, 30), (64, 32), ("fp64", "fp32", "fp32", "bf16x3"), 7.0e8),
    "hybrid": ((2, 3), (6, 30), (60, 20), ("fp64", "fp32"), 2.0e8),
    "gradient": ((2,), (4, 18), (32, 32), ("fp64", "fp32"), 1.0e9),
    "hgrad": ((3,), (4, 12), (16, 16), ("fp64", "fp32"), 6.0e7),
    "gateway": ((2,), (4, 12), (32, 32), ("fp64", "fp32"), 2.0e7),
}


def draw(rng):
    kind = rng.choice(("roundtrip", "inverse", "forward", "step", "step", "hybrid", "gradient", "hgrad", "gateway"))
    dims, (b0, b1), (n2, n3), precisions, most = _RANGES[kind]
    while True:
        dim = rng.choice(dims)
        B = rng.randint(b0, b1)
        N = 1 if dim == 0 else 2 * int(round(math.exp(rng.uniform(math.log(4), math.log((n2 if dim == 2 else n3) / 2)))))
        precision = rng.choice(precisions)
        if precision == "bf16x3" and N > 32:
            continue
        if 8 * B ** 3 * N ** dim <= most:
            break
    case = dict(kind=kind, dim=dim, B=B, N=N, precision=precision)
    if kind in ("gradient", "hgrad"):
        case["steps"] = rng.randint(2, 10) if kind == "gradient" else 2
        case["checkpoint"] = rng.choice((1, 5)) if kind == "gradient" else 1
    return case


# ------------------------------------------------------------------ model --

def _model(case):
    """Plan keywords of the case: the drivers' time steps and omega boxes."""
    dim = case["dim"]
    if case["kind"] in ("hybrid", "hgrad"):
        L, dt = (12.0, 0.003) if dim == 3 else (3.4, 0.0025)
    else:
        L, dt = 10.0, 0.004
    return dict(L=L, dt=dt, b=(DAMP,) * dim + (0.0,) * (3 - dim), G=np.eye(max(dim, 1)) * NOISE,
                Jt=np.diag(JT), method="rk4")


def _reset(case):
    return dict(WALL, epsilon=EPS, **(dict(tilt=TILT, jacobian=True) if case["dim"] == 3 else {}))


@functools.lru_cache(maxsize=4)
def _rows(B):
    """(l, m, n) of the compact rotation rows: m outermost, then l, then n."""
    r = [(l, m, n) for m in range(1 - B, B) for l in range(abs(m), B) for n in range(-l, l + 1)]
    return np.array(r, dtype=np.int64).T


@functools.lru_cache(maxsize=4)
def _quadrature(B):
    j = np.arange(2 * B)
    beta = math.pi / (4 * B) * (2 * j + 1)
    t = np.arange(B)
    s = (np.sin(np.outer(beta, 2 * t + 1)) / (2 * t + 1)).sum(axis=1)
    return beta, np.sin(beta) * s / (4 * B ** 3)


@functools.lru_cache(maxsize=4)
def _wigner(B):
    """d^l_mn(beta_j) as (B, 2B-1, 2B-1, 2B), zero off the triangle, from the
    spectral form of exp(-i beta J_y)."""
    beta, _ = _quadrature(B)
    d = np.zeros((B, 2 * B - 1, 2 * B - 1, 2 * B))
    for l in range(B):
        m = np.arange(-l, l)
        jp = np.diag(np.sqrt(l * (l + 1) - m * (m + 1)), -1)  # J_+ |m> = sqrt(..) |m + 1>
        _, v = np.linalg.eigh((jp - jp.T) / 2j)
        ph = np.exp(-1j * np.outer(np.arange(-l, l + 1), beta))
        s = slice(B - 1 - l, B + l)
        d[l, s, s] = np.einsum("ae,ej,be->abj", v, ph, v.conj(), optimize=True).real
    return d


def _angles(B):
    """e^{i m alpha_a} as (2B-1, 2B)."""
    return torch.as_tensor(np.exp(1j * math.pi / B * np.outer(np.arange(1 - B, B), np.arange(2 * B))), device=DEV)


def _rotations(B):
    """R(alpha, beta, gamma) = Rz Ry Rz on the grid, (9, (2B)^3) column-major
    matrices, alpha fastest."""
    a = math.pi / B * np.arange(2 * B)
    ca, sa = np.cos(a)[None, None, :], np.sin(a)[None, None, :]
    cb, sb = (g(_quadrature(B)[0])[None, :, None] for g in (np.cos, np.sin))
    cg, sg = np.cos(a)[:, None, None], np.sin(a)[:, None, None]
    one = np.ones((2 * B,) * 3)
    R = [ca * cb * cg - sa * sg, sa * cb * cg + ca * sg, -sb * cg * one, -ca * cb * sg - sa * cg,
         -sa * cb * sg + ca * cg, sb * sg * one, ca * sb * one, sa * sb * one, cb * one]
    return np.stack([np.broadcast_to(x, one.shape).reshape(-1) for x in R])


def _axis(N, L):
    return -L / 2 + L / N * np.arange(N)


def _components(case, seed):
    """Mixture components (weight, fR over the rotation grid, the omega
    Gaussian's factor along each axis): fR = exp(tr((U S)^T R))."""
    B, dim, N, L = case["B"], case["dim"], case["N"], _model(case)["L"]
    rng = np.random.default_rng(seed)
    R = torch.as_tensor(_rotations(B), device=DEV)
    out = []
    for weight in (0.6, 0.4):
        q, _ = np.linalg.qr(rng.standard_normal((3, 3)))
        q[:, 0] *= np.sign(np.linalg.det(q))
        s = np.array([10.0, 5.0, 1.0]) * rng.uniform(0.8, 1.2, 3) * min(1.0, B / 12)
        US = torch.as_tensor((q @ np.diag(s)).T.reshape(9).copy(), device=DEV)
        e = US @ R
        fR = torch.exp(e - e.max())
        sig, mu = L * rng.uniform(0.06, 0.12, max(dim, 1)), L * rng.uniform(-0.1, 0.1, max(dim, 1))
        fx = [torch.as_tensor(np.exp(-0.5 * ((_axis(N, L) - mu[a]) / sig[a]) ** 2), device=DEV) for a in range(dim)]
        w = torch.as_tensor(_quadrature(B)[1], device=DEV).view(1, -1, 1)
        mass = (fR.view(2 * B, 2 * B, 2 * B) * w).sum()
        for f in fx:
            mass = mass * f.sum() * (L / N)
        out.append((weight, fR / mass, fx))
    return out


def _outer(fx):
    """Product over the omega axes, the first axis fastest."""
    y = torch.ones(1, dtype=F64, device=DEV) if not fx else fx[0]
    for f in fx[1:]:
        y = torch.outer(f, y.reshape(-1)).reshape(-1)
    return y


def _density(case, seed):
    """Flat grid density, rotation index fastest, FP64."""
    f = None
    for weight, fR, fx in _components(case, seed):
        if f is None:
            f = torch.outer(_outer(fx) * weight, fR)
        else:
            f.addr_(_outer(fx) * weight, fR)
    return f.reshape(-1)


def _coefficients(case, seed):
    """Compact coefficients of the same density, complex128."""
    F = None
    for weight, fR, fx in _components(case, seed):
        FR = _forward(dict(case, dim=0, N=1), fR)
        X = [_dft(case["N"]) @ f.to(C128) for f in fx]
        x = (_outer(X) if X else torch.ones(1, dtype=C128, device=DEV)) * weight
        F = torch.outer(FR, x) if F is None else F.addr_(FR, x)
    return F.reshape(-1)


def _ctype(case):
    return C128 if case["precision"] == "fp64" else torch.complex64


def _rtype(case):
    return F64 if case["precision"] == "fp64" else torch.float32


# ---------------------------------------------------------------- prepare --

def prepare(case, seed):
    kind, dim, B, N = case["kind"], case["dim"], case["B"], case["N"]
    if kind == "gateway":
        return dict(kind=kind, args=_gateway_arrays(case, seed), f32=case["precision"] != "fp64")
    kw = _model(case)
    if kind in ("gradient", "hgrad"):
        F = _coefficients(case, seed).to(_ctype(case))
        g = _coefficients(case, seed + 1000003).to(_ctype(case))  # dJ/dF_K of a linear objective
        if kind == "gradient":
            h = Gradient(B, N, kw["L"], b=kw["b"][:2], G=kw["G"], dt=kw["dt"], method="rk4",
                         precision=case["precision"])
        else:
            h = HybridGradient(B, dim, N, kw["L"], _reset(case), b=kw["b"], G=kw["G"], Jt=kw["Jt"], dt=kw["dt"],
                               method="rk4", precision=case["precision"])
        return dict(kind=kind, h=h, F=F, g=g, steps=case["steps"], checkpoint=case["checkpoint"])
    p = hpup.Plan(B, dim, N, precision=case["precision"], **kw)
    s = dict(kind=kind, plan=p, stat=kind == "hybrid" and dim == 2)
    if kind == "forward":
        s["f"], s["F"] = _density(case, seed).to(_rtype(case)), p.empty_coeffs()
        return s
    s["F"] = _coefficients(case, seed).to(_ctype(case))
    if kind != "step":
        s["f"] = p.empty_grid()
    if kind == "roundtrip":
        s["out"] = p.empty_coeffs()
    if kind == "hybrid":
        p.set_reset(**_reset(case))
    return s


def _gateway_arrays(case, seed):
    """The arrays the drivers hold for pendulum_propagate_reduced: F in the
    full layout, X = fftn of the coordinates, the degree-1 gravity moment, u
    and the Clebsch-Gordan cells {l1, 1}."""
    B, N, kw = case["B"], case["N"], _model(case)
    dt = np.float64 if case["precision"] == "fp64" else np.float32
    ct = np.complex128 if case["precision"] == "fp64" else np.complex64
    M, lmax = 2 * B - 1, B - 1
    l, m, n = _rows(B)
    Fc = _coefficients(case, seed).cpu().numpy().reshape(-1, N, N)  # [r][k2][k1]
    F = np.zeros((M, M, B, N, N), dtype=ct, order="F")
    F[m + lmax, n + lmax, l] = Fc.transpose(0, 2, 1)
    ax = _axis(N, kw["L"])
    X = np.zeros((N, N, 2), dtype=ct, order="F")
    X[:, 0, 0] = np.fft.fft(ax) * N
    X[0, :, 1] = np.fft.fft(ax) * N
    MR = np.zeros((M, M, B, 2), dtype=ct, order="F")
    for p in range(2):
        for n2, v in _gravity(p):
            MR[lmax, lmax + n2, 1, p] = v / 3
    u = np.zeros((M, M, B, 3), dtype=ct, order="F")
    for ll in range(B):
        for nn in range(-ll, ll + 1):
            lo, hi = math.sqrt((ll + nn) * (ll - nn + 1)), math.sqrt((ll - nn) * (ll + nn + 1))
            if nn > -ll:
                u[nn - 1 + lmax, nn + lmax, ll, 0], u[nn - 1 + lmax, nn + lmax, ll, 1] = -0.5j * lo, 0.5 * lo
            if nn < ll:
                u[nn + 1 + lmax, nn + lmax, ll, 0], u[nn + 1 + lmax, nn + lmax, ll, 1] = -0.5j * hi, -0.5 * hi
            u[nn + lmax, nn + lmax, ll, 2] = -1j * nn
    CG = {}
    for l1 in range(B):
        nc = 3 * (2 * l1 + 1)
        cell = np.zeros((nc, nc), dtype=dt, order="F")
        for L2 in range(abs(l1 - 1), l1 + 2):
            for mm in range(-L2, L2 + 1):
                for m2 in (-1, 0, 1):
                    if abs(mm - m2) <= l1:
                        cell[(l1 + mm - m2) * 3 + 1 + m2, L2 * L2 - (1 - l1) ** 2 + L2 + mm] = _cg(l1, mm - m2, m2, L2)
        CG[(l1, 1)] = cell
    b = np.array(kw["b"][:2], dtype=dt)
    return [F, X, MR, b, kw["G"].astype(dt), kw["dt"], kw["L"], u, CG, "rk4"]


# -------------------------------------------------------------------- run --

def run(state):
    kind = state["kind"]
    if kind == "gateway":
        fn = hpup.pendulum_propagate_reduced32 if state["f32"] else hpup.pendulum_propagate_reduced
        return fn(*state["args"])
    if kind in ("gradient", "hgrad"):
        FK, gF, grads = state["h"].run(state["F"], state["steps"], lambda F: state["g"],
                                       checkpoint=state["checkpoint"])
        return {"F": FK, "gF": gF, "grads": grads}
    p = state["plan"]
    if kind == "step":
        return p.step(state["F"], 1)
    if kind == "inverse":
        return p.backward(state["F"], state["f"])
    if kind == "forward":
        return p.forward(state["f"], state["F"])
    if kind == "roundtrip":
        f = p.backward(state["F"], state["f"])
        return {"f": f, "F": p.forward(f, state["out"])}
    p.hybrid_step(state["F"], state["f"], 1)
    out = {"F": state["F"], "f": state["f"]}
    if state["stat"]:
        # the fit's frame-dependent moments (zero at the fit up to rounding)
        # and its iteration count are diagnostics and left out
        st = p.get_stat(state["f"], return_fx=True)
        out["stat"] = {k: st[k] for k in ("ER", "Ex", "Varx", "U", "S", "V", "Sigma", "fx")}
    return out


# ------------------------------------------------------------------- work --

def work(case):
    kind, dim, B, N = case["kind"], case["dim"], case["B"], case["N"]
    s = 16 if case["precision"] == "fp64" else 8
    nrc, nx = B * (4 * B * B - 1) // 3, N ** dim
    C, grid = nrc * nx, 8 * B ** 3 * nx
    # one derivative: a real circulant per omega axis product (4N flops a
    # coefficient), six rotation neighbours, the diagonal terms
    deriv = C * ((5 if dim == 3 else 4) * 4 * N + 6 * 18 + 40)
    # a transform: two angular FFTs of a real grid, the beta sums of half the
    # rows, the omega FFTs of half the rows
    xform = 2.5 * grid * math.log2(4 * B * B) + 4 * B * C + 2.5 * C * dim * math.log2(max(N, 2))
    if kind == "step":
        return {"bytes": 2 * C * s, "flops": 4 * deriv}
    if kind == "gateway":  # the full layout in and out
        return {"bytes": 2 * (2 * B - 1) ** 2 * B * nx * s, "flops": 4 * deriv}
    if kind in ("inverse", "forward"):
        return {"bytes": C * s + grid * s // 2, "flops": xform}
    if kind == "roundtrip":
        return {"bytes": 2 * C * s + grid * s // 2, "flops": 2 * xform}
    if kind == "hybrid":
        return {"bytes": 2 * C * s + grid * s // 2, "flops": 4 * deriv + 2 * xform}
    K = case["steps"]
    if kind == "gradient":  # F0, dJ in; F_K, dJ/dF0 out
        return {"bytes": 4 * C * s, "flops": K * 8 * deriv}
    return {"bytes": 4 * C * s, "flops": K * (8 * deriv + 4 * xform)}


# ------------------------------------------------------------------ exact --

def _dft(N, inverse=False):
    k = np.arange(N)
    e = np.exp((2j if inverse else -2j) * math.pi * (np.outer(k, k) % N) / N) / (N if inverse else 1)
    return torch.as_tensor(e, device=DEV)


def _apply(A, F, dim, N, axis):
    """The N x N matrix A along omega axis `axis` (0 fastest) of rows F."""
    y = F.reshape((-1,) + (N,) * dim)
    return torch.movedim(torch.matmul(torch.movedim(y, dim - axis, -1), A.T), -1, dim - axis).reshape(F.shape[0], -1)


def _omega(F, dim, N, inverse):
    for a in range(dim):
        F = _apply(_dft(N, inverse), F, dim, N, a)
    return F


def _gather_index(B):
    l, m, n = (torch.as_tensor(v, device=DEV) for v in _rows(B))
    return m + B - 1, n + B - 1, l


def _forward(case, f):
    """Grid (flat) -> coefficients (nrc * nx,), complex128."""
    B, dim, N = case["B"], case["dim"], case["N"]
    M, n2, nx = 2 * B - 1, 2 * B, N ** dim
    E = _angles(B)
    beta, w = _quadrature(B)
    W = torch.as_tensor(np.ascontiguousarray(_wigner(B).transpose(1, 2, 0, 3) * w), device=DEV).reshape(M * M, B, n2)
    im, ino, il = _gather_index(B)
    f = f.reshape(nx, n2, n2, n2)  # [x][gamma][j][alpha]
    parts, step = [], max(1, int(2e8 // (M * M * n2)))
    for x0 in range(0, nx, step):
        y = f[x0:x0 + step].to(C128) @ E.T  # [x][g][j][m]
        y = torch.matmul(E, y.permute(0, 2, 1, 3))  # [x][j][n][m]
        y = torch.view_as_real(y.permute(3, 2, 1, 0).contiguous()).reshape(M * M, n2, -1)  # [(m, n)][j][(x, re/im)]
        y = torch.view_as_complex(torch.bmm(W, y).reshape(M, M, B, -1, 2))
        parts.append(y[im, ino, il])
    F = parts[0] if len(parts) == 1 else torch.cat(parts, dim=1)
    return _omega(F, dim, N, False).reshape(-1)


def _inverse(case, F):
    """Coefficients -> grid (flat), float64 (the real part)."""
    B, dim, N = case["B"], case["dim"], case["N"]
    M, n2, nx = 2 * B - 1, 2 * B, N ** dim
    E = _angles(B).conj()
    W = torch.as_tensor(np.ascontiguousarray((_wigner(B) * (2 * np.arange(B) + 1)[:, None, None, None])
                                             .transpose(1, 2, 3, 0)), device=DEV).reshape(M * M, n2, B)
    im, ino, il = _gather_index(B)
    y = _omega(F.reshape(-1, nx), dim, N, True)
    parts, step = [], max(1, int(2e8 // (M * M * n2)))
    for x0 in range(0, nx, step):
        c = y[:, x0:x0 + step]
        full = torch.zeros((M, M, B, c.shape[1]), dtype=C128, device=DEV)
        full = full.index_put((im, ino, il), c)
        h = torch.bmm(W, torch.view_as_real(full).reshape(M * M, B, -1))
        h = torch.view_as_complex(h.reshape(M, M, n2, -1, 2)).permute(3, 2, 1, 0)  # [x][j][n][m]
        h = torch.matmul(E.T, h.contiguous()).permute(0, 2, 1, 3)  # [x][g][j][m]
        parts.append(torch.matmul(h, E).real.contiguous())
    f = parts[0] if len(parts) == 1 else torch.cat(parts, dim=0)
    return f.reshape(-1)


def _cg(j, mj, m2, J):
    """<j mj; 1 m2 | J mj + m2> (Condon-Shortley)."""
    M = mj + m2
    if abs(M) > J or abs(mj) > j:
        return 0.0
    if J == j + 1:
        d = (2 * j + 1) * (2 * j + 2) if m2 else (2 * j + 1) * (j + 1)
        v = {1: (j + M) * (j + M + 1), 0: (j - M + 1) * (j + M + 1), -1: (j - M) * (j - M + 1)}[m2]
        return math.sqrt(v / d)
    if J == j:
        d = 2 * j * (j + 1)
        if m2 == 0:
            return M / math.sqrt(j * (j + 1))
        return -math.sqrt((j + M) * (j - M + 1) / d) if m2 == 1 else math.sqrt((j - M) * (j + M + 1) / d)
    d = 2 * j * (2 * j + 1) if m2 else j * (2 * j + 1)
    v = {1: (j - M) * (j - M + 1), 0: (j - M) * (j + M), -1: (j + M + 1) * (j + M)}[m2]
    return -math.sqrt(v / d) if m2 == 0 else math.sqrt(v / d)


def _gravity(p):
    """3 x the degree-1 coefficients (n2, value), at m2 = 0, of R32 (p = 0) or
    -R31 (p = 1)."""
    s = 1 / math.sqrt(2)
    return ((-1, 1j * s), (1, 1j * s)) if p == 0 else ((-1, -s), (1, s))


class _Operator:
    """The drift of a model in 64 bits: rotation mixings as gathers, omega
    products as N x N matrices (DFT, coordinate, inverse DFT)."""

    def __init__(self, case, b, G):
        B, self.dim, self.N = case["B"], case["dim"], case["N"]
        L, dim, N = _model(case)["L"], self.dim, self.N
        l, m, n = _rows(B)
        at = {t: i for i, t in enumerate(zip(l.tolist(), m.tolist(), n.tolist()))}
        terms = []  # lists of (row, source, coefficient)
        for p in range(2):  # u_1, u_2
            t = []
            for (ll, mm, nn), r in at.items():
                for d in (1, -1):
                    if abs(nn + d) > ll:
                        continue
                    v = math.sqrt((ll - d * nn) * (ll + d * nn + 1))
                    t.append((r, at[ll, mm, nn + d], -0.5j * v if p == 0 else 0.5 * d * v))
            terms.append(t)
        terms.append([(r, r, -1j * nn) for (ll, mm, nn), r in at.items()])
        for p in range(2):  # gravity: coefficients of the product with R32 / -R31
            t = []
            for (ll, mm, nn), r in at.items():
                for l1 in (ll - 1, ll, ll + 1):
                    for n2, v in _gravity(p):
                        src = at.get((l1, mm, nn - n2))
                        if src is None:
                            continue
                        c = (2 * l1 + 1) / (2 * ll + 1) * _cg(l1, mm, 0, ll) * _cg(l1, nn - n2, n2, ll) * v
                        if c != 0:
                            t.append((r, src, c / (JT[p] if dim == 3 else 1.0)))
            terms.append(t)
        self.mix = [self._table(t, len(l)) for t in terms]
        x = torch.as_tensor(_axis(N, L), device=DEV)
        T = _dft(N) @ torch.diag(x.to(C128)) @ _dft(N, True)
        self.T = [T] * dim
        k = np.arange(N)
        k = np.where(k < N // 2, k, k - N)
        kc = 2 * math.pi / L * np.where(k == -(N // 2), 0, k)
        kd = -(2 * math.pi / L * k) ** 2
        grid = lambda v, a: torch.as_tensor(v, device=DEV).reshape((N,) + (1,) * a).expand((N,) * (a + 1)) \
            .reshape((1,) * (dim - 1 - a) + (N,) * (a + 1)).expand((N,) * dim).reshape(-1)
        self.kc = [grid(kc, a) for a in range(dim)]
        self.kd = [grid(kd, a) for a in range(dim)]
        self.a = [(JT[(p + 1) % 3] - JT[(p + 2) % 3]) / JT[p] for p in range(3)] if dim == 3 else []
        self.b, self.G = b, G

    @staticmethod
    def _table(terms, nrow):
        cnt = [0] * nrow
        width = 0
        for r, _, _ in terms:
            cnt[r] += 1
            width = max(width, cnt[r])
        src, cf, cnt = np.zeros((width, nrow), np.int64), np.zeros((width, nrow), np.complex128), [0] * nrow
        for r, s, c in terms:
            src[cnt[r], r], cf[cnt[r], r] = s, c
            cnt[r] += 1
        return [(torch.as_tensor(s, device=DEV), torch.as_tensor(c, device=DEV)[:, None]) for s, c in zip(src, cf)]

    def _mix(self, i, F):
        out = None
        for s, c in self.mix[i]:
            y = F[s] * c
            out = y if out is None else out + y
        return out

    def __call__(self, F):
        dim, N = self.dim, self.N
        TF = [_apply(self.T[p], F, dim, N, p) for p in range(dim)]
        dF = 0
        for p in range(dim):
            dF = dF - _apply(self.T[p], self._mix(p, F), dim, N, p)
            dF = dF + (1j * self.kc[p] * self.b[p]) * TF[p]
            if dim == 3:
                dF = dF - (1j * self.kc[p] * self.a[p]) * _apply(self.T[(p + 1) % 3], TF[(p + 2) % 3], dim, N, (p + 1) % 3)
            if p < 2:
                dF = dF - (1j * self.kc[p]) * self._mix(3 + p, F)
        D = 0
        for i in range(dim):
            for j in range(dim):
                D = D + self.G[i, j] * (self.kd[i] if i == j else -self.kc[i] * self.kc[j])
        return dF + D * F

    def rk4(self, F, dt):
        """One step of P(dt A), P the fourth-order Taylor polynomial."""
        F = F.reshape(len(self.mix[2][0][0]), -1)
        y = F
        for j in (4, 3, 2, 1):
            y = F + (dt / j) * self(y)
        return y.reshape(-1)


def _operator(case, b=None, G=None):
    dim = case["dim"]
    b = torch.full((dim,), DAMP, dtype=F64, device=DEV) if b is None else b
    return _Operator(case, b, torch.eye(dim, dtype=F64, device=DEV) * NOISE if G is None else G)


def _reset_rows(case):
    """The collision region and its geometry (host, FP64)."""
    B, dim = case["B"], case["dim"]
    d, h, r, tt, lm = (WALL[k] for k in ("d", "h", "r", "theta_t", "lambda_max"))
    ew = (math.cos(TILT), 0.0, math.sin(TILT)) if dim == 3 else (1.0, 0.0, 0.0)
    R = _rotations(B)
    th = np.arcsin(R[6] * ew[0] + R[7] * ew[1] + R[8] * ew[2])
    th0 = math.asin(d / math.sqrt(h * h + r * r)) - math.asin(r / math.sqrt(h * h + r * r))
    rows = np.nonzero(th >= th0 - tt)[0]
    R, th = R[:, rows], th[rows]
    lam = np.where(th > th0 + tt, lm, lm / 2 * np.sin(math.pi / (2 * tt) * (th - th0)) + lm / 2)
    PC = np.stack([(h - r * np.tan(th)) * R[6 + a] + r / np.cos(th) * ew[a] for a in range(3)])
    t = np.stack([R[7] * ew[2] - R[8] * ew[1], R[8] * ew[0] - R[6] * ew[2], R[6] * ew[1] - R[7] * ew[0]])
    t = t / np.sqrt((t ** 2).sum(axis=0))
    sigma = np.stack([PC[1] * ew[2] - PC[2] * ew[1], PC[2] * ew[0] - PC[0] * ew[2], PC[0] * ew[1] - PC[1] * ew[0]])
    g = lambda v: torch.as_tensor(v, device=DEV)
    return g(rows), g(R), g(t), g((sigma * t).sum(axis=0)), g(lam)


def _jump(case, f, eps):
    """f + dt df of the reset law on the flat grid f, differentiable in f and
    eps (the masks held fixed)."""
    B, dim, N, L, dt = case["B"], case["dim"], case["N"], _model(case)["L"], _model(case)["dt"]
    nx = N ** dim
    f = f.reshape(nx, -1)
    rows, R, t, sigma, lam = _reset_rows(case)
    h, x0 = L / N, -L / 2
    ax = torch.as_tensor(_axis(N, L), device=DEV)
    ix = torch.arange(nx, device=DEV)
    Om = [ax[(ix // N ** a) % N][:, None] for a in range(dim)]
    parts, step = [], max(1, int(4e7 // nx))
    for k in range(0, len(rows), step):
        s = slice(k, k + step)
        Rk, tk, fk = R[:, s], t[:, s], f[:, rows[s]]
        w = [sum(Rk[a + 3 * c] * Om[c] for c in range(dim)) for a in range(3)]
        dot = sum(w[a] * tk[a] for a in range(3))
        vq = sigma[s] * dot
        fac = (1 + eps) / eps * dot
        w = [w[a] - fac * tk[a] for a in range(3)]
        Oo = [sum(Rk[3 * a + c] * w[c] for c in range(3)) for a in range(dim)]
        if dim == 3:  # outflow and inflow on the two sides of the switching plane
            out_on, in_on = vq > 0, vq < 0
        else:  # the reduced law counts the plane itself on both sides
            out_on, in_on = vq >= 0, vq <= 0
        cell, frac = [], []
        for a in range(dim):
            c = torch.floor((Oo[a].detach() - x0) / h)
            if dim == 3:
                in_on = in_on & (c >= -1) & (c <= N - 1)
            else:
                o = Oo[a].detach()
                in_on = in_on & (o >= ax[0] + 1e-10) & (o <= ax[-1] - 1e-10) & (c >= 0) & (c <= N - 2)
            cell.append(c.to(torch.int64).clamp(-1, N - 1))
            frac.append((Oo[a] - (x0 + h * c)) / h)
        v = 0
        for q in range(2 ** dim):
            wt, j, inside = 1.0, 0, in_on
            for a in range(dim):
                up = (q >> a) & 1
                wt = wt * (frac[a] if up else 1 - frac[a])
                ja = cell[a] + up
                inside = inside & (ja >= 0) & (ja < N)
                j = j + ja.clamp(0, N - 1) * N ** a
            v = v + torch.where(inside, wt * torch.gather(fk, 0, j), torch.zeros((), dtype=F64, device=DEV))
        J = 1 / eps if dim == 3 else 1.0
        parts.append(fk + dt * lam[s] * (J * v - torch.where(out_on, fk, torch.zeros((), dtype=F64, device=DEV))))
    if not parts:
        return f.reshape(-1)
    return f.index_copy(1, rows, torch.cat(parts, dim=1)).reshape(-1)


def _moments(case, f):
    """get_stat's grid sums: E[R], E[x], Var[x] and the omega marginal."""
    B, dim, N, L = case["B"], case["dim"], case["N"], _model(case)["L"]
    nx, n2 = N ** dim, 2 * B
    w = torch.as_tensor(_quadrature(B)[1], device=DEV).view(1, n2, 1).expand(n2, n2, n2).reshape(-1)
    f = f.reshape(nx, -1)
    dv = (L / N) ** dim
    fx = f @ w
    ER = (torch.as_tensor(_rotations(B), device=DEV) @ (f.sum(dim=0) * w)) * dv
    ix = np.arange(nx)
    x = torch.as_tensor(np.stack([_axis(N, L)[(ix // N ** a) % N] for a in range(dim)]), device=DEV)
    Ex = (x @ fx) * dv
    Varx = (x * fx) @ x.T * dv - torch.outer(Ex, Ex)
    return {"ER": ER.reshape(3, 3).T.cpu().numpy(), "Ex": Ex.cpu().numpy(), "Varx": Varx.cpu().numpy(),
            "fx": fx.reshape((N,) * dim).permute(*reversed(range(dim))).cpu().numpy()}


def exact(case, seed):
    kind, dim, dt = case["kind"], case["dim"], _model(case)["dt"]
    if kind == "forward":
        return _forward(case, _density(case, seed).to(_rtype(case)).to(F64))
    F = _coefficients(case, seed).to(_ctype(case)).to(C128)
    if kind in ("gradient", "hgrad"):
        b = torch.full((dim,), DAMP, dtype=F64, device=DEV).requires_grad_(kind == "gradient")
        G = (torch.eye(dim, dtype=F64, device=DEV) * NOISE).requires_grad_(kind == "gradient")
        eps = torch.tensor(EPS, dtype=F64, device=DEV).requires_grad_(kind == "hgrad")
        g = _coefficients(case, seed + 1000003).to(_ctype(case)).to(C128)
        F0 = F.requires_grad_(True)
        A, y = _operator(case, b, G), F0
        for _ in range(case["steps"]):
            y = A.rk4(y, dt)
            if kind == "hgrad":
                y = _forward(case, _jump(case, _inverse(case, y), eps))
        torch.sum(torch.view_as_real(y) * torch.view_as_real(g)).backward()
        grads = ({"b": b.grad.cpu().numpy(), "G": G.grad.cpu().numpy()} if kind == "gradient"
                 else {"epsilon": float(eps.grad)})
        return {"F": y.detach(), "gF": F0.grad, "grads": grads}
    with torch.no_grad():
        if kind == "step":
            return _operator(case).rk4(F, dt)
        if kind == "inverse":
            return _inverse(case, F)
        if kind == "roundtrip":
            f = _inverse(case, F)
            return {"f": f, "F": _forward(case, f)}
        if kind == "gateway":
            B, N = case["B"], case["N"]
            y = _operator(case).rk4(F, dt).reshape(-1, N, N).cpu().numpy()
            l, m, n = _rows(B)
            full = np.zeros((2 * B - 1, 2 * B - 1, B, N, N), dtype=np.complex128, order="F")
            full[m + B - 1, n + B - 1, l] = y.transpose(0, 2, 1)
            return full
        y = _operator(case).rk4(F, dt)
        f = _jump(case, _inverse(case, y), torch.tensor(EPS, dtype=F64, device=DEV))
        out = {"F": _forward(case, f), "f": f}
        if dim == 2:
            out["stat"] = dict(_moments(case, f), U=None, S=None, V=None, Sigma=None)
        return out
