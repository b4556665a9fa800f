"""The reduced model's reset at small restitution coefficients, where the rounding
of the pulled-back position grows with (1 + eps)/eps: the masks of omega points that
map onto an edge of the interpolation box are those of the law's own chain of
operations (here in Python's doubles, which are not contracted), not of the kernels'
short form.

The cases are searched for: a region row and an omega point with a small s . y, and
the eps between the one at which the chain lets the point cross the edge and the one
at which the short form does.  On a density of ones the jump term at a point is
lambda (in - out); 1e-6 lambda allows for the weights' sum."""
import math

import numpy as np
import pytest

import hpup

pytestmark = pytest.mark.gpu
WALL = dict(d=0.12, h=0.2, r=0.025, theta_t=5 * math.pi / 180, lambda_max=11.73)


def _geometry(B):
    """(iR, R, t, PC, lambda) of the region's rows."""
    n2 = 2 * B
    ca, sa = ([f(math.pi / B * i) for i in range(n2)] for f in (math.cos, math.sin))
    cb, sb = ([f(math.pi / (4.0 * B) * (2 * i + 1)) for i in range(n2)] for f in (math.cos, math.sin))
    d, h, r, tt, lm = (WALL[k] for k in ("d", "h", "r", "theta_t", "lambda_max"))
    hr = math.sqrt(h * h + r * r)
    th0 = math.asin(d / hr) - math.asin(r / hr)
    for iR in range(n2 ** 3):
        i, j, k = iR % n2, iR // n2 % n2, iR // (n2 * n2)
        a, s, b, t, c, u = ca[i], sa[i], cb[j], sb[j], ca[k], sa[k]
        R = [a * b * c - s * u, s * b * c + a * u, -t * c, -a * b * u - s * c, -s * b * u + a * c, t * u, a * t, s * t, b]
        th = math.asin(R[6])
        if th < th0 - tt:
            continue
        lam = lm if th > th0 + tt else lm / 2 * math.sin(math.pi / (2 * tt) * (th - th0)) + lm / 2
        lr3 = h - r * math.tan(th)
        PC = [lr3 * R[6] + r / math.cos(th), lr3 * R[7], lr3 * R[8]]
        nt = math.sqrt(R[7] * R[7] + R[8] * R[8])
        yield iR, R, [0.0, R[8] / nt, -R[7] / nt], PC, lam


def _chain(R, t, P, xg, eps, i0, i1):
    kf, lo, hi = (1.0 + eps) / eps, xg[0] + 1e-10, xg[-1] - 1e-10
    x1, x2 = xg[i0], xg[i1]
    o0, o1, o2 = R[0] * x1 + R[3] * x2, R[1] * x1 + R[4] * x2, R[2] * x1 + R[5] * x2
    out = not o1 * P[2] - o2 * P[1] < 0.0
    ot = kf * (o1 * t[1] + o2 * t[2])
    o1 -= ot * t[1]
    o2 -= ot * t[2]
    a0, a1 = R[0] * o0 + R[1] * o1 + R[2] * o2, R[3] * o0 + R[4] * o1 + R[5] * o2
    return out, not (o1 * P[2] - o2 * P[1] < 0.0 or a0 < lo or a0 > hi or a1 < lo or a1 > hi)


def _cases(B, N, L, want):
    xg = [-L / 2 + L / N * float(i) for i in range(N)]
    edges = (1e-10 * N / L, N - 1 - 1e-10 * N / L)
    y = np.arange(N) - N // 2
    found = []
    for iR, R, t, P, lam in _geometry(B):
        s = [R[3 * a] * t[0] + R[3 * a + 1] * t[1] + R[3 * a + 2] * t[2] for a in range(2)]
        dots = np.abs(s[0] * y[:, None] + s[1] * y)
        dots[dots < 1e-9] = 9.0
        m = int(np.argmin(dots))
        for i in ((m // N, m % N), ((N - m // N) % N, (N - m % N) % N)):
            dot = s[0] * (i[0] - N // 2) + s[1] * (i[1] - N // 2)
            for a in range(2):
                for e in edges:
                    if abs(dot * s[a]) < 1e-12 or (i[a] - e) / (dot * s[a]) < 1e4:
                        continue
                    eps = 1.0 / ((i[a] - e) / (dot * s[a]) - 1.0)
                    kf = (1.0 + eps) / eps
                    if not 0.5 < i[1 - a] - kf * dot * s[1 - a] < N - 1.5:
                        continue

                    def chain(x):
                        return _chain(R, t, P, xg, x, *i)[1]

                    def short(x):
                        return all(edges[0] <= i[b] - (1.0 + x) / x * dot * s[b] <= edges[1] for b in range(2))

                    def flip(f):
                        lo, hi = eps * (1 - 1e-9), eps * (1 + 1e-9)
                        f0 = f(lo)
                        if f(hi) == f0:
                            return None
                        for _ in range(70):
                            mid = (lo + hi) / 2
                            lo, hi = (mid, hi) if f(mid) == f0 else (lo, mid)
                        return hi

                    c, h = flip(chain), flip(short)
                    if c is None or h is None:
                        continue
                    mid = (c + h) / 2
                    if chain(mid) != short(mid):
                        found.append((abs(c - h) / eps * N, iR, i, mid, R, t, P, lam))
    found.sort(key=lambda v: -v[0])
    return xg, found[:want]


@pytest.mark.parametrize("B,N,L", [(10, 64, 3.4), (7, 62, 4.0)])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_edge_masks_at_small_epsilon(B, N, L, precision):
    import torch
    print("case small epsilon", B, N, precision, flush=True)
    xg, cases = _cases(B, N, L, 8)
    assert len(cases) == 8
    p = hpup.Plan(B, 2, N, L, precision=precision)
    f = torch.ones(p.ngrid, dtype=p.rdtype, device="cuda")
    wrong = []
    for _, iR, i, eps, R, t, P, lam in cases:
        p.set_reset(**WALL, epsilon=eps)
        out = p.reset(f, mode=1)
        torch.cuda.synchronize()
        o, n = _chain(R, t, P, xg, eps, *i)
        got = out[iR + (2 * B) ** 3 * (i[0] + N * i[1])].item()
        if abs(got - lam * (n - o)) > 1e-6 * lam:
            wrong.append((eps, iR, i, got / lam, n - o))
    print("  wrong:", wrong, flush=True)
    assert not wrong
