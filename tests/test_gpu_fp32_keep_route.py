"""Which kernels an FP32 plan runs before and after it keeps its rounding
(Plan.keep_rounding, or set_reset in the reduced model), by the kernel names the plan
reports and by its bits: a plan that keeps through either call, at any time, gives
the same bits as one that did from the start, a plan that does not keep gives other
ones, and the gradient classes' plans keep.  Equal bits: the same kernels on the same
inputs, none of which depends on timing."""
import math

import numpy as np
import pytest

import hpup
from hpup.adjoint import Gradient, HybridGradient

pytestmark = pytest.mark.gpu

WALL = dict(d=0.12, h=0.2, r=0.025, theta_t=5 * math.pi / 180, lambda_max=11.73, epsilon=0.8)
JT = np.diag([1.0, 0.93539, 0.24935])


def _plan(dim, B, N, precision="fp32"):
    return hpup.Plan(B, dim, N, 3.4 if dim == 2 else 12.0, b=(0.1, 0.2, 0.15), G=np.eye(dim) * 0.05, Jt=JT, dt=0.002,
                     method="rk4", precision=precision)


def _drift(p):
    import torch
    F = torch.zeros(p.ncoef, dtype=p.cdtype, device="cuda")
    return [n for n, _, _ in p.profile(F, 1)][-1]


def _run(p, f):
    import torch
    F = p.forward(f)
    b = p.backward(F, p.empty_grid())
    S = p.step(F.clone(), 2)
    torch.cuda.synchronize()
    return F, b, S


def _same(a, b):
    import torch
    return [bool(torch.equal(x, y)) for x, y in zip(a, b)]


@pytest.mark.parametrize("dim,B,N,fast,kept", [(2, 6, 12, "k_drift_tile", "k_drift_fused_c"),
                                               (2, 5, 20, "k_drift_fold", "k_drift_fused_c"),
                                               (2, 18, 24, "k_drift_fold", "k_drift_fused"),
                                               (3, 4, 8, "k_drift_tile", "k_drift_fused_c"),
                                               (3, 3, 24, "k_drift_fold", "k_drift_fused")])
def test_route(dim, B, N, fast, kept):
    import torch
    print("case route", dim, B, N, flush=True)
    g = torch.Generator().manual_seed(B * N)
    p0 = _plan(dim, B, N)
    f = torch.rand(p0.ngrid, generator=g, dtype=torch.float32).cuda()
    assert _drift(p0) == fast
    plain = _run(p0, f)
    k = _plan(dim, B, N).keep_rounding()
    assert _drift(k) == kept
    want = _run(k, f)
    assert not any(_same(plain, want))
    # later, and twice
    assert all(_same(_run(p0.keep_rounding().keep_rounding(), f), want)) and _drift(p0) == kept
    # by the reset: the reduced model only
    r = _plan(dim, B, N)
    assert all(_same(_run(r, f), plain))
    r.set_reset(**WALL, **(dict(tilt=0.1, jacobian=True) if dim == 3 else {}))
    assert _drift(r) == (kept if dim == 2 else fast)
    assert all(_same(_run(r, f), want if dim == 2 else plain))
    # FP64 does not change
    d = _plan(dim, B, N, "fp64")
    a, name = _run(d, f.double()), _drift(d)
    assert all(_same(_run(d.keep_rounding(), f.double()), a)) and _drift(d) == name


def test_gradient_classes_keep():
    print("case gradient classes", flush=True)
    gr = Gradient(5, 20, 8.0, b=(0.3, 0.2), G=np.eye(2) * 0.1, dt=0.01, method="rk4", precision="fp32")
    assert _drift(gr.fwd) == "k_drift_fused_c"
    for dim, N in ((2, 12), (3, 8)):
        hg = HybridGradient(4, dim, N, 3.4 if dim == 2 else 12.0,
                            dict(WALL, **(dict(tilt=0.1, jacobian=True) if dim == 3 else {})), b=(0.1,) * 3,
                            G=np.eye(dim) * 0.05, Jt=JT, dt=0.002, method="rk4", precision="fp32")
        assert _drift(hg.fwd) == "k_drift_fused_c" and _drift(hg.adj) == "k_drift_fused"
