"""FP32 plans behind 64-bit figures (the reduced model with a reset, the gradient
sweeps' plans: Plan.keep_rounding) keep the direct (alpha, gamma) stages and the
Toeplitz or direct (k1, k2) DFTs: against the FP64 plan at the edges of those
kernels (B = 16 | 17, the FFT bandlimit 15; N = 32 | 34, 64; the smallest grids), and
the same plan's transforms before it keeps them, which take the MFMA forms.

Tolerance: relative L2 2e-5, the other FP32 tests' (a transform is about 2 N + 6 B
products deep, rounding below 300 * 6e-8 = 1.8e-5)."""
import math

import numpy as np
import pytest

import hpup

pytestmark = pytest.mark.gpu

WALL = dict(d=0.12, h=0.2, r=0.025, theta_t=5 * math.pi / 180, lambda_max=11.73, epsilon=0.8)


@pytest.mark.parametrize("dim,B,N", [(2, 3, 4), (2, 8, 16), (2, 15, 30), (2, 16, 32), (2, 16, 34), (2, 17, 20), (2, 6, 64),
                                     (3, 3, 4), (3, 10, 16), (3, 16, 12), (3, 17, 6)])
def test_against_fp64(dim, B, N):
    import torch
    print("case keep", dim, B, N, flush=True)
    g = torch.Generator(device="cpu").manual_seed(100 * B + N)
    out = {}
    kw = dict(b=(0.1, 0.2, 0.15), G=np.eye(dim) * 0.05, Jt=np.diag([1.0, 0.93539, 0.24935]), dt=0.002, method="rk4")
    f0 = None
    for precision in ("fp64", "fp32"):
        p = hpup.Plan(B, dim, N, 3.4 if dim == 2 else 12.0, precision=precision, **kw)
        if f0 is None:
            f0 = torch.rand(p.empty_grid().shape, generator=g, dtype=torch.float64)
        rt = torch.float64 if precision == "fp64" else torch.float32
        F = p.forward(f0.to(rt).cuda())
        b = p.backward(F, p.empty_grid())
        if dim == 3:
            p.keep_rounding()
        p.set_reset(**WALL, **(dict(tilt=0.1, jacobian=True) if dim == 3 else {}))
        H, f = F.clone(), p.empty_grid()
        p.hybrid_step(H, f, 1)
        torch.cuda.synchronize()
        out[precision] = [x.cpu().to(torch.complex128) for x in (F, b, H, f)]
        del p
    for name, a, c in zip(("forward", "backward", "hybrid F", "hybrid f"), out["fp64"], out["fp32"]):
        e = float(torch.linalg.vector_norm(a - c) / torch.linalg.vector_norm(a))
        print("  %s rel err %.2e" % (name, e), flush=True)
        assert e < 2e-5
