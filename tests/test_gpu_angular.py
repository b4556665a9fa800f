"""The MFMA (alpha, gamma) stages of the plan transforms at the edges of their
tiles: bandlimits around the K steps (multiples of 4) and row tiles (16, 32),
omega counts that leave the last block of points partly empty, and a grid
tensor that starts off a vector boundary.  Inputs are generic (no bandlimit,
no Hermitian symmetry), against the FP64 oracle.  Tolerances: a K = 2B sum in
each of five stages, a few units of rounding: 1e-12 (FP64), 2e-6 (FP32)."""
import numpy as np
import pytest

import hpup
import oracle as O
from helpers import rel_l2, valid_mask

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("fp32", 2e-6)])
@pytest.mark.parametrize("B,dim,N", [(1, 2, 2), (2, 0, 1), (3, 2, 2), (4, 2, 6), (7, 2, 2), (8, 0, 1), (11, 2, 6),
                                     (12, 2, 4), (16, 2, 2), (17, 2, 6), (20, 2, 2), (23, 0, 1), (31, 2, 2), (32, 2, 2)])
def test_transforms_at_tile_edges(B, dim, N, precision, tol):
    import torch
    print("case", B, dim, N, precision, flush=True)
    rng = np.random.default_rng(100 * B + N)
    n2, M = 2 * B, 2 * B - 1
    om = (N,) * dim
    real = np.float64 if precision == "fp64" else np.float32
    f = rng.standard_normal((n2, n2, n2) + om).astype(real).astype(np.float64)
    F = rng.standard_normal((M, M, B) + om) + 1j * rng.standard_normal((M, M, B) + om)
    mask = np.broadcast_to(valid_mask(B, om), F.shape)
    F = np.asfortranarray(np.where(mask, F, 0))
    F = F if precision == "fp64" else F.astype(np.complex64).astype(np.complex128)
    d = O.wigner_table(B)
    _, _, _, w = O.grid(B)
    p = hpup.Plan(B, dim, N, 6.0, precision=precision)
    buf = torch.zeros(p.ngrid + 1, dtype=p.rdtype, device="cuda")
    off = 1 if precision == "fp32" else 0  # FP32: a start that is not a multiple of a pair
    fdev = buf[off:off + p.ngrid]
    fdev.copy_(torch.from_numpy(np.asfortranarray(f).ravel(order="F")))
    Fd = p.forward(fdev)
    ref = O.fft_forward(B, np.asfortranarray(f), d, w, dim, N)
    assert rel_l2(p.download_full(Fd)[mask], ref[mask]) < tol
    g = p.backward(p.upload_full(F), fdev)
    torch.cuda.synchronize()
    assert rel_l2(g.cpu().numpy().astype(np.float64), O.fft_backward(B, F, d, dim, N).ravel(order="F")) < tol
