"""The omega DFTs of the plan transforms at the edges of the slab kernel's
tiles: omega counts around its K steps (N / 2 + 1 in steps of 4) and row tiles
(N = 30/32 and 62/64), several slabs per block with a last block partly
filled, the half-row and the all-rows paths (bandlimit 33; a 3-D grid of more
than 32 points).  Generic inputs against the FP64 oracle; tolerances as the
other transform tests: a few units of rounding over sums of at most 64 terms,
1e-12 (FP64) and 2e-6 (FP32)."""
import numpy as np
import pytest

import hpup
import oracle as O
from helpers import rel_l2, valid_mask

pytestmark = pytest.mark.gpu

CASES = [(3, 2, 2), (3, 2, 6), (3, 2, 8), (2, 2, 14), (3, 2, 16), (2, 2, 22), (3, 2, 30), (3, 2, 32), (2, 2, 34),
         (2, 2, 46), (2, 2, 62), (2, 2, 64), (3, 3, 2), (2, 3, 10), (2, 3, 32), (1, 3, 34), (33, 2, 2), (33, 3, 2)]


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("fp32", 2e-6)])
@pytest.mark.parametrize("B,dim,N", CASES)
def test_omega_dft_tile_edges(B, dim, N, precision, tol):
    import torch
    print("case", B, dim, N, precision, flush=True)
    rng = np.random.default_rng(1000 * B + N)
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
    fdev = torch.from_numpy(np.asfortranarray(f).ravel(order="F").astype(real)).cuda()
    Fd = p.forward(fdev)
    ref = O.fft_forward(B, np.asfortranarray(f), d, w, dim, N)
    assert rel_l2(p.download_full(Fd)[mask], ref[mask]) < tol
    Fu = p.upload_full(F)
    keep = Fu.clone()
    g = p.backward(Fu)
    torch.cuda.synchronize()
    assert torch.equal(Fu, keep)  # the inverse works on a copy
    assert rel_l2(g.cpu().numpy().astype(np.float64), O.fft_backward(B, F, d, dim, N).ravel(order="F")) < tol
