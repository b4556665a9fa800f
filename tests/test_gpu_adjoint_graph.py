"""Reverse stages under HIP graph capture: a captured adjoint_stage holds the
address of the plan's partial sums, which no later call of the plan may move.

The replays are compared with the eager stage: the same kernels on the same
inputs, so the outputs and the sums are equal bit for bit."""
import numpy as np
import pytest

import hpup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_captured_stage_before_adjoint_step(precision):
    """adjoint_stage (warm-up, then captured), adjoint_step, replays."""
    import torch
    print("case captured stage", precision, flush=True)
    kw = dict(b=(0.3, 0.2, 0.0), G=np.array([[0.12, 0.03], [0.05, 0.18]]), dt=0.02, method="rk4", precision=precision)
    fwd, adj = hpup.Plan(5, 2, 12, 8.0, **kw), hpup.Plan(5, 2, 12, 8.0, operator=1, **kw)
    g = torch.Generator().manual_seed(3)

    def rand():
        v = torch.randn(2, adj.ncoef, generator=g, dtype=torch.float64)
        return torch.complex(v[0], v[1]).to(adj.cdtype).cuda()

    ybar, y, lam, F = rand(), rand(), rand(), rand()
    out, fbar = torch.empty_like(y), torch.zeros_like(y)
    grad = torch.zeros(5, dtype=torch.float64, device="cuda")
    scale = 0.02

    def stage():
        adj.adjoint_stage(ybar, y, scale, grad, out=out, fbar=fbar, fbar_init=True)

    stage()
    torch.cuda.synchronize()
    ref_out, ref_fbar, ref_grad = out.clone(), fbar.clone(), grad.clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        stage()
    # the plan's next call needs the partial sums of four stages
    ys = [torch.empty_like(F) for _ in range(3)]
    fwd.step_stages(F, ys)
    acc = torch.zeros(5, dtype=torch.float64, device="cuda")
    adj.adjoint_step(F, ys, lam, acc)
    torch.cuda.synchronize()
    for _ in range(3):
        out.zero_()
        fbar.zero_()
        grad.zero_()
        other = torch.randn(1 << 20, device="cuda") * 2.0  # the program's own work between the replays
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref_out) and torch.equal(fbar, ref_fbar)
        assert torch.equal(grad, ref_grad), (grad, ref_grad)
        del other
    # and the sums of the step are what a fresh plan's are
    acc2 = torch.zeros_like(acc)
    hpup.Plan(5, 2, 12, 8.0, operator=1, **kw).adjoint_step(F, ys, lam, acc2)
    torch.cuda.synchronize()
    assert torch.equal(acc, acc2)
