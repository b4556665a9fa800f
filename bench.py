#!/usr/bin/env python3
"""Propagation steps/s of the spectral Fokker-Planck step on the 3-D pendulum,
SO(3) x R^3 with bandlimit B = 15 (30^3 rotation grid) and a 30^3 omega grid
over [-5, 5]^3, dt = 0.004, 200 steps, coefficients resident in HBM.

The integrator is RK4 (one step = four derivative evaluations): explicit
Euler, midpoint and RK2 are unstable on this advective spectrum within 200
steps (the FP64 solution itself grows by orders of magnitude), so the
precision gate would compare amplified rounding.  The mixed-precision path
(default --precision fp32) is timed next to the plain FP64 path from the same
initial coefficients, and its relative L2 error against the FP64 coefficients
is taken after the workload's 200 steps (propagated untimed when --steps
differs).  Prints one JSON line (the bench contract).
Single GPU: --gpus N > 1 exits with a message.
"""
import argparse
import json
import math
import os
import sys
import time

REPO = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(REPO, "hybridpendulum-up_amd"))

HBM_PEAK_GBS = 8000.0  # MI355X HBM3E
# MI355X dense MFMA peaks, TFLOP/s.  A 3xBF16 product (three-piece splits,
# the six products of order <= 2) costs six bf16 MFMAs, so its FP32-equivalent
# peak is a sixth of the bf16 one.
MFMA_PEAK_TFLOPS = {"fp32": 157.3, "fp64": 78.6, "bf16x3": 2500.0 / 6}

# HBM bytes per launch measured with rocprofv3 --pmc FETCH_SIZE and WRITE_SIZE
# (scaled by the copy-probe factors) for the kernels of this workload; the
# summaries are under profiles/.  None where not measured.
MEASURED_TRAFFIC = {
    ("k_drift_fused", "fp32", "RK4"): 5.085e9,   # profiles/k_drift_fused_B15_N30_RK4.md
    ("k_drift_fused", "fp64", "RK4"): 9.451e9,
    ("k_drift_fold", "fp32", "RK4"): 4.362e9,    # profiles/kernels_by_workload.md
    ("k_drift_fold", "fp64", "RK4"): 8.108e9,
}


def kernel_flops(name, B, N):
    """Algorithmic MFMA FLOPs per launch.  Each circulant along an omega axis
    acts on a (r, k3) slab of N^2 points; kappa_p = c0 + i (real circulant) for
    the coordinate ramps of this workload, so one application is two real
    N^3-MAC products (4 N^3 FLOPs) plus an axis sum.  The fused kernel applies
    four per slab (T1 F, T2 F, T1 V1, T2 V2), the axis-3 kernel one; the folded
    kernel applies the four to parity planes, half the products of each; nRc =
    B(2B-1)(2B+1)/3 rotation rows, N slabs each."""
    nrc = B * (2 * B - 1) * (2 * B + 1) // 3
    per = {"k_drift_fused": 4, "k_drift_fold": 2, "k_axis3_mfma": 1}.get(name, 0)
    return per * 4.0 * N ** 3 * nrc * N

ERR_STEPS = 200  # the workload's step count, at which the precision gate is taken

CFG = dict(B=15, dim=3, N=30, L=10.0, b=(0.2, 0.2, 0.2), G=0.1, Jt=(1.0, 0.93539, 0.24935), dt=0.004,
           s=(10.0, 5.0, 1.0), seed=2026)


def log(*a):
    print("[bench]", *a, file=sys.stderr, flush=True)


def initial_coeffs(plan, cfg):
    """Matrix Fisher (seeded R0 diag(10,5,1)) x Gaussian with a seeded SPD
    covariance (eigenvalues in [0.3, 1.5]), forward-transformed on the GPU."""
    import numpy as np
    import torch
    from hpup import density as D
    rng = np.random.default_rng(cfg["seed"])
    R0 = D.random_rotation(rng)
    Q = D.random_rotation(rng)
    Sigma = Q @ np.diag(rng.uniform(0.3, 1.5, 3)) @ Q.T
    fR, fx = D.matrix_fisher_gaussian(cfg["B"], cfg["dim"], cfg["N"], cfg["L"], cfg["s"], R0, Sigma=Sigma)
    f = D.grid_density(fR, fx)
    F = plan.forward(f)
    torch.cuda.synchronize()
    del f
    return F


def make_plan(cfg, precision, method):
    import numpy as np
    import hpup
    return hpup.Plan(cfg["B"], cfg["dim"], cfg["N"], cfg["L"], b=cfg["b"], G=np.eye(3) * cfg["G"],
                     Jt=np.diag(cfg["Jt"]), dt=cfg["dt"], method=method, precision=precision)


def timed_steps(plan, F, steps, warmup):
    """Warmup steps on a scratch copy (the device clocks up under load), then
    `steps` timed steps on F itself, bracketed by synchronizations."""
    import torch
    if warmup:
        Fw = F.clone()
        plan.step(Fw, warmup)
        del Fw
    torch.cuda.synchronize()
    e0 = torch.cuda.Event(enable_timing=True)
    e1 = torch.cuda.Event(enable_timing=True)
    e0.record()
    plan.step(F, steps)
    e1.record()
    torch.cuda.synchronize()
    return e0.elapsed_time(e1) / steps


def gradient_row(B=15, N=30, L=10.0, K=20, precision="fp64", checkpoints=(1, 5, 20), dt=0.004):
    """Cost of the gradient sweep (hpup.adjoint, reduced model, RK4) against a
    forward step: per step of the sweep beyond the forward pass, for the given
    checkpoint spacings (defaults: B = 15, 30^2 omega grid, every 1, 5 and 20
    steps; the gradient workload itself is B = 10, 32^2 over [-4, 4]^2, 50
    steps of 0.01, checkpoint every 10)."""
    import numpy as np
    import torch
    from hpup.adjoint import Gradient
    gr = Gradient(B, N, L, b=(0.2, 0.2), G=np.eye(2) * 0.1, dt=dt, method="rk4", precision=precision)
    g = torch.Generator(device="cpu").manual_seed(5)
    F0 = (torch.randn(gr.fwd.ncoef, generator=g, dtype=torch.complex128) * 1e-3).to(gr.fwd.cdtype).cuda()
    w = torch.randn(gr.fwd.ncoef, generator=g, dtype=torch.complex128).to(gr.fwd.cdtype).cuda()
    F = F0.clone()
    gr.fwd.step(F, 3)
    gr.run(F0, 2, lambda F: w, checkpoint=1)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    F = F0.clone()
    gr.fwd.step(F, K)
    torch.cuda.synchronize()
    tf = (time.perf_counter() - t0) / K
    out = {"config": "reduced model, B=%d, %d^2 omega grid, RK4, %s, %d steps" % (B, N, precision, K),
           "coefficients": gr.fwd.ncoef, "forward_step_ms": tf * 1e3}
    for cp in checkpoints:
        t0 = time.perf_counter()
        gr.run(F0, K, lambda F: w, checkpoint=cp)
        torch.cuda.synchronize()
        tg = (time.perf_counter() - t0) / K
        out["sweep_over_forward_checkpoint_%d" % cp] = (tg - tf) / tf
    return out


def output_errors(p64, F64, pm, Fm):
    """Each output of the path after the timed steps, from the reduced-precision
    plan against the FP64 plan on the same initial coefficients: relative L2
    (Frobenius) errors of the grid density, the omega marginal fx, the
    attitude mean E[R], the angular-velocity mean and covariance, and the
    fitted matrix-Fisher S and Gaussian Sigma of get_stat."""
    import numpy as np
    import torch
    f64 = p64.backward(F64)
    fm = pm.backward(Fm)
    out = {"grid_density": float(torch.linalg.vector_norm(fm.to(torch.float64) - f64) / torch.linalg.vector_norm(f64))}
    s64, sm = p64.get_stat(f64, return_fx=True), pm.get_stat(fm, return_fx=True)
    del f64, fm

    def rel(a, b):
        a, b = np.asarray(a, dtype=np.float64), np.asarray(b, dtype=np.float64)
        return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))
    for key, name in (("fx", "omega_marginal"), ("ER", "attitude_mean_ER"), ("Ex", "omega_mean_Ex"),
                      ("Varx", "omega_covariance_Varx"), ("S", "matrix_fisher_S"), ("Sigma", "gaussian_Sigma")):
        out[name] = rel(sm[key], s64[key])
    return out


def reset_row(B=15, N=32, L=3.4, nD=10, reps=3):
    """The hybrid reset gateways with the reduced hybrid driver's wall, contact
    and noise parameters (d = 0.12, h = 0.2, r = 0.025, theta_t = 5 deg,
    lambda_max = 100 t_scale, epsilon = 0.8, Gd = 0.05^2 I, nD = 10) on a
    B = 15, 32^2 grid over [-1.7, 1.7]^2: the best of `reps` wall times per
    call.  The gateways take and return host arrays, as the MEX functions they
    replace do, so these times include the host copies; the kernel times come
    from a kernel trace of the same run."""
    import numpy as np
    import hpup
    from hpup.density import rotation_grid
    n2 = 2 * B
    R = rotation_grid(B, device="cpu").numpy().reshape(3, 3, n2, n2, n2, order="F")
    ax = -L / 2 + L / N * np.arange(N)
    x = np.stack(np.meshgrid(ax, ax, indexing="ij"))
    par = dict(d=0.12, h=0.2, r=0.025, theta_t=5 * np.pi / 180, lambda_max=100.0 * 0.1177)
    t = {}

    def timed(key, fn):
        best, out = float("inf"), None
        for _ in range(reps):
            t0 = time.perf_counter()
            out = fn()
            best = min(best, time.perf_counter() - t0)
        t[key] = best * 1e3
        return out
    lam, indR, PC = timed("getLambda_ms", lambda: hpup.getLambda_mex(R, x, **par))
    Om = timed("getOmega_ms", lambda: hpup.getOmega_mex(R, x, indR, 0.8, PC, "new"))
    fcL, idx = timed("getFcL_ms", lambda: hpup.getFcL_mex(x, Om, lam, np.eye(2) * 0.05 ** 2, nD))
    f = np.asfortranarray(np.random.default_rng(3).random((n2, n2, n2, N, N)))
    timed("discrete_propagate_noise_ms", lambda: hpup.pendulum_reduced_discrete_propagate(True, f, lam, indR, fcL, idx))
    lc, indc, lists, PCc = hpup.getLambda_mex(R, x, compact=True, **par)
    Omo = hpup.getOmega_mex(R, x, indc, 0.8, PCc, "old")
    ind, co = timed("getIndRule_ms", lambda: hpup.getIndRule_mex(x, Omo))
    timed("discrete_propagate_nonoise_ms",
          lambda: hpup.pendulum_reduced_discrete_propagate(False, f, lc, indc, lists, ind, co))
    return dict({"config": "reduced hybrid reset, B=%d, %d^2 omega grid, nD=%d (gateway wall times, host copies "
                           "included)" % (B, N, nD), "numR": int(len(indR)), "grid_bytes": int(f.nbytes),
                 "fcL_bytes": int(fcL.nbytes + idx.nbytes)}, **t)


def hybrid_size_row(B=30, N=60, L=3.4, steps=3, precision="fp64"):
    """The reduced hybrid driver's own grid (bandlimit 30, 60^2 omega grid over
    [-1.7, 1.7]^2): one RK4 step of the continuous part (the 64-point MFMA
    drift kernel) and the inverse and forward transforms, device-resident,
    HIP events on the plan's stream."""
    import numpy as np
    import torch
    import hpup
    from hpup import density as D
    p = hpup.Plan(B, 2, N, L, b=(0.2, 0.2, 0.0), G=np.eye(2) * 0.1, dt=0.0025, method="RK4", precision=precision)
    rng = np.random.default_rng(30)
    fR, fx = D.matrix_fisher_gaussian(B, 2, N, L, (8, 4, 2), D.random_rotation(rng), Sigma=np.eye(2) * 0.3)
    f = D.grid_density(fR, fx, p.rdtype)
    del fR, fx
    F = p.forward(f)
    ev = [torch.cuda.Event(enable_timing=True) for _ in range(6)]
    p.step(F, 1)
    torch.cuda.synchronize()
    ev[0].record()
    p.step(F, steps)
    ev[1].record()
    ev[2].record()
    g = p.backward(F, f)
    ev[3].record()
    ev[4].record()
    p.forward(g, F)
    ev[5].record()
    torch.cuda.synchronize()
    row = {"config": "reduced hybrid driver grid, B=%d, %d^2 omega grid, RK4 dt=0.0025, %s" % (B, N, precision),
           "coefficients": p.ncoef, "rk4_step_ms": ev[0].elapsed_time(ev[1]) / steps,
           "transform_backward_ms": ev[2].elapsed_time(ev[3]), "transform_forward_ms": ev[4].elapsed_time(ev[5])}
    for name, ms, nbytes in p.profile(F, 2):
        if ms > 0 and name.startswith("k_drift"):
            row["drift_kernel"] = name
            row["drift_kernel_ms"] = ms
            row["drift_kernel_tb_s"] = nbytes / ms / 1e9
    return row


# the large hybrid workload: B = 30 (60^3 rotation grid), 20^3 omega grid
# over [-6, 6]^3, a 0.6 / 0.4 mixture of two matrix-Fisher x Gaussian
# components (seeded rotations, F = U diag(12, 6, 2); Gaussians of unit width
# at seeded means in [-1, 1]^3), the reflection reset with restitution 0.8 on
# a wall tilted by 0.2 rad (probability-conserving 1/eps Jacobian), RK4 with
# dt = 0.003
HYB = dict(B=30, N=20, L=12.0, dt=0.003, eps=0.8, tilt=0.2,
           reset=dict(d=0.12, h=0.2, r=0.025, theta_t=5 * 3.141592653589793 / 180, lambda_max=100.0 * 0.1173))


def hybrid_plan(precision, B=None, N=None):
    import numpy as np
    import hpup
    c = HYB
    B, N = B or c["B"], N or c["N"]
    p = hpup.Plan(B, 3, N, c["L"], b=(0.2, 0.2, 0.2), G=np.eye(3) * 0.1, Jt=np.diag([1.0, 0.93539, 0.24935]),
                  dt=c["dt"], method="RK4", precision=precision)
    p.set_reset(**c["reset"], epsilon=c["eps"], tilt=c["tilt"], jacobian=True)
    return p


def hybrid_initial(p):
    import numpy as np
    from hpup import density as D
    rng = np.random.default_rng(5)
    comps = [dict(s=(12, 6, 2), U=D.random_rotation(rng), mu=rng.uniform(-1, 1, 3), Sigma=np.eye(3))
             for _ in range(2)]
    f = D.mixture_density(p.B, 3, p.N, p.model.L, comps, (0.6, 0.4), dtype=p.rdtype)
    F = p.forward(f)
    del f
    return F


def hybrid_row(steps=3, err_steps=3):
    """The large hybrid workload (HYB), FP32 plan: per hybrid step the RK4
    step, the inverse transform, the reset (f += dt df on the grid) and the
    forward transform, HIP events on the plan's stream; the FP32 coefficients
    against an FP64 plan after err_steps hybrid steps; the restitution
    gradient sweep (HybridGradient, checkpoint every step) against the
    forward hybrid steps."""
    import torch
    from hpup.adjoint import HybridGradient
    p = hybrid_plan("fp32")
    F = hybrid_initial(p)
    f = p.empty_grid()
    p.hybrid_step(F, f, 1)  # warm-up
    torch.cuda.synchronize()
    ev = [torch.cuda.Event(enable_timing=True) for _ in range(9)]
    acc = [0.0] * 4
    ev[8].record()
    for _ in range(steps):
        ev[0].record()
        p.step(F, 1)
        ev[1].record()
        p.backward(F, f)
        ev[2].record()
        p.reset(f, f, p.model.dt, 0)
        ev[3].record()
        p.forward(f, F)
        ev[4].record()
        torch.cuda.synchronize()
        for i in range(4):
            acc[i] += ev[i].elapsed_time(ev[i + 1])
    whole = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
    whole[0].record()
    p.hybrid_step(F, f, steps)
    whole[1].record()
    torch.cuda.synchronize()
    step_ms = whole[0].elapsed_time(whole[1]) / steps
    out = {"config": "hybrid SO(3)xR^3, B=%d, %d^3 omega grid over [-6,6]^3, 0.6/0.4 matrix-Fisher x Gaussian "
                     "mixture, reflection reset eps=%.1f tilt=%.1f rad, RK4 dt=%.3f, FP32" %
                     (HYB["B"], HYB["N"], HYB["eps"], HYB["tilt"], HYB["dt"]),
           "coefficients": p.ncoef, "grid_points": p.ngrid, "region_rotations": int(len(p.reset_rows)),
           "hybrid_step_ms": step_ms, "hybrid_steps_per_s": 1000.0 / step_ms,
           "rk4_step_ms": acc[0] / steps, "transform_backward_ms": acc[1] / steps, "reset_ms": acc[2] / steps,
           "transform_forward_ms": acc[3] / steps}
    del F, f
    torch.cuda.empty_cache()
    # FP32 against FP64 after err_steps hybrid steps from the same initial coefficients
    p64 = hybrid_plan("fp64")
    F64 = hybrid_initial(p64)
    F32 = F64.to(torch.complex64)
    p64.hybrid_step(F64, p64.empty_grid(), err_steps)
    g32 = p.empty_grid()
    p.hybrid_step(F32, g32, err_steps)
    torch.cuda.synchronize()
    out["rel_l2_fp32_vs_fp64"] = float(torch.linalg.vector_norm(F32.to(torch.complex128) - F64) /
                                       torch.linalg.vector_norm(F64))
    out["rel_l2_after_steps"] = err_steps
    del p64, F64, F32, g32
    torch.cuda.empty_cache()
    # restitution gradient sweep, FP32, K = 2 hybrid steps, checkpoint every step
    K = 2
    hg = HybridGradient(HYB["B"], 3, HYB["N"], HYB["L"], dict(HYB["reset"], epsilon=HYB["eps"], tilt=HYB["tilt"],
                                                               jacobian=True),
                        b=(0.2, 0.2, 0.2), G=[[0.1, 0, 0], [0, 0.1, 0], [0, 0, 0.1]],
                        Jt=[[1.0, 0, 0], [0, 0.93539, 0], [0, 0, 0.24935]], dt=HYB["dt"], method="RK4",
                        precision="fp32")
    F0 = hybrid_initial(hg.fwd)
    wv = F0.clone()
    t0, t1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    t0.record()
    _, _, g = hg.run(F0, K, lambda F: wv, checkpoint=1)
    t1.record()
    torch.cuda.synchronize()
    out["restitution_gradient"] = g["epsilon"]
    out["gradient_sweep_ms_per_step"] = t0.elapsed_time(t1) / K
    out["gradient_over_forward"] = out["gradient_sweep_ms_per_step"] / step_ms
    return out


def row_timings(plan, F, reps=3):
    """The other rows of the path on this workload, timed with HIP events on
    torch's current stream (the plan's stream): inverse transform (coefficients
    -> grid), forward transform (grid -> coefficients) and get_stat (one device
    pass over the grid plus the host fit).  Bytes are the algorithmic floor of
    a transform: the real grid once plus the compact coefficients once."""
    import torch
    f = plan.backward(F)
    F2 = plan.forward(f)
    st = plan.get_stat(f)
    torch.cuda.synchronize()
    ev = [torch.cuda.Event(enable_timing=True) for _ in range(3)]
    tb = tf = 0.0
    for _ in range(reps):
        ev[0].record()
        plan.backward(F, f)
        ev[1].record()
        plan.forward(f, F2)
        ev[2].record()
        torch.cuda.synchronize()
        tb += ev[0].elapsed_time(ev[1]) / reps
        tf += ev[1].elapsed_time(ev[2]) / reps
    t0 = time.perf_counter()
    for _ in range(reps):
        st = plan.get_stat(f)
    ts = (time.perf_counter() - t0) * 1e3 / reps
    rt = float(torch.linalg.vector_norm((F2 - F).to(torch.complex128)) / torch.linalg.vector_norm(F.to(torch.complex128)))
    nbytes = f.numel() * f.element_size() + F.numel() * F.element_size()
    del f, F2
    row = lambda ms: {"ms": ms, "GBs": nbytes / (ms * 1e-3) / 1e9, "hbm_frac": nbytes / (ms * 1e-3) / 1e9 / HBM_PEAK_GBS,
                      "algorithmic_bytes": nbytes}
    return {"transform_backward": row(tb), "transform_forward": row(tf), "roundtrip_rel_l2": rt,
            "get_stat_ms": ts, "get_stat_fit_ok": bool(st["fit_ok"])}


def transforms_b30_row(reps=3):
    """The transforms of the large hybrid workload (B = 30, 20^3 omega grid,
    FP32 plan), HIP events on the plan's stream."""
    import torch
    p = hybrid_plan("fp32")
    F = hybrid_initial(p)
    f = p.backward(F)
    p.forward(f, F)
    torch.cuda.synchronize()
    ev = [torch.cuda.Event(enable_timing=True) for _ in range(3)]
    tb = tf = 0.0
    for _ in range(reps):
        ev[0].record()
        p.backward(F, f)
        ev[1].record()
        p.forward(f, F)
        ev[2].record()
        torch.cuda.synchronize()
        tb += ev[0].elapsed_time(ev[1]) / reps
        tf += ev[1].elapsed_time(ev[2]) / reps
    return {"transform_backward_ms": tb, "transform_forward_ms": tf, "coefficients": p.ncoef, "grid_points": p.ngrid}


def profile_rows(cfg, names):
    """--rows-only: the named rows alone (a short program to run under a
    profiler)."""
    import torch
    rows = {}
    for name in names:
        if name == "transforms":
            p64 = make_plan(cfg, "fp64", "RK4")
            F0 = initial_coeffs(p64, cfg)
            p32 = make_plan(cfg, "fp32", "RK4")
            for tag, pl, Fr in (("fp64", p64, F0), ("fp32", p32, F0.to(torch.complex64))):
                rows[tag] = row_timings(pl, Fr)
                log("rows %s: backward %.2f ms, forward %.2f ms" % (tag, rows[tag]["transform_backward"]["ms"],
                                                                      rows[tag]["transform_forward"]["ms"]))
            del p64, p32, F0
        elif name == "transforms_b30":
            rows[name] = transforms_b30_row()
            log("rows %s: backward %.2f ms, forward %.2f ms" % (name, rows[name]["transform_backward_ms"],
                                                                  rows[name]["transform_forward_ms"]))
        else:
            raise SystemExit("bench.py: unknown row %r for --rows-only" % name)
        torch.cuda.empty_cache()
    return rows


def _omp_threads():
    env = os.environ.get("OMP_NUM_THREADS", "")
    return int(env) if env.isdigit() and int(env) > 0 else len(os.sched_getaffinity(0))


def cpu_structured(Ffull, cfg, method):
    """One full step of this workload (all 121 M coefficients) with the
    oracle's structured FP64 form (oracle/refcpu_structured.c: the same
    operator on its exact nonzero support -- 1-D circulants along the omega
    axes, the gyroscopic quadratic form, banded Clebsch-Gordan, sparse u --
    with OpenMP on every host core): the optimized-CPU comparison."""
    sys.path.insert(0, os.path.join(REPO, "oracle"))
    import numpy as np
    import oracle as O
    B, N, L = cfg["B"], cfg["N"], cfg["L"]
    Jt = np.diag(cfg["Jt"])
    X = O.build_X(3, N, L)
    MR = O.build_MR(B, 3, Jt)
    u = O.getu(B - 1)
    cells = O.cg_table(B)
    threads = _omp_threads()
    t0 = time.perf_counter()
    O.integrate_structured(B, 3, N, Ffull, X, Jt, MR, np.array(cfg["b"]), np.eye(3) * cfg["G"], cfg["dt"], L, u,
                           cells, method)
    t = time.perf_counter() - t0
    log("cpu structured step %.2f s" % t)
    return {"value": 1.0 / t, "unit": "steps/s", "cores": threads, "kind": "port",
            "sample": "one full %s step of the whole workload (B=15, 30^3 omega grid, all coefficients) with the "
                      "oracle's structured FP64 derivative (oracle/refcpu_structured.c), %d OpenMP threads: %.1f s"
                      % (method, threads, t)}


def cpu_baseline(Ffull, cfg, stages, budget_s=25.0):
    """The reference's dense derivative (oracle, FP64) on a bounded sample of
    output omega points of this workload, extrapolated linearly in the number
    of output points to one derivative evaluation; a step costs `stages` of
    them.  The oracle spreads output points over its OpenMP threads, so the
    samples are T and 2T points (T threads): the slope is the cost of T more
    points, not the wall time of one."""
    sys.path.insert(0, os.path.join(REPO, "oracle"))
    import numpy as np
    import oracle as O
    B, N, L = cfg["B"], cfg["N"], cfg["L"]
    Jt = np.diag(cfg["Jt"])
    X = O.build_X(3, N, L)
    OJO = O.build_OJO(N, L, Jt)
    MR = O.build_MR(B, 3, Jt)
    u = O.getu(B - 1)
    cells = O.cg_table(B)
    bt = np.array(cfg["b"])
    G = np.eye(3) * cfg["G"]
    threads = _omp_threads()
    nx = N ** 3
    samples = []
    for S in (threads, 2 * threads):
        t0 = time.perf_counter()
        O.derivative(B, 3, N, Ffull, X, OJO, MR, bt, G, L, u, cells, 0, S)
        samples.append((S, time.perf_counter() - t0))
        log("cpu sample", S, "points", "%.2f s" % samples[-1][1])
        if samples[-1][1] > budget_s:
            break
    if len(samples) == 2 and samples[1][1] > samples[0][1]:
        (s1, t1), (s2, t2) = samples
        b = (t2 - t1) / (s2 - s1)
        a = max(t1 - b * s1, 0.0)
    else:
        s1, t1 = samples[-1]
        a, b = 0.0, t1 / s1
    t_eval = a + b * nx
    t_step = stages * t_eval
    return {"value": 1.0 / t_step, "unit": "steps/s", "cores": threads, "kind": "port",
            "sample": "reference dense derivative (oracle/refcpu.c, FP64, %d OpenMP threads) on the first %s of %d "
                      "output omega points of this workload, extrapolated linearly in the point count to one "
                      "derivative evaluation (%.1f s), times %d evaluations per step"
                      % (threads, "/".join(str(s) for s, _ in samples), nx, t_eval, stages)}


def main():
    ap = argparse.ArgumentParser(description=__doc__)
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=200)
    ap.add_argument("--warmup", type=int, default=10)
    ap.add_argument("--precision", default="fp32", choices=["fp32", "bf16x3", "fp64"])
    ap.add_argument("--method", default="RK4", choices=["euler", "midpoint", "RK2", "RK4"])
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline leg")
    ap.add_argument("--no-rows", action="store_true", help="skip the transform and get_stat timings")
    ap.add_argument("--profile-reps", type=int, default=20)
    ap.add_argument("--rows-only", default="",
                    help="profiling mode: run only these rows (comma list of 'transforms' -- the B=15, 30^3 "
                         "FP64 and FP32 transforms and get_stat -- and 'transforms_b30' -- the B=30, 20^3 FP32 "
                         "transforms of the large hybrid workload), print them as one JSON line and exit")
    ap.add_argument("--copy-probe-gib", type=float, default=0.0,
                    help="at the end, run a plain copy kernel (torch.neg, 4-byte elements) over this many GiB "
                         "three times: the known-size reference for scaling HBM counters")
    args = ap.parse_args()
    if args.gpus != 1:
        print("bench.py: this build runs on one GPU; --gpus %d is not supported (sharding the slabs "
              "across GPUs is not implemented)" % args.gpus, file=sys.stderr)
        sys.exit(2)
    import torch
    cfg = dict(CFG)
    K, W = args.steps, args.warmup
    if args.rows_only:
        print(json.dumps({"rows": profile_rows(cfg, args.rows_only.split(","))}), flush=True)
        copy_probe(args.copy_probe_gib)
        return

    stages = {"euler": 1, "midpoint": 2, "RK2": 2, "RK4": 4}[args.method]
    log("building FP64 plan and initial coefficients")
    p64 = make_plan(cfg, "fp64", args.method)
    F0 = initial_coeffs(p64, cfg)
    im = p64.mass_index  # F^0_00(k = 0)
    mass0 = float(F0[im].real)
    F64 = F0.clone()
    ms64 = timed_steps(p64, F64, K, W)
    log("fp64 %.3f ms/step" % ms64)
    mass_drift = abs(float(F64[im].real) - mass0) / abs(mass0)

    if args.precision == "fp64":
        pm, Fm, msm = p64, F64, ms64
        err = 0.0
    else:
        pm = make_plan(cfg, args.precision, args.method)
        Fm = F0.to(torch.complex64)
        msm = timed_steps(pm, Fm, K, W)
        log("%s %.3f ms/step" % (args.precision, msm))

    # the precision gate is taken after the workload's full 200 steps,
    # whatever --steps timed (untimed extra propagation when they differ)
    if args.precision != "fp64":
        if K == ERR_STEPS:
            F64e, Fme = F64, Fm
        else:
            F64e, Fme = F0.clone(), F0.to(torch.complex64)
            p64.step(F64e, ERR_STEPS)
            pm.step(Fme, ERR_STEPS)
            torch.cuda.synchronize()
        err = float(torch.linalg.vector_norm((Fme.to(torch.complex128) - F64e)) / torch.linalg.vector_norm(F64e))
        log("%s rel L2 vs fp64 after %d steps: %.2e" % (args.precision, ERR_STEPS, err))

    out_err = None
    if args.precision != "fp64":
        try:
            out_err = output_errors(p64, F64e, pm, Fme)
            log("outputs vs fp64:", ", ".join("%s %.1e" % kv for kv in out_err.items()))
        except Exception as e:  # an optional report must not hide the headline result
            log("output errors failed:", repr(e))

    # the other mixed-precision variant: 3xBF16 split-product circulants
    # (three bf16 pieces per operand, six products, FP32 accumulation), its
    # step time and its error after the workload's 200 steps
    split_row = None
    if args.precision == "fp32" and not args.no_rows:
        try:
            pb = make_plan(cfg, "bf16x3", args.method)
            Fb = F0.to(torch.complex64)
            msb = timed_steps(pb, Fb, K, W)
            Fbe = Fb if K == ERR_STEPS else F0.to(torch.complex64)
            if K != ERR_STEPS:
                pb.step(Fbe, ERR_STEPS)
            torch.cuda.synchronize()
            eb = float(torch.linalg.vector_norm(Fbe.to(torch.complex128) - F64e) / torch.linalg.vector_norm(F64e))
            split_row = {"ms_per_step": msb, "steps_per_s": 1000.0 / msb, "speedup_vs_fp64": ms64 / msb,
                         "rel_l2_vs_fp64": eb, "rel_l2_vs_fp64_after_steps": ERR_STEPS}
            log("bf16x3 %.3f ms/step, rel L2 vs fp64 after %d steps %.2e" % (msb, ERR_STEPS, eb))
            del pb, Fb, Fbe
            torch.cuda.empty_cache()
        except Exception as e:
            log("bf16x3 row failed:", repr(e))

    # per-kernel timing with HIP events on the stream the kernels run on
    Fp = Fm.clone()
    prof = pm.profile(Fp, args.profile_reps)
    del Fp
    name, kms, kbytes = max(prof, key=lambda t: t[1])
    log("kernels:", ", ".join("%s %.3f ms" % (n, t) for n, t, _ in prof))
    # the dominant kernel's two roofs: MFMA (useful circulant FLOPs) and HBM
    # (algorithmic bytes); the binding one is the larger ideal time
    kflops = kernel_flops(name, cfg["B"], cfg["N"])
    peak_tf = MFMA_PEAK_TFLOPS[args.precision]
    # the path's algorithmic bytes per derivative evaluation: read F, write
    # F' once, 2 C s (C coefficients of s bytes); one launch of the dominant
    # kernel is one derivative evaluation
    csize = 16 if args.precision == "fp64" else 8
    alg_bytes = 2.0 * pm.ncoef * csize
    hbm_gbs = alg_bytes / (kms * 1e-3) / 1e9
    mfma_tf = kflops / (kms * 1e-3) / 1e12
    traffic = MEASURED_TRAFFIC.get((name, args.precision, args.method))
    roof = {"bound": "hbm", "kernel": name, "achieved": hbm_gbs, "peak": HBM_PEAK_GBS, "unit": "GB/s",
            "frac": hbm_gbs / HBM_PEAK_GBS, "traffic": traffic, "kernel_ms": kms, "algorithmic_bytes": alg_bytes,
            "algorithmic_bytes_rule": "2 C s per derivative evaluation (read F, write F'), C = %d coefficients, "
                                      "s = %d bytes" % (pm.ncoef, csize),
            "kernel_stream_bytes": kbytes, "kernel_stream_frac": kbytes / (kms * 1e-3) / 1e9 / HBM_PEAK_GBS,
            "mfma": {"useful_flops": kflops, "achieved_TFLOPs": mfma_tf, "peak_TFLOPs": peak_tf,
                     "frac": mfma_tf / peak_tf},
            "ideal_ms": {"mfma": kflops / (peak_tf * 1e12) * 1e3, "hbm": alg_bytes / (HBM_PEAK_GBS * 1e9) * 1e3},
            "path_GBs_per_step": stages * alg_bytes / (msm * 1e-3) / 1e9,
            "path_frac": stages * alg_bytes / (msm * 1e-3) / 1e9 / HBM_PEAK_GBS}

    rows = {}
    if not args.no_rows:
        for tag, pl, Fr in (("fp64", p64, F0), (args.precision, pm, Fm)):
            if tag not in rows:
                rows[tag] = row_timings(pl, Fr if tag != "fp64" else F0)
                log("rows %s: backward %.2f ms, forward %.2f ms, get_stat %.2f ms"
                    % (tag, rows[tag]["transform_backward"]["ms"], rows[tag]["transform_forward"]["ms"],
                       rows[tag]["get_stat_ms"]))
        try:
            rows["gradient"] = gradient_row()
            rows["gradient_fp32"] = gradient_row(precision="fp32")
            for key in ("gradient", "gradient_fp32"):
                log("rows %s: sweep / forward step %s (checkpoint 1, 5, 20)" % (key, ", ".join(
                    "%.2f" % rows[key]["sweep_over_forward_checkpoint_%d" % cp] for cp in (1, 5, 20))))
            for prec in ("fp64", "fp32"):
                key = "gradient_workload" + ("" if prec == "fp64" else "_fp32")
                rows[key] = gradient_row(B=10, N=32, L=8.0, K=50, precision=prec, checkpoints=(1, 10), dt=0.01)
                log("rows %s: sweep / forward step %.2f (checkpoint 10), %.2f (checkpoint 1); forward %.3f ms"
                    % (key, rows[key]["sweep_over_forward_checkpoint_10"], rows[key]["sweep_over_forward_checkpoint_1"],
                       rows[key]["forward_step_ms"]))
        except Exception as e:  # an optional row must not hide the headline result
            log("gradient row failed:", repr(e))
        try:
            rows["hybrid_size"] = hybrid_size_row()
            hs = rows["hybrid_size"]
            log("rows hybrid_size: RK4 step %.2f ms, backward %.2f ms, forward %.2f ms, %s %.3f ms per launch "
                "(%.2f TB/s)" % (hs["rk4_step_ms"], hs["transform_backward_ms"], hs["transform_forward_ms"],
                                 hs.get("drift_kernel", "?"), hs.get("drift_kernel_ms", 0.0),
                                 hs.get("drift_kernel_tb_s", 0.0)))
        except Exception as e:
            log("hybrid-size row failed:", repr(e))
        try:
            rows["hybrid"] = hybrid_row()
            log("rows hybrid:", ", ".join("%s %s" % (k, ("%.4g" % v) if isinstance(v, float) else v)
                                          for k, v in rows["hybrid"].items() if k != "config"))
        except Exception as e:
            log("hybrid row failed:", repr(e))
        try:
            rows["reset"] = reset_row()
            log("rows reset:", ", ".join("%s %s" % (k, ("%.2f" % v) if isinstance(v, float) else v)
                                         for k, v in rows["reset"].items() if k != "config"))
        except Exception as e:
            log("reset row failed:", repr(e))

    cpu = None
    if not args.no_cpu:
        try:
            Ffull = p64.download_full(F0)
            cpu = cpu_structured(Ffull, cfg, args.method)
            cpu["dense_reference_algorithm"] = cpu_baseline(Ffull, cfg, stages)
            del Ffull
        except Exception as e:  # the CPU leg must not hide the GPU result
            log("cpu baseline failed:", repr(e))

    steps_s = 1000.0 / msm
    out = {
        "metric": "propagation steps/s, B=15 SO(3)xR^3: FP32-MFMA vs FP64 at <=1e-6 rel L2",
        "value": steps_s,
        "unit": "steps/s",
        "n_gpus": 1,
        "steps": K,
        "warmup": W,
        "ms_per_step": msm,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": {"fp32": "f32", "bf16x3": "bf16x3-f32acc", "fp64": "f64"}[args.precision],
        "data": "synthetic (seeded matrix-Fisher x Gaussian initial density, forward-transformed on the GPU)",
        "config": {"workload": "3-D pendulum SO(3)xR^3, B=15, 30^3 omega grid over [-5,5]^3, %s dt=0.004, "
                               "%d steps" % (args.method, K),
                   "B": 15, "omega_grid": [30, 30, 30], "coefficients": pm.ncoef, "method": args.method,
                   "derivative_evals_per_step": stages, "precision": args.precision,
                   "parallelism": "single GPU"},
        "fp64_steps_per_s": 1000.0 / ms64,
        "speedup_vs_fp64": ms64 / msm,
        "rel_l2_vs_fp64": err,
        "rel_l2_vs_fp64_after_steps": ERR_STEPS,
        "output_errors_vs_fp64": out_err,
        "fp64_mass_drift": mass_drift,
        "bf16x3": split_row,
        "roofline": roof,
        "kernels_ms": {n: t for n, t, _ in prof},
        "rows": rows,
        "cpu_baseline": cpu,
    }
    print(json.dumps(out), flush=True)
    copy_probe(args.copy_probe_gib)


def copy_probe(gib):
    """A plain copy kernel (torch.neg, 4-byte elements) over `gib` GiB, three
    launches: the known-size reference for scaling HBM counters."""
    import torch
    if gib <= 0:
        return
    n = int(gib * 2 ** 30 / 4)
    x = torch.ones(n, dtype=torch.float32, device="cuda")
    y = torch.empty_like(x)
    for _ in range(3):
        torch.neg(x, out=y)
    torch.cuda.synchronize()
    log("copy probe: %d bytes read and %d written per launch" % (4 * n, 4 * n))


if __name__ == "__main__":
    main()
