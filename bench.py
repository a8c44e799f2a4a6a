"""BP5 matrix-free operator benchmark on one MI355X.

Workload (one "step"): one operator apply (vmult, deal.II semantics: dst = 0,
gather/apply/scatter, constrained rows copied) for each of p = 4, 6, 8 of the
BP5 plain method: scalar Laplacian, Q_p with GLL collocation (q = p+1), unit
cube deformed by x += 0.05 sin(2 pi x) sin(2 pi y) sin(2 pi z), n^3 cells with
n = 80 / 52 / 40 (33.1M / 30.7M / 33.1M DoFs), FP64, input uniform[-1,1] from
SplitMix64 seed 1.  Value = aggregate GDoF/s = sum_p N_p / sum_p t_p.  (The
cell counts have enough factors of two for the multigrid hierarchy to reach a
directly solvable coarse mesh.)

Each degree is measured with the metric terms stored (G, 48 q^3 B per cell,
patch kernel) and computed on the fly from the cell vertices (plane kernel
at p = 2, 4, 6, patch kernel at p = 8); the faster mode per degree enters the aggregate.  Also reported
per degree: the apply kernel's time (HIP events on the launch stream), its
algorithmic bytes and FLOPs, Jacobi-CG and mixed-precision multigrid CG
time-to-1e-8 relative residual on the same operator and right-hand side, the
BP3 unit-cube case (Q4, Gauss q=6, 8^3 affine cells, 35937 DoFs: vmult
checksum and time, Jacobi-CG to 1e-10 with the manufactured solution's
nodal error), the mixed-precision BP3 solve (Q4, Gauss q=6, deformed 128^3 cells, 135M
DoFs, manufactured-solution right-hand side, FP64 CG to 1e-10 with an FP32
p/h-multigrid V-cycle) with its error against an FP64 solution, and the
batched solve of 64 BP5 problems of uneven size and degree (per-instance
Jacobi-CG in one hipGraph-replayed batch) against solving them one by one,
and the learned-preconditioner flexible CG (Q4 BP5 on 64^3 cells) with its
training cost, against the same method without the network, Jacobi-CG and
multigrid CG.
"""
import argparse
import ctypes as C
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

HBM_PEAK = 8.0e12
FP64_PEAK = 78.6e12
CELLS = {2: 160, 4: 80, 6: 52, 8: 40}
STORED, ON_THE_FLY = 0, 1


def algorithmic_bytes(p, N, E, geometry, patch_cells=None, n_patches=0):
    """Bytes an apply must move at least once: src read + dst write (8 B per
    DoF each) + the DoF map + the geometry.  Stored: uint32 map (4 (p+1)^3
    per cell) and G (6 doubles per quadrature point).  On the fly: the patch
    DoF map (4 B per patch DoF, patches of patch_cells cells) and 8 vertices
    per cell (192 B)."""
    q = p + 1
    if geometry == STORED:
        return 16 * N + 4 * (p + 1) ** 3 * E + 48 * q ** 3 * E
    bx, by, bz = patch_cells
    return 16 * N + 4 * (bx * p + 1) * (by * p + 1) * (bz * p + 1) * n_patches + 192 * E


def flops_per_cell(p, geometry=STORED):
    """FP64 operations of one cell's apply (an FMA counts 2).  Stored metric:
    the sum-factorized BK5 count 12 q^4 + 15 q^3 (rooflineBK5.py:23-35:
    6 q^4 gradient + 6 q^4 transposed gradient + 15 per point for G grad u).
    On the fly (patch kernel): per point, 73 in place of the 15 (cofactor
    polynomials 24, det 5, reciprocal 9, weight 2, W 15, three projections
    18) and per (x,y) column 180 for the trilinear coefficients."""
    q = p + 1
    if geometry == STORED:
        return 12 * q ** 4 + 15 * q ** 3
    return 12 * q ** 4 + 73 * q ** 3 + 180 * q ** 2


def _events():
    import torch
    return torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)


def per_call_ms(fn, calls, stream):
    """Sorted per-call times (ms) of `calls` launches of fn(), each bracketed
    by its own pair of HIP events on `stream` (the stream the library
    launches on).  A stall of the device during one call moves one sample,
    not the median."""
    import torch
    ev = [_events() for _ in range(calls)]
    for a, b in ev:
        a.record(stream)
        fn()
        b.record(stream)
    torch.cuda.synchronize()
    return sorted(a.elapsed_time(b) for a, b in ev)


def bench_mode(p, geometry, steps, warmup, det_timing=True):
    import torch

    from benchmarks_amd.laplace import LaplaceOperator, random_vector
    n = CELLS[p]
    op = LaplaceOperator(p, p + 1, 1, n_cells=n, deform=0.05, geometry=geometry)
    N, E = op.m(), op.n_cells()
    x = random_vector(N, 1)
    y = op.initialize_dof_vector()
    stream = torch.cuda.current_stream()
    for _ in range(warmup):
        op.vmult(y, x)
    torch.cuda.synchronize()
    e0, e1 = _events()
    e0.record(stream)
    for _ in range(steps):
        op.vmult(y, x)
    e1.record(stream)
    torch.cuda.synchronize()
    t_vmult = e0.elapsed_time(e1) * 1e-3 / steps
    # per-call times of the same vmult (an event pair around each call), for
    # the best and the median
    per_call = per_call_ms(lambda: op.vmult(y, x), steps, stream)
    # the element kernel alone (vmult_add: no zero-fill, no constrained copy),
    # per call; its median cannot exceed the median of the vmult that
    # contains it, so a violation means the device was disturbed during the
    # sample: it is taken once more, and flagged if it persists
    scratch = torch.zeros(N, dtype=torch.float64, device="cuda")
    for _ in range(3):
        op.vmult_add(scratch, x)
    torch.cuda.synchronize()
    med_vmult = per_call[len(per_call) // 2]
    for attempt in range(2):
        k_calls = per_call_ms(lambda: op.vmult_add(scratch, x), steps, stream)
        med_kernel = k_calls[len(k_calls) // 2]
        if med_kernel <= med_vmult:
            break
    t_kernel = med_kernel * 1e-3
    # known-size probes for hardware-counter scaling: the deterministic dot
    # reads exactly 16 N bytes, vmult's zero-fill writes exactly 8 N bytes
    from benchmarks_amd._lib import check, lib
    dot = C.c_double()
    check(lib().mfx_vec_dot(C.c_void_p(x.data_ptr()), C.c_void_p(y.data_ptr()), N,
                            C.byref(dot), C.c_void_p(stream.cuda_stream)))
    info = op.info
    b_alg = algorithmic_bytes(p, N, E, geometry, tuple(info.patch_cells), info.n_patches)
    f_alg = flops_per_cell(p, geometry) * E
    det = {}
    if geometry == ON_THE_FLY and det_timing:
        # the price of bitwise reproducibility: the same vmult with the
        # deterministic scatter (patch sums stored, then added per DoF in a
        # fixed order)
        op.set_deterministic(True)
        for _ in range(3):
            op.vmult(y, x)
        d_calls = per_call_ms(lambda: op.vmult(y, x), steps, stream)
        op.set_deterministic(False)
        det = {"ms_vmult_deterministic_median": d_calls[len(d_calls) // 2]}
    res = {"geometry": "stored" if geometry == STORED else "on_the_fly", "ms_vmult": t_vmult * 1e3,
           "ms_vmult_best": per_call[0], "ms_vmult_median": med_vmult,
           "gdofs_vmult": N / t_vmult * 1e-9, "ms_kernel": med_kernel,
           "ms_kernel_best": k_calls[0], "kernel_samples": len(k_calls),
           "kernel_timing_valid": med_kernel <= med_vmult, "bytes_alg": b_alg,
           "flops_alg": f_alg, "kernel_GBs": b_alg / t_kernel * 1e-9,
           "kernel_TFLOPs": f_alg / t_kernel * 1e-12, **det}
    return op, x, y, res


def bench_degree(p, steps, warmup, do_cg, modes, det_timing=True):
    import torch

    from benchmarks_amd.laplace import (DiagonalMatrix, ReductionControl, SolverCG,
                                        random_vector)
    out = {"p": p, "n_cells_1d": CELLS[p], "modes": {}}
    best = None
    for g in modes:
        op, x, y, r = bench_mode(p, g, steps, warmup, det_timing)
        out["n_dofs"], out["n_cells"] = op.m(), op.n_cells()
        out["modes"][r["geometry"]] = r
        if best is None or r["ms_vmult"] < best[1]["ms_vmult"]:
            best = (g, r)
        del op, x, y
        torch.cuda.empty_cache()
    g, r = best
    out.update({"geometry": r["geometry"], "ms_vmult": r["ms_vmult"],
                "gdofs_vmult": r["gdofs_vmult"], "ms_kernel": r["ms_kernel"],
                "bytes_alg": r["bytes_alg"], "flops_alg": r["flops_alg"]})
    if "stored" in out["modes"]:
        # the HBM roofline of the apply with stored metric terms (its
        # algorithmic bytes at 8 TB/s), against which either mode's vmult
        # rate is measured
        roof = out["n_dofs"] * HBM_PEAK / out["modes"]["stored"]["bytes_alg"] * 1e-9
        out["stored_G_hbm_roofline_gdofs"] = roof
        out["frac_of_stored_G_hbm_roofline"] = r["gdofs_vmult"] / roof
    if do_cg:
        from benchmarks_amd.laplace import LaplaceOperator
        op = LaplaceOperator(p, p + 1, 1, n_cells=CELLS[p], deform=0.05, geometry=g)
        N = op.m()
        b = random_vector(N, 1)
        op.zero_constrained(b)
        inv = op.compute_inverse_diagonal()
        sol = op.initialize_dof_vector()
        ctl = ReductionControl(100000, 1e-300, 1e-8)
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        SolverCG(ctl).solve(op, sol, b, DiagonalMatrix(inv))
        torch.cuda.synchronize()
        t_cg = time.perf_counter() - t0
        out.update({"cg_jacobi_its": ctl.last_step(), "cg_jacobi_s": t_cg,
                    "cg_final_rel_res": ctl.last_value() / ctl.initial_value()})
        out.update(cg_split(t_cg, ctl.last_step(), r["ms_kernel"], N, r["bytes_alg"], "jacobi"))
        out.update(mg_solve(p, p + 1, 1, CELLS[p], ON_THE_FLY, b, sol, 1e-8))
        del op, b, inv, sol
        torch.cuda.empty_cache()
    return out


# N-vector passes of one CG step outside the operator apply (mfx_cg_solve,
# vector.hip): the direction pass reads r, the inverse diagonal, p and x and
# writes p, x (the previous step's x += alpha p) and Ap = 0; the update pass
# reads r, Ap and the inverse diagonal and writes r.  The identity
# preconditioner reads no inverse diagonal.  p.Ap is summed inside the apply.
CG_VECTOR_PASSES = {"jacobi": 11, "identity": 9}


def cg_split(seconds, steps, ms_apply, n_dofs, apply_bytes, kind):
    """Per-step split of a CG solve as the reference logs it
    (CEED_bp/results/1xGH200_P4.txt:630: time per iteration and the matvec's
    share): ms per step, the share of the median element-kernel time, the
    vector passes per step and the step's algorithmic bytes
    (apply + passes x 8 N) at that rate."""
    ms_step = seconds / max(steps, 1) * 1e3
    k = CG_VECTOR_PASSES[kind]
    step_bytes = apply_bytes + k * 8 * n_dofs
    return {f"cg_{kind}_ms_per_step": ms_step, f"cg_{kind}_apply_share": ms_apply / ms_step,
            f"cg_{kind}_vector_passes": k,
            f"cg_{kind}_step_bytes_alg": step_bytes,
            f"cg_{kind}_step_GBs": step_bytes / (ms_step * 1e-3) * 1e-9}


def _timed_solve(A, x, b, precond, rel_tol, max_steps):
    import torch

    from benchmarks_amd.laplace import ReductionControl, SolverCG
    ctl = ReductionControl(max_steps, 1e-300, rel_tol)
    x.zero_()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    SolverCG(ctl).solve(A, x, b, precond)
    torch.cuda.synchronize()
    return time.perf_counter() - t0, ctl


def _rel(a, b):
    import torch
    return (torch.linalg.norm(a - b) / torch.linalg.norm(b)).item()


def mg_solve(p, nq, quad, n, geometry, b, x_ref_jacobi, rel_tol):
    """FP64 CG preconditioned by the FP32 p/h-multigrid V-cycle on the same
    problem as a Jacobi-CG solve: set-up time, time and steps to rel_tol, and
    the errors of both solutions against an FP64 solution whose residual is
    certified to 1e-13 by the FP64 outer CG."""
    import torch

    from benchmarks_amd.laplace import PreconditionMG
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    mg = PreconditionMG(p, nq, quad, n, deform=0.05, geometry=geometry)
    torch.cuda.synchronize()
    t_setup = time.perf_counter() - t0
    A = mg.operator()
    x = A.initialize_dof_vector()
    _timed_solve(A, x, b, mg, rel_tol, 500)  # warm-up (kernel loading)
    t_mg, ctl = _timed_solve(A, x, b, mg, rel_tol, 500)
    x_ref = A.initialize_dof_vector()
    _timed_solve(A, x_ref, b, mg, 1e-13, 200)
    res = {"mg_levels": [(mg.level(l)["degree"], mg.level(l)["n_cells"][0])
                         for l in range(mg.n_levels())],
           "mg_setup_s": t_setup, "cg_mg_its": ctl.last_step(), "cg_mg_s": t_mg,
           "cg_mg_final_rel_res": ctl.last_value() / ctl.initial_value(),
           "cg_mg_err_vs_fp64": _rel(x, x_ref),
           "cg_jacobi_err_vs_fp64": _rel(x_ref_jacobi, x_ref)}
    del mg, A, x, x_ref
    torch.cuda.empty_cache()
    return res


def bench_c1(n=8, p=4, nq=6):
    """BP3 on the unit cube, n^3 affine cells, Q4, Gauss q=6 (35937 DoFs):
    one vmult of a SplitMix64 seed-0 vector in [-1, 1] (its 2-norm is the
    checksum; best of 5 x 200 vmults, as CEED_bp/src/bp3.cc:331-408 times
    small meshes), then Jacobi-CG to 1e-10 relative with
    f = 3 pi^2 prod sin(pi x_d), u = 0 on the boundary, x0 = 0: steps, time
    and the nodal error against the exact solution prod sin(pi x_d)."""
    import math

    import torch

    from benchmarks_amd.laplace import DiagonalMatrix, LaplaceOperator, random_vector
    A = LaplaceOperator(p, nq, 0, n_cells=n)
    x = random_vector(A.m(), 0)
    y = A.initialize_dof_vector()
    A.vmult(y, x)
    e0, e1 = _events()
    best = float("inf")
    for _ in range(5):
        e0.record()
        for _ in range(200):
            A.vmult(y, x)
        e1.record()
        torch.cuda.synchronize()
        best = min(best, e0.elapsed_time(e1) / 200)
    b = A.rhs(1)
    A.zero_constrained(b)
    u_h = A.initialize_dof_vector()
    _timed_solve(A, u_h, b, DiagonalMatrix(A.compute_inverse_diagonal()), 1e-10, 100000)
    t, ctl = _timed_solve(A, u_h, b, DiagonalMatrix(A.compute_inverse_diagonal()), 1e-10, 100000)
    xyz = A.dof_coordinates()
    u = torch.sin(math.pi * xyz[:, 0]) * torch.sin(math.pi * xyz[:, 1]) * torch.sin(math.pi * xyz[:, 2])
    return {"workload": f"BP3 Q{p} Gauss q={nq}, unit cube {n}^3 affine cells, manufactured sin RHS",
            "n_dofs": A.m(), "vmult_checksum_l2": torch.linalg.norm(y).item(),
            "ms_vmult_best": best, "cg_jacobi_its_1e-10": ctl.last_step(), "cg_jacobi_s_1e-10": t,
            "nodal_max_err_vs_exact": ((u_h - u).abs().max() / u.abs().max()).item()}


def bp3_cycle_mesh(cycle):
    """Mesh of cycle `cycle` of CEED_bp/src/bp3.cc:452-474: n_ref = cycle / 3
    global refinements of the box [-1,-1,-1]-[p2] with p2_d = 2.8 and two
    subdivisions for d < cycle % 3, else 0.9 and one.  Returns (cells per
    direction, lo, hi)."""
    nref, rem = cycle // 3, cycle % 3
    n = tuple((2 if d < rem else 1) * (1 << nref) for d in range(3))
    hi = tuple(2.8 if d < rem else 0.9 for d in range(3))
    return n, (-1.0, -1.0, -1.0), hi


# The reference's published figures for this problem on one GH200
# (CEED_bp/results/1xGH200_P4.txt:630, 648): best matvec 9.396 ms, CG to
# 1e-9 in 1389 steps, 15.53 s, 11.18 ms per step.
BP3_PUBLISHED = {"hardware": "1x GH200", "n_dofs": 67634433, "ms_matvec": 9.396,
                 "gdofs_matvec": 67634433 / 9.396e-3 * 1e-9, "cg_its": 1389, "cg_s": 15.53,
                 "cg_ms_per_step": 11.18, "source": "CEED_bp/results/1xGH200_P4.txt:630,648"}


def bench_bp3_reference(cycle=20, p=4, nq=6):
    """The reference's own published problem: BP3 Q4, Gauss q=6, on cycle 20
    of the bp3.cc box family (128 x 128 x 64 affine cells, 67,634,433 DoFs),
    f = 1, homogeneous Dirichlet, with the protocol of
    CEED_bp/src/bp3.cc:290-319: the best of 5 rounds of 50 matvecs of the
    right-hand side, and CG with the identity preconditioner and
    ReductionControl(1e9, 1e-16, 1e-9) from x = 0.  The matvec is timed with
    the metric terms stored (the reference's own form) and computed from the
    cell vertices; CG runs on the faster form, one timed solve after a short
    warm-up solve (the reference takes the best of ten)."""
    import torch

    from benchmarks_amd.laplace import (LaplaceOperator, PreconditionIdentity, ReductionControl,
                                        SolverCG)
    n, lo, hi = bp3_cycle_mesh(cycle)
    stream = torch.cuda.current_stream()
    forms = {}
    for g, name in ((STORED, "stored"), (ON_THE_FLY, "on_the_fly")):
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        A = LaplaceOperator(p, nq, 0, n_cells=n, lo=lo, hi=hi, geometry=g)
        b = A.rhs(0)
        torch.cuda.synchronize()
        t_setup = time.perf_counter() - t0
        N, E = A.m(), A.n_cells()
        y = A.initialize_dof_vector()
        A.vmult(y, b)
        best = float("inf")
        for _ in range(5):
            e0, e1 = _events()
            e0.record(stream)
            for _ in range(50):
                A.vmult(y, b)
            e1.record(stream)
            torch.cuda.synchronize()
            best = min(best, e0.elapsed_time(e1) / 50)
        scratch = torch.zeros(N, dtype=torch.float64, device="cuda")
        k_calls = per_call_ms(lambda: A.vmult_add(scratch, b), 20, stream)
        b_alg = 16 * N + 4 * (p + 1) ** 3 * E + (48 * nq ** 3 * E if g == STORED else 192 * E)
        forms[name] = {"setup_s": t_setup, "ms_matvec_best": best, "gdofs_matvec": N / best * 1e-6,
                       "ms_kernel_median": k_calls[len(k_calls) // 2], "kernel_bytes_alg": b_alg,
                       "kernel_GBs": b_alg / k_calls[len(k_calls) // 2] * 1e-6}
        del A, b, y, scratch
        torch.cuda.empty_cache()
    fast = min(forms, key=lambda k: forms[k]["ms_matvec_best"])
    A = LaplaceOperator(p, nq, 0, n_cells=n, lo=lo, hi=hi,
                        geometry=STORED if fast == "stored" else ON_THE_FLY)
    b = A.rhs(0)
    N, E = A.m(), A.n_cells()
    x = A.initialize_dof_vector()
    _timed_solve(A, x, b, PreconditionIdentity(), 1e-2, 1000)  # warm-up
    x.zero_()
    ctl = ReductionControl(1000000000, 1e-16, 1e-9)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    SolverCG(ctl).solve(A, x, b, PreconditionIdentity())
    torch.cuda.synchronize()
    t_cg = time.perf_counter() - t0
    f = forms[fast]
    out = {"workload": f"BP3 Q{p} Gauss q={nq}, bp3.cc cycle {cycle}: {n[0]}x{n[1]}x{n[2]} "
                       f"affine cells on [-1,-1,-1]-[{hi[0]},{hi[1]},{hi[2]}], f = 1, identity CG "
                       "to 1e-9",
           "n_dofs": N, "n_cells": E, "matvec": forms, "geometry": fast,
           "ms_matvec_best": f["ms_matvec_best"], "gdofs_matvec": f["gdofs_matvec"],
           "cg_its": ctl.last_step(), "cg_s": t_cg,
           "cg_reduction_per_step": (ctl.last_value() / ctl.initial_value())
           ** (1.0 / max(ctl.last_step(), 1)),
           "cg_its_match_reference_log": ctl.last_step() == BP3_PUBLISHED["cg_its"]}
    out.update(cg_split(t_cg, ctl.last_step(), f["ms_kernel_median"], N, f["kernel_bytes_alg"],
                        "identity"))
    out["published"] = BP3_PUBLISHED
    out["speedup_matvec_vs_published"] = BP3_PUBLISHED["ms_matvec"] / f["ms_matvec_best"]
    out["speedup_matvec_stored_vs_published"] = (BP3_PUBLISHED["ms_matvec"]
                                                 / forms["stored"]["ms_matvec_best"])
    out["speedup_cg_vs_published"] = BP3_PUBLISHED["cg_s"] / t_cg
    del A, b, x
    torch.cuda.empty_cache()
    return out


def bench_c3(n=128, p=4, nq=6):
    """Mixed-precision BP3 solve: Q4, Gauss q=6, deformed n^3 cells,
    f = 3 pi^2 prod sin(pi x_d), u = 0 on the boundary; FP64 CG with the FP32
    multigrid V-cycle to 1e-10 (and 1e-8), in three forms: the metric terms
    of every level stored; computed from the cell vertices; computed from the
    cell vertices with the fine level smoothing with Gauss q = p+1 (the outer
    CG always applies the q = nq operator).  The fastest form to 1e-8 is
    reported as the result; Jacobi-CG to 1e-8 on the same operator; errors
    against an FP64 solution certified to 1e-13 and, at the nodes, against
    the exact solution prod sin(pi x_d)."""
    import math

    import torch

    from benchmarks_amd.laplace import DiagonalMatrix, PreconditionMG
    forms = {}
    settings = {"stored": (STORED, 0), "on_the_fly": (ON_THE_FLY, 0),
                f"on_the_fly_fine_smoother_q{p + 1}": (ON_THE_FLY, p + 1)}
    for name, (g, qs) in settings.items():
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        mg = PreconditionMG(p, nq, 0, n, deform=0.05, geometry=g, fine_smoother_n_q_points_1d=qs)
        torch.cuda.synchronize()
        t_setup = time.perf_counter() - t0
        A = mg.operator()
        b = A.rhs(1)
        A.zero_constrained(b)
        x = A.initialize_dof_vector()
        _timed_solve(A, x, b, mg, 1e-6, 500)  # warm-up
        t8, c8 = _timed_solve(A, x, b, mg, 1e-8, 500)
        t10, c10 = _timed_solve(A, x, b, mg, 1e-10, 500)
        forms[name] = {"mg_setup_s": t_setup, "cg_mg_its_1e-10": c10.last_step(),
                       "cg_mg_s_1e-10": t10, "cg_mg_its_1e-8": c8.last_step(),
                       "cg_mg_s_1e-8": t8,
                       "mg_levels": [(mg.level(l)["degree"], mg.level(l)["n_cells"][0])
                                     for l in range(mg.n_levels())]}
        del mg, A, b, x
        torch.cuda.empty_cache()
    fast = min(forms, key=lambda k: forms[k]["cg_mg_s_1e-8"])
    g, qs = settings[fast]
    mg = PreconditionMG(p, nq, 0, n, deform=0.05, geometry=g, fine_smoother_n_q_points_1d=qs)
    A = mg.operator()
    b = A.rhs(1)
    A.zero_constrained(b)
    x = A.initialize_dof_vector()
    _timed_solve(A, x, b, mg, 1e-10, 500)
    x_ref = A.initialize_dof_vector()
    _timed_solve(A, x_ref, b, mg, 1e-13, 200)
    xyz = A.dof_coordinates()
    u = torch.sin(math.pi * xyz[:, 0]) * torch.sin(math.pi * xyz[:, 1]) * torch.sin(math.pi * xyz[:, 2])
    err_exact = ((x - u).abs().max() / u.abs().max()).item()
    del xyz, u
    inv = A.compute_inverse_diagonal()
    xj = A.initialize_dof_vector()
    tj, cj = _timed_solve(A, xj, b, DiagonalMatrix(inv), 1e-8, 100000)
    f = forms[fast]
    out = {"workload": f"BP3 Q{p} Gauss q={nq}, deformed {n}^3 cells, manufactured sin RHS",
           "n_dofs": A.m(), "form": fast, "forms": forms, "mg_levels": f["mg_levels"],
           "mg_setup_s": f["mg_setup_s"], "cg_mg_its_1e-10": f["cg_mg_its_1e-10"],
           "cg_mg_s_1e-10": f["cg_mg_s_1e-10"], "cg_mg_its_1e-8": f["cg_mg_its_1e-8"],
           "cg_mg_s_1e-8": f["cg_mg_s_1e-8"],
           "cg_jacobi_its_1e-8": cj.last_step(), "cg_jacobi_s_1e-8": tj,
           "speedup_1e-8": tj / f["cg_mg_s_1e-8"],
           "cg_mg_err_vs_fp64_1e-10": _rel(x, x_ref), "cg_jacobi_err_vs_fp64_1e-8": _rel(xj, x_ref),
           "nodal_max_err_vs_exact": err_exact}
    del mg, A, b, x, x_ref, inv, xj
    torch.cuda.empty_cache()
    return out


def bench_batch(count=64, seed=2):
    """Batched solves: `count` BP5 problems (cells per direction log-uniform
    in [4, 32], degree uniform in 2..6, SplitMix64 seed 2), per-instance
    uniform[-1,1] right-hand side, per-instance Jacobi-CG to 1e-8, all in one
    batch (hipGraph of CG steps, autotuned tile per degree), next to the same
    instances solved one after another with mfx_cg_solve (each on its
    operator with stored metric terms and on an on-the-fly one; the speedup is
    against the faster of the two)."""
    import torch

    from benchmarks_amd.laplace import (BatchedLaplace, DiagonalMatrix, ReductionControl,
                                        SolverCG, batch_instances, random_vector)
    inst = batch_instances(count, seed)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    B = BatchedLaplace(inst, autotune=True)
    torch.cuda.synchronize()
    t_setup = time.perf_counter() - t0
    b = random_vector(B.m(), seed)
    B.zero_constrained(b)
    inv = B.compute_inverse_diagonal()
    x = B.initialize_dof_vector()
    B.solve(x, b, inv, rel_tol=1e-2)  # warm-up (kernel loading)
    res = {}
    for graph in (True, False):
        x.zero_()
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        ctls = B.solve(x, b, inv, rel_tol=1e-8, use_graph=graph)
        torch.cuda.synchronize()
        res["graph" if graph else "direct"] = (time.perf_counter() - t0, ctls)
    # the same solves one after another (mfx_cg_solve), on each instance's
    # operator with stored metric terms and on an on-the-fly one
    from benchmarks_amd.laplace import LaplaceOperator
    seq = {}
    for form in ("stored", "on_the_fly"):
        t_seq, steps_seq = 0.0, []
        for i, (p, n) in enumerate(inst):
            a, e = B.offsets[i], B.offsets[i + 1]
            op = (B.instance_operator(i) if form == "stored" else
                  LaplaceOperator(p, p + 1, 1, n, deform=0.05, geometry=ON_THE_FLY))
            bi, ii = b[a:e].clone(), inv[a:e].clone()
            xi = op.initialize_dof_vector()
            SolverCG(ReductionControl(100000, 1e-300, 1e-2)).solve(op, xi, bi, DiagonalMatrix(ii))
            xi.zero_()
            c = ReductionControl(100000, 1e-300, 1e-8)
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            SolverCG(c).solve(op, xi, bi, DiagonalMatrix(ii))
            torch.cuda.synchronize()
            t_seq += time.perf_counter() - t0
            steps_seq.append(c.last_step())
        seq[form] = (t_seq, steps_seq)
    t_seq = min(v[0] for v in seq.values())
    steps_seq = seq["stored"][1]
    ctls = res["graph"][1]
    tuning = {}
    for p in sorted({p for p, _ in inst}):
        t = B.tuning(p)
        v, d = t["variant"], t["default_variant"]
        tuning[p] = {"cells": t["n_cells"], "chosen_geometry": t["geometry"][v],
                     "chosen_cells_per_wg_or_patch": t["cells_per_workgroup"][v],
                     "chosen_prefetch": t["prefetch"][v], "ms_chosen": t["ms"][v],
                     "ms_default": t["ms"][d],
                     "ms_per_variant": {
                         (f"{g} {c} cells per workgroup, prefetch {pf}" if g == "stored"
                          else f"{g} patch of {c} cells"): ms
                         for g, c, pf, ms in zip(t["geometry"], t["cells_per_workgroup"],
                                                 t["prefetch"], t["ms"])}}
    out = {"workload": f"{count} BP5 instances, cells/dir log-uniform 4..32, degree 2..6, "
                       f"seed {seed}, Jacobi-CG to 1e-8 each",
           "n_dofs": B.m(), "n_cells": sum(n ** 3 for _, n in inst),
           "setup_s": t_setup, "batch_graph_s": res["graph"][0], "batch_direct_s": res["direct"][0],
           "sequential_stored_s": seq["stored"][0], "sequential_on_the_fly_s": seq["on_the_fly"][0],
           "speedup_vs_sequential": t_seq / res["graph"][0],
           "steps_max": max(c.last_step() for c in ctls),
           "steps_total": sum(c.last_step() for c in ctls),
           "steps_differing_from_sequential": sum(1 for c, s in zip(ctls, steps_seq)
                                                  if c.last_step() != s),
           "autotune": tuning}
    del B, b, inv, x
    torch.cuda.empty_cache()
    return out


def bench_learned(n=64, p=4, n_fields=4096, mse_steps=512, energy_steps=1024, degree=4, seed=3):
    """Learned-preconditioner FCG (configuration C5): Q4 BP5 (GLL, on-the-fly
    geometry) on n^3 deformed cells.  Two-grid preconditioner: `degree`
    Chebyshev(Jacobi) steps (FP32), the U-Net as the coarse solve on the
    node grid of Q1 on (n/2)^3 cells (restricted residual in, prolongated
    correction out, energy-optimal weight), `degree` Chebyshev steps again.
    The network is trained on `n_fields` (residual, error) pairs of that Q1
    operator, solved by its FP64 multigrid CG to 1e-10: half are smooth
    coarse fields (32 random Fourier modes, wave numbers up to n/4,
    SplitMix64 seed 3), half restricted residuals of smooth fine fields
    (wave numbers up to n/2) after the cycle's Chebyshev pre-smoothing.
    Mean squared error (one pass over the pairs at batch 8), then the
    energy-norm loss.  Flexible CG to 1e-8 on a fresh smooth right-hand
    side with the multigrid fallback armed, next to the same cycle without
    the network, Jacobi-CG and multigrid CG; errors against an FP64
    solution certified to 1e-12 by the FP64 residual of the multigrid CG."""
    import torch

    from benchmarks_amd.laplace import DiagonalMatrix, LearnedPreconditioner, PreconditionMG
    from benchmarks_amd.learned import _stream, smooth_rhs, train_coarse
    mg = PreconditionMG(p, p + 1, 1, n, deform=0.05, geometry=ON_THE_FLY)
    A = mg.operator()
    coarse_mg = PreconditionMG(1, 2, 1, n // 2, deform=0.05)  # Q1 on the coarse box
    net = LearnedPreconditioner(seed)
    st = train_coarse(net, coarse_mg, n_fields=n_fields, mse_steps=mse_steps,
                      energy_steps=energy_steps, seed=seed, fine=A, smoother_degree=degree)
    b = smooth_rhs(A, A.dof_coordinates(), _stream(seed + 1), 32)
    x_ref = A.initialize_dof_vector()
    _timed_solve(A, x_ref, b, mg, 1e-12, 200)
    net.set_mode(degree, True)
    net.set_fallback(mg)
    without = LearnedPreconditioner(seed)
    without.set_mode(degree, False)
    x = A.initialize_dof_vector()
    out = {"workload": f"BP5 Q{p} GLL, deformed {n}^3 cells, smooth RHS (32 Fourier modes), "
                       f"flexible CG to 1e-8",
           "n_dofs": A.m(),
           "network_grid": f"Q1 on {n // 2}^3 cells ({st['coarse_dims'][0]}^3 nodes)",
           "training": f"{n_fields} FP64 {st['data_solver']} solves on the coarse grid "
                       f"({n_fields - st['n_restricted_fields']} coarse fields up to k "
                       f"{st['k_max']}, {st['n_restricted_fields']} restricted pre-smoothed "
                       f"fine fields up to k {st['fine_k_max']}), "
                       f"{mse_steps} MSE steps (batch 8) + {energy_steps} energy-norm steps "
                       f"(batch 2)",
           "n_training_pairs": n_fields,
           "data_s": st["data_s"], "train_mse_s": st["mse"]["seconds"],
           "train_energy_s": st["energy"]["seconds"],
           "mse_loss_first_last": [st["mse"]["loss_first"], st["mse"]["loss_last"]],
           "energy_loss_first_last": [st["energy"]["loss_first"], st["energy"]["loss_last"]],
           "smoother_degree": degree}
    for name, P, steps in [("learned_fcg", net, 2000), ("chebyshev_fcg_without_network", without, 5000),
                           ("jacobi_cg", DiagonalMatrix(A.compute_inverse_diagonal()), 100000),
                           ("multigrid_cg", mg, 200)]:
        _timed_solve(A, x, b, P, 1e-4, steps)  # warm-up
        t, c = _timed_solve(A, x, b, P, 1e-8, steps)
        out[name] = {"steps": c.last_step(), "seconds": t, "err_vs_fp64": _rel(x, x_ref)}
        if P is net:
            out[name]["fallback_step"] = net.fallback_step
    out["learned_speedup_vs_jacobi"] = out["jacobi_cg"]["seconds"] / out["learned_fcg"]["seconds"]
    out["learned_speedup_vs_chebyshev"] = (out["chebyshev_fcg_without_network"]["seconds"]
                                          / out["learned_fcg"]["seconds"])
    del mg, A, net, without, x, x_ref, b, coarse_mg
    torch.cuda.empty_cache()
    return out


def stream_copy_GBs(n=1 << 28, reps=10):
    """Measured HBM ceiling: device-to-device copy of 2 GiB (read + write bytes)."""
    import torch
    a = torch.ones(n, dtype=torch.float64, device="cuda")
    b = torch.empty_like(a)
    b.copy_(a)
    e0, e1 = _events()
    e0.record()
    for _ in range(reps):
        b.copy_(a)
    e1.record()
    torch.cuda.synchronize()
    t = e0.elapsed_time(e1) * 1e-3 / reps
    del a, b
    torch.cuda.empty_cache()
    return 16.0 * n / t * 1e-9


def _cpu_worker(args):
    """One host process: its slice of the full apply (cells [lo, hi) of the
    degree's mesh, stored metric terms, E-vector form), `calls` applies of
    the reference kernel after one untimed one; returns (cells processed,
    seconds).  The inputs are generated in the process, so nothing is shared.
    The reference kernel returns before its delete[] and leaks its three
    nq^3-per-cell scratch arrays on every call; `calls` is capped by the
    caller so that the leak stays bounded, and the memory goes with the
    process."""
    p, cells, calls, use_ref, seed = args
    import numpy as np

    from oracle import oracle as O
    nq = p + 1
    _, D, _, _ = O.basis_tables(p, nq, O.GLL)
    rng = np.random.default_rng(seed)
    G = rng.standard_normal(cells * 6 * nq ** 3)
    u = rng.standard_normal(cells * nq ** 3)
    out = np.zeros(cells * nq ** 3)
    if use_ref:
        fn = O.ref_lib(fast=True).ref_bk5_serial
        run = lambda: fn(nq, cells, D, G, u, out)  # noqa: E731
    else:
        run = lambda: O.bk5_evec(nq, cells, D, G, u)  # noqa: E731
    run()  # first touch of the scratch pages, untimed
    t0 = time.perf_counter()
    for _ in range(calls):
        run()
    return calls * cells, time.perf_counter() - t0


def host_cpu_info():
    """Host CPU model (/proc/cpuinfo), os.cpu_count() and the CPUs this
    process may run on (sched_getaffinity)."""
    model = "unknown"
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    model = line.split(":", 1)[1].strip()
                    break
    except OSError:
        pass
    try:
        affinity = len(os.sched_getaffinity(0))
    except AttributeError:
        affinity = os.cpu_count() or 1
    return {"cpu_model": model, "os_cpu_count": os.cpu_count(), "affinity_cpus": affinity,
            "omp_num_threads": os.environ.get("OMP_NUM_THREADS")}


def cpu_baseline(degrees, budget_s=12.0, leak_cap_bytes=1 << 30):
    """The reference's own serial BK5 kernel
    (sum_factorization/include/kernels/BK5/serial_kernels.hpp:9-87, built by
    oracle/Makefile into oracle/_ref/) on the host's CPU share: one process
    per core, each on its own slice of the degree's FULL mesh (E / T cells,
    hundreds of MB per process, far beyond the last-level cache), so the
    timed work is the whole apply at the configured size, not a
    cache-resident sample.  E-vector form: the reference CPU path has no
    gather or scatter.  The core count is the CPU share the host grants
    this process: OMP_NUM_THREADS when set (a GPU box sets it to the cores
    allotted to its GPU), else the affinity mask.  Each degree's applies are
    repeated to about budget_s / len(degrees) seconds, within the reference
    kernel's per-call leak cap."""
    import multiprocessing as mp

    from oracle import oracle as O
    use_ref = True
    try:
        O.ref_lib(fast=True)
    except (FileNotFoundError, OSError):
        use_ref = False
    info = host_cpu_info()
    share = info["omp_num_threads"]
    procs = int(share) if share and share.isdigit() and int(share) > 0 else info["affinity_cpus"]
    procs = max(1, min(procs, info["affinity_cpus"]))
    per_deg = budget_s / len(degrees)
    t_tot, n_tot, samples = 0.0, 0, []
    ctx = mp.get_context("fork")
    for p in degrees:
        nq = p + 1
        n = CELLS[p]
        E, N = n ** 3, (n * p + 1) ** 3
        base, extra = divmod(E, procs)
        slices = [base + (1 if i < extra else 0) for i in range(procs)]
        # one apply of the largest slice, to size the repetitions
        with ctx.Pool(procs, maxtasksperchild=1) as pool:
            probe = pool.map(_cpu_worker, [(p, c, 1, use_ref, 100 + i)
                                           for i, c in enumerate(slices)])
        t_one = max(r[1] for r in probe)
        leak_per_call = 3 * 8 * nq ** 3 * max(slices)
        calls = max(1, min(int(per_deg / max(t_one, 1e-6)), leak_cap_bytes // leak_per_call))
        with ctx.Pool(procs, maxtasksperchild=1) as pool:
            res = pool.map(_cpu_worker, [(p, c, calls, use_ref, 100 + i)
                                         for i, c in enumerate(slices)])
        wall = max(r[1] for r in res)
        t_tot += wall / calls
        n_tot += N
        slice_mb = max(slices) * (6 + 2) * nq ** 3 * 8 / 2 ** 20
        samples.append(f"p={p}: {calls} full applies of {E} cells ({max(slices)} cells, "
                       f"{slice_mb:.0f} MB per process) in {wall:.1f}s")
    return {"value": n_tot / t_tot * 1e-9, "unit": "GDoF/s", "cores": procs,
            "kind": "reference" if use_ref else "port",
            "host": info,
            "sample": f"{'reference' if use_ref else 'oracle'} BK5 serial kernel (E-vector, no "
                      f"gather/scatter, stored metric terms), {procs} processes (the host's CPU "
                      "share for this GPU), each on 1/" + str(procs) + " of the full p=4,6,8 "
                      "meshes; value = sum N / sum of the full-apply times; " +
                      "; ".join(samples)}


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=100)
    ap.add_argument("--warmup", type=int, default=10)
    ap.add_argument("--degrees", default="4,6,8")
    ap.add_argument("--extra-degrees", default=None,
                    help="degrees reported per degree but outside the p=4-8 aggregate "
                         "(default: 2 when --degrees is left at 4,6,8, else none)")
    ap.add_argument("--geometry", choices=["both", "stored", "otf"], default="both")
    ap.add_argument("--no-cg", action="store_true")
    ap.add_argument("--no-deterministic", action="store_true",
                    help="skip timing the deterministic scatter (one apply kernel per mode, "
                         "for counter profiles)")
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-c1", action="store_true", help="skip the 35937-DoF BP3 unit-cube case")
    ap.add_argument("--no-bp3-reference", action="store_true",
                    help="skip the reference's published BP3 problem (67.6M DoFs)")
    ap.add_argument("--no-c3", action="store_true", help="skip the 135M-DoF mixed-precision solve")
    ap.add_argument("--no-batch", action="store_true", help="skip the 64-instance batched solve")
    ap.add_argument("--no-learned", action="store_true", help="skip the learned-preconditioner solve")
    args = ap.parse_args()
    if args.gpus != 1 or int(os.environ.get("WORLD_SIZE", "1")) != 1:
        print("bench.py measures one GPU: the multi-GPU path (slab decomposition with halo "
              "exchange) is designed but not built; run with --gpus 1", file=sys.stderr)
        sys.exit(2)
    degrees = [int(d) for d in args.degrees.split(",")]
    modes = {"both": [STORED, ON_THE_FLY], "stored": [STORED], "otf": [ON_THE_FLY]}[args.geometry]
    # host baseline first, before anything initialises the GPU in this process
    cpu = None if args.no_cpu_baseline else cpu_baseline(degrees)
    import torch
    torch.cuda.synchronize()
    stream_copy = stream_copy_GBs()
    per = [bench_degree(p, args.steps, args.warmup, not args.no_cg, modes, not args.no_deterministic)
           for p in degrees]
    if args.extra_degrees is None:
        args.extra_degrees = "2" if args.degrees == "4,6,8" else ""
    extra = [int(d) for d in args.extra_degrees.split(",") if d.strip()]
    per_extra = [bench_degree(p, args.steps, args.warmup, not args.no_cg, modes,
                              not args.no_deterministic) for p in extra
                 if p not in degrees]
    t_sum = sum(r["ms_vmult"] for r in per) * 1e-3
    n_sum = sum(r["n_dofs"] for r in per)
    # the dominant kernel: the longest median element-kernel time among the
    # kernels the aggregate runs (each degree's faster mode)
    dom = max(per, key=lambda r: r["modes"][r["geometry"]]["ms_kernel"])
    dm = dom["modes"][dom["geometry"]]
    t_k = dm["ms_kernel"] * 1e-3
    bw, flops = dm["bytes_alg"] / t_k, dm["flops_alg"] / t_k
    # the roof that bounds the kernel: FP64 arithmetic (on the vector ALUs)
    # when its arithmetic intensity exceeds the machine balance
    # (78.6 TFLOP/s / 8 TB/s), else HBM
    intensity = dm["flops_alg"] / dm["bytes_alg"]
    if intensity > FP64_PEAK / HBM_PEAK:
        roof = {"bound": "fp64-valu", "achieved": flops * 1e-12, "peak": FP64_PEAK * 1e-12,
                "unit": "TFLOP/s", "frac": flops / FP64_PEAK}
    else:
        roof = {"bound": "hbm", "achieved": bw * 1e-9, "peak": HBM_PEAK * 1e-9,
                "unit": "GB/s", "frac": bw / HBM_PEAK}
    roof.update({"traffic": None, "kernel": f"BK5 apply p={dom['p']} ({dom['geometry']})",
                 "vmult_frac_of_stored_G_hbm_roofline": {
                     r["p"]: r["frac_of_stored_G_hbm_roofline"] for r in per
                     if "frac_of_stored_G_hbm_roofline" in r},
                 # the stored-metric apply is memory-bound: its own kernel's
                 # algorithmic bytes per second against 8 TB/s
                 "stored_kernel_hbm_frac": {
                     r["p"]: r["modes"]["stored"]["kernel_GBs"] * 1e9 / HBM_PEAK for r in per
                     if "stored" in r["modes"]},
                 "ms_per_launch": dm["ms_kernel"], "ms_per_launch_best": dm["ms_kernel_best"],
                 "ms_vmult_median": dm["ms_vmult_median"],
                 "timing": f"median of {dm['kernel_samples']} per-call HIP event pairs on the "
                           "launch stream",
                 "timing_valid": dm["kernel_timing_valid"],
                 "flops_per_launch": dm["flops_alg"],
                 "bytes_per_launch": dm["bytes_alg"], "flop_per_byte": intensity,
                 "hbm_GBs": bw * 1e-9, "hbm_frac": bw / HBM_PEAK,
                 "fp64_TFLOPs": flops * 1e-12, "fp64_frac": flops / FP64_PEAK,
                 "note": "FP64 arithmetic on the vector ALUs (the kernel issues no MFMA); "
                         "78.6 TFLOP/s is MI355X's FP64 peak, vector and matrix alike"})
    out = {
        "metric": "BP5 matvec GDoF/s at p=4-8 (aggregate over p=4,6,8); CG time-to-1e-8 per degree",
        "value": n_sum / t_sum * 1e-9,
        "unit": "GDoF/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": t_sum * 1e3,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64",
        "data": "synthetic (deformed unit-cube mesh, SplitMix64 seed-1 input)",
        "config": {"workload": "BP5 GLL q=p+1, deformed unit cube, p=4/6/8 on 80^3/52^3/40^3 "
                               "cells (33.1M / 30.7M / 33.1M DoFs), FP64 vmult; metric terms stored or "
                               "on the fly, faster per degree",
                   "degrees": degrees, "geometry": {r["p"]: r["geometry"] for r in per},
                   "parallelism": "single GPU"},
        "roofline": roof,
        "per_degree": per,
        "per_degree_outside_aggregate": per_extra,
        "stream_copy_GBs": stream_copy,
    }
    traffic = measured_traffic(dom)
    if traffic is not None:
        out["roofline"]["traffic"] = traffic[0]
        out["roofline"]["traffic_source"] = traffic[1]
    if not args.no_cg and not args.no_c1:
        out["bp3_unit_cube"] = bench_c1()
    if not args.no_cg and not args.no_bp3_reference:
        out["bp3_reference_problem"] = bench_bp3_reference()
    if not args.no_cg and not args.no_c3:
        out["mixed_precision_bp3"] = bench_c3()
    if not args.no_cg and not args.no_batch:
        out["batched_solves"] = bench_batch()
    if not args.no_cg and not args.no_learned:
        out["learned_preconditioner"] = bench_learned()
    if cpu is not None:
        out["cpu_baseline"] = cpu
    print(json.dumps(out))


def measured_traffic(dom):
    """HBM bytes per launch of the dominant kernel -- this degree and
    geometry mode -- from its own committed rocprofv3 FETCH_SIZE/WRITE_SIZE
    summary (profiles/), with the file it came from; None when that kernel
    has no summary."""
    name = f"bk5_apply_bp5_p{dom['p']}_{dom['geometry']}_traffic.md"
    path = os.path.join(ROOT, "profiles", name)
    if not os.path.exists(path):
        return None
    for line in open(path):
        if line.startswith("APPLY_TRAFFIC_BYTES"):
            return float(line.split()[-1]), "profiles/" + name
    return None


if __name__ == "__main__":
    main()
