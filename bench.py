#!/usr/bin/env python3
"""Seconds per BFGS iteration (eigensolve + adjoint + force) on one MI355X.

Workload inverse_24c_p5: domain [-12,12]^3, 24^3 cells, degree 5 (121^3 =
1,771,561 nodes), v_xc on the linear 49^3 child mesh, soft-Coulomb wells
(Z=3 at the origin, Z=1 at (0,0,3)), 8 occupied + 4 buffer orbitals,
Chebyshev degree 30, FP64 Cholesky-QR + Rayleigh-Ritz, adjoint MINRES and
force, L-BFGS with the CP line search and one line-search step, so one
iteration is two getForceVector evaluations.  Inputs are synthetic (the
target density is the FP64 ground state of the wells alone; v_xc starts at a
seeded sum of 8 Gaussians).

The mixed-precision run (FP32 sum-factorised cell operator, defect-corrected
FP32 Chebyshev filter, FP64 MINRES recurrence whose cell operator drops to
FP32 once the residual is near the tolerance, FP64 everything else) is timed
over K iterations after W warm-up iterations, then the FP64 run on the same
problem.  Every library call returns only after its work on the GPU stream
has completed, so host wall-clock brackets are synchronised.

After the headline line's measurements, `detail.c3` times one iteration of
the batched workload (40^3 cells, degree 4, 4.17 M nodes, 64 occupied + 16
buffer states) per precision: its two getForceVector evaluations, at the
starting potential and at one step along the negative force (the CP line
search's first point), with the force error of mixed against FP64 at both.
"""
import argparse
import json
import os
import sys
import time

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, HERE)

METRIC = "s per BFGS iter (eigen+adjoint+force), mixed vs FP64 on GPU, force err ≤1e-6"
HBM_PEAK_GBS = 8000.0
FP32_PEAK_TFLOPS = 157.3  # MI355X published FP32 vector / dense matrix peak
FP64_PEAK_TFLOPS = 78.6   # MI355X published FP64 vector / dense matrix peak


def sf_flops_per_cell_column(p):
    """Flops of the sum-factorised cell product per cell and column.  Every 1D
    contraction y = A x (A of R x C, centro-symmetric) runs in even-odd form:
    C/2 sums and differences of the input, ceil(R/2) even rows of
    ceil(C/2) multiply-adds, floor(R/2) odd rows of floor(C/2), and one sum
    and one difference per output pair.  Two tables into one output (the
    kinetic D + M lines) share the output pairs.  A multiply-add counts 2."""
    n1, q = p + 1, p + 3

    def split(c):
        return 2 * (c // 2)

    def contract(r, c, tables=1):
        fma = tables * (((r + 1) // 2) * ((c + 1) // 2) + (r // 2) * (c // 2))
        return 2 * fma + 2 * (r // 2)

    x_lines = n1 ** 2 * (split(n1) + contract(q, n1) + 2 * contract(n1, n1))
    y_lines = (n1 * q * (split(n1) + contract(q, n1))
               + n1 ** 2 * (2 * split(n1) + contract(n1, n1) + contract(n1, n1, 2)))
    z_lines = (q ** 2 * (split(n1) + contract(q, n1) + q + split(q) + contract(n1, q))
               + n1 ** 2 * (2 * split(n1) + contract(n1, n1, 2)))
    y_back = n1 * q * (split(q) + contract(n1, q))
    x_back = n1 ** 2 * (split(q) + contract(n1, q) + 2 * n1)  # + (h/4) kinetic, fused
    return x_lines + y_lines + z_lines + y_back + x_back


# HBM bytes per launch of the cell-product kernels from two rocprofv3 --pmc runs
# (FETCH_SIZE, WRITE_SIZE) of `bench.py --kernels-only --shape ...`, FETCH_SIZE
# scaled by the copy calibration (x1.926), WRITE_SIZE as read; the summaries
# with the commands are profiles/cell_plane_pmc.md (shape 1 4 4 2) and
# profiles/cell_gemm_inverse_24c_p5_pmc.md (2 16 4 0 and 1 16 0 1).
MEASURED_TRAFFIC = {
    ("inverse_24c_p5", "k_cell_plane<float,float,5,false,true>"): 276.7e6,
    ("inverse_24c_p5", "k_cell_plane<double,double,5,false,true>"): 554.4e6,
    ("batched_40c_p4", "k_cell_plane<float,float,4,false,true>"): 4263.6e6,
    ("batched_40c_p4", "k_cell_plane<double,double,4,false,true>"): 9255.1e6,
    ("inverse_24c_p5", "k_cell_gemm<float,float,5,1>"): 2613e6,
    ("inverse_24c_p5", "k_cell_symm<float,float,5,1>"): 1691e6,
}


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def fma_probe(lib, chains=16):
    """TFLOP/s of an FMA loop with `chains` independent chains per thread,
    FP64 and unpacked FP32 (idft_fma_probe)."""
    import ctypes as C
    from invdft_amd import abi
    fn = lib.idft_fma_probe
    fn.restype = C.c_int
    fn.argtypes = [C.c_int32, C.c_int32, C.POINTER(C.c_double)]
    out = {}
    for name, prec in (("fp64", abi.FP64), ("fp32", abi.MIXED)):
        v = C.c_double()
        rc = fn(prec, chains, C.byref(v))
        if rc != 0:
            raise RuntimeError(f"idft_fma_probe failed ({rc})")
        out[name] = round(v.value, 2)
    log(f"attainable FMA rate ({chains} chains per thread): {out} TFLOP/s")
    return out


def mixed_vs_fp64_errors(lib, prob, x, tol_kw):
    """getForceVector at potential x in both precisions with the given
    tolerances: relative force and density (L2 over the quadrature values)
    errors, the largest eigenvalue difference over the occupied states (Ha)
    and the relative loss difference of mixed against FP64."""
    from invdft_amd import abi
    out = {}
    for prec in (abi.MIXED, abi.FP64):
        c = prob.context(lib, precision=prec, **tol_kw)
        f, L = c.get_force(x)
        out[prec] = (f, L, c.eigenvalues(), c.density())
        c.close()
    (fm, lm, em, rm), (ff, lf, ef, rf) = out[abi.MIXED], out[abi.FP64]
    nocc = int(round(prob.desc.n_electrons / 2))
    return {"force": float(np.linalg.norm(fm - ff) / np.linalg.norm(ff)),
            "eigenvalues_occupied_Ha": float(np.max(np.abs(em[:nocc] - ef[:nocc]))),
            "density_l2": float(np.linalg.norm(rm - rf) / np.linalg.norm(rf)),
            "loss": float(abs(lm - lf) / abs(lf))}


def run_bfgs(lib, prob, precision, warmup, steps, tol_kw):
    from invdft_amd import abi
    ctx = prob.context(lib, precision=precision, **tol_kw)
    ctx.set_potential(prob.vxc0)  # cell operator for the autotuner (untimed)
    log("  autotuning the FP64 cell operator")
    tuned = {"fp64": ctx.autotune_apply(prob.desc.n_eig, abi.FP64)}
    if precision == abi.MIXED:
        log("  autotuning the FP32 cell operator")
        tuned["fp32"] = ctx.autotune_apply(prob.desc.n_eig, abi.MIXED)
    log(f"  autotuned cell-product tile shapes: {tuned}")
    t0 = time.perf_counter()
    if warmup > 0:
        ctx.bfgs_solve(ls_type=abi.LS_CP, max_iter=warmup)
        ctx.set_initial_guess(ctx.get_solution())
    st0 = ctx.stats()
    log(f"  warmup {warmup} iterations: {time.perf_counter() - t0:.2f} s")
    loss, gnorm, n = ctx.bfgs_solve(ls_type=abi.LS_CP, max_iter=steps)
    th = ctx.bfgs_times_ms
    st1 = ctx.stats()
    timed_ms = th[n] - th[0]
    evals = st1["n_evaluations"] - st0["n_evaluations"]
    per_eval = {k: (st1[k] - st0[k]) / max(evals, 1)
                for k in ("applies_fp64", "applies_fp32", "apply_cols_fp64", "apply_cols_fp32")}
    log(f"  timed {n} iterations: {timed_ms:.1f} ms, loss {loss[0]:.4e} -> {loss[-1]:.4e}, "
        f"last eval: passes={st1['cheb_passes']} minres_max={st1['minres_iters_max']} "
        f"refinements={st1['refinements']} t_eig={st1['t_eigen_ms']:.1f} "
        f"t_adj={st1['t_adjoint_ms']:.1f} t_force={st1['t_force_ms']:.1f} ms")
    return ctx, dict(iters=n, timed_ms=timed_ms, s_per_iter=timed_ms / 1000.0 / n, loss=list(loss),
                     gnorm=list(gnorm), per_eval=per_eval, last=st1, evals=evals, tuned=tuned)


def _oracle_samples(olib, prob):
    """Oracle H_e build and one n_eig-column Loewdin apply (median of three)
    on prob's mesh (s)."""
    ctx = prob.context(olib)
    s = ctx.sizes
    t0 = time.perf_counter()
    ctx.set_veff_quad(prob.pot_base_q)
    t_build = time.perf_counter() - t0
    B = prob.desc.n_eig
    x = np.random.default_rng(0).standard_normal((s.n_nodes, B))
    # median of three applications: one is too noisy on shared host cores
    ts = []
    for _ in range(3):
        t0 = time.perf_counter()
        ctx.apply_hamiltonian(x)
        ts.append(time.perf_counter() - t0)
    t_apply = float(np.median(ts))
    ctx.close()
    return t_build, t_apply


def cpu_baseline(lib, prob, per_eval, evals_per_iter, tol_kw):
    """The oracle (FP64 CPU restatement) on the host cores.  The headline
    workload's evaluation is too long to time whole on the CPU (~5 min), so
    its value is a model: the oracle's H_e build and one n_eig-column apply
    on this mesh, timed, scaled by the GPU run's per-evaluation count of
    column applications plus two cell-matrix builds.  The model is checked
    where a whole evaluation is affordable: one full oracle getForceVector
    on the 16^3-cell degree-4 adjoint workload, timed, against the same
    model built from that run's own counts."""
    from oracle import oracle
    from invdft_amd import synthetic
    olib = oracle.load()
    cores = int(os.environ.get("OMP_NUM_THREADS", os.cpu_count() or 1))
    t_build, t_apply = _oracle_samples(olib, prob)
    B = prob.desc.n_eig
    cols = per_eval["apply_cols_fp64"] + per_eval["apply_cols_fp32"]
    t_eval = 2.0 * t_build + cols * t_apply / B
    # model check on the small workload: one whole evaluation, timed
    cfg1 = dict(synthetic.CONFIGS["adjoint_16c_p4"])
    p1 = synthetic.make_problem(lib, seed=1, target_tol=1e-10, **cfg1)
    c1 = p1.context(olib, **tol_kw)
    t0 = time.perf_counter()
    c1.get_force(p1.vxc0)
    t_meas = time.perf_counter() - t0
    st = c1.stats()
    c1.close()
    b1, a1 = _oracle_samples(olib, p1)
    t_model1 = 2.0 * b1 + st["apply_cols_fp64"] * a1 / p1.desc.n_eig
    log(f"  oracle C1 evaluation {t_meas:.2f} s measured, {t_model1:.2f} s modelled")
    return {"value": round(t_eval * evals_per_iter, 3), "unit": "s/iter", "cores": cores,
            "kind": "port",
            "sample": (f"FP64 oracle on this mesh: H_e build {t_build:.2f} s + one {B}-column "
                       f"Loewdin apply {t_apply:.2f} s (median of 3), scaled to {cols:.0f} column-applies and "
                       f"2 cell-matrix builds per evaluation, {evals_per_iter} evaluations per "
                       f"iteration"),
            "measured_check": {"workload": "adjoint_16c_p4", "s_per_eval_measured": round(t_meas, 3),
                               "s_per_eval_model": round(t_model1, 3),
                               "model_rel_error": round(t_model1 / t_meas - 1.0, 4),
                               "column_applies": st["apply_cols_fp64"]}}


def c3_leg(lib, cheb_tol):
    """One BFGS iteration of the batched workload per precision: getForceVector
    at the starting potential x0 and at x0 - g0 (the CP line search's first
    point), each context autotuned first (untimed)."""
    from invdft_amd import abi, synthetic
    cfg = dict(synthetic.CONFIGS["batched_40c_p4"])
    t0 = time.perf_counter()
    prob = synthetic.make_problem(lib, seed=2, target_tol=1e-10, **cfg)
    log(f"  C3 set-up: {time.perf_counter() - t0:.1f} s")
    kw = dict(cheb_tol=cheb_tol, initial_tol_cheb=cheb_tol)
    out, forces, states = {}, {}, {}
    B = prob.desc.n_eig
    for name, prec in (("mixed", abi.MIXED), ("fp64", abi.FP64)):
        ctx = prob.context(lib, precision=prec, **kw)
        ctx.set_potential(prob.vxc0)
        tuned = {"fp64": ctx.autotune_apply(B, abi.FP64)}
        if prec == abi.MIXED:
            tuned["fp32"] = ctx.autotune_apply(B, abi.MIXED)
        x0 = prob.vxc0.copy()
        t0 = time.perf_counter()
        f0, l0 = ctx.get_force(x0.copy())
        st0 = ctx.stats()
        states[name] = (ctx.eigenvalues(), ctx.density())
        f1, l1 = ctx.get_force(x0 - f0)
        dt = time.perf_counter() - t0
        st1 = ctx.stats()
        forces[name] = (f0, f1)
        ms64, cell64 = ctx.profile_apply(B, abi.FP64, reps=10)
        out[name] = {"s_per_iter": round(dt, 3), "loss": [l0, l1],
                     "eigen_ms": [round(st0["t_eigen_ms"], 1), round(st1["t_eigen_ms"], 1)],
                     "adjoint_ms": [round(st0["t_adjoint_ms"], 1), round(st1["t_adjoint_ms"], 1)],
                     "minres_iters_max": [st0["minres_iters_max"], st1["minres_iters_max"]],
                     "minres_column_steps": st1["minres_column_steps"],
                     "minres_compactions": st1["minres_compactions"],
                     "tile_shapes": tuned,
                     "fp64_cell_product_ms": round(cell64, 4), "fp64_operator_ms": round(ms64, 4)}
        log(f"  C3 {name}: {out[name]}")
        ctx.close()
    fm, ff = forces["mixed"], forces["fp64"]
    err = [float(np.linalg.norm(a - b) / np.linalg.norm(b)) for a, b in zip(fm, ff)]
    nocc = int(round(prob.desc.n_electrons / 2))
    (em, rm), (ef, rf) = states["mixed"], states["fp64"]
    state_err = {"eigenvalues_occupied_Ha": float(np.max(np.abs(em[:nocc] - ef[:nocc]))),
                 "density_l2": float(np.linalg.norm(rm - rf) / np.linalg.norm(rf))}
    # roofline of this workload's FP64 cell product (the FP64 run's tuned
    # shape), measured live by idft_profile_apply as for the headline kernel
    roof = None
    sh = out["fp64"]["tile_shapes"]["fp64"]
    if sh["kernel"] == 2:
        p, nc = prob.desc.degree, prob.desc.n_cells
        cells, N = nc ** 3, (nc * p + 1) ** 3
        flops = cells * B * sf_flops_per_cell_column(p)
        nbytes = 8 * (cells * (p + 3) ** 3 + N * (B + 1) + cells * (p + 1) ** 3 * B)
        ms = out["fp64"]["fp64_cell_product_ms"]
        ach = flops / (ms * 1e-3) / 1e12
        kname = f"k_cell_plane<double,double,{p},false,true>"
        roof = {"bound": "valu", "kernel": kname,
                "achieved": round(ach, 2), "peak": FP64_PEAK_TFLOPS, "unit": "TFLOP/s",
                "frac": round(ach / FP64_PEAK_TFLOPS, 4),
                "traffic": MEASURED_TRAFFIC.get(("batched_40c_p4", kname)), "ms_per_launch": ms,
                "flops_per_launch": flops, "bytes_per_launch": nbytes,
                "achieved_GBs": round(nbytes / (ms * 1e-3) / 1e9, 1)}
    return {"workload": "batched_40c_p4", "nodes": int(prob.desc.n_cells * prob.desc.degree + 1) ** 3,
            "orbitals": B, "evals_per_iter": 2, "mixed": out["mixed"], "fp64": out["fp64"],
            "speedup_mixed_vs_fp64": round(out["fp64"]["s_per_iter"] / out["mixed"]["s_per_iter"], 3),
            "force_rel_err_mixed_vs_fp64": err,
            "state_err_mixed_vs_fp64_first_eval": state_err, "roofline": roof}


def c4_large(lib, evals):
    """The large gradient workload (32^3 cells, degree 5, 4.17 M nodes, 32
    orbitals, child 65^3): `evals` getForceVector evaluations with the FP64
    eigenvector block resident between the passes and with it checkpointed
    (FP32 copy, recomputed by one ChFSI pass for the backward pass); time per
    evaluation, the library's peak device memory and the force difference."""
    import ctypes as C
    from invdft_amd import abi, synthetic
    fn = lib.idft_device_memory
    fn.restype = C.c_int
    fn.argtypes = [C.POINTER(C.c_int64), C.POINTER(C.c_int64), C.c_int32]
    cur, peak = C.c_int64(), C.c_int64()
    cfg = dict(synthetic.CONFIGS["gradcheck_32c_p5"])
    t0 = time.perf_counter()
    prob = synthetic.make_problem(lib, seed=4, target_tol=1e-10, **cfg)
    log(f"set-up: {time.perf_counter() - t0:.1f} s")
    out, forces = {}, {}
    for ck in (0, 1):
        fn(C.byref(cur), C.byref(peak), 1)
        base = cur.value
        ctx = prob.context(lib, psi_checkpoint=ck, cheb_tol=1e-8, initial_tol_cheb=1e-8)
        t0 = time.perf_counter()
        fs = []
        for k in range(evals):
            f, L = ctx.get_force(prob.vxc0 * (1.0 + 0.02 * k))
            fs.append(f)
        dt = (time.perf_counter() - t0) / evals
        fn(C.byref(cur), C.byref(peak), 0)
        st = ctx.stats()
        out["checkpointed" if ck else "resident"] = {
            "s_per_eval": round(dt, 3), "peak_device_GiB": round((peak.value - base) / 2**30, 3),
            "psi_recomputes": st["psi_recomputes"], "t_eigen_ms": round(st["t_eigen_ms"], 1),
            "t_adjoint_ms": round(st["t_adjoint_ms"], 1)}
        forces[ck] = fs
        log(f"  psi_checkpoint={ck}: {out['checkpointed' if ck else 'resident']}")
        ctx.close()
    err = [float(np.linalg.norm(a - b) / np.linalg.norm(b)) for a, b in zip(forces[1], forces[0])]
    print(json.dumps({"workload": "gradcheck_32c_p5", "nodes": 161 ** 3, "orbitals": cfg["n_eig"],
                      "evals": evals, **out, "force_rel_diff": err}), flush=True)


def kernels_only(lib, cfg, shape, reps):
    """Operator kernels alone, for hardware-counter runs: the cell operator of
    the workload's mesh (soft-Coulomb potential) applied `reps` times to a
    block of n_eig columns in FP32 and FP64 at a fixed launch shape, after
    three Jacobi-preconditioner calls that stream a known number of bytes
    (read N*B*8 + N*8, write N*B*8) to calibrate the byte counters."""
    from invdft_amd import abi, synthetic
    d = abi.default_desc(lib, n_cells=cfg["n_cells"], degree=cfg["degree"],
                         half_width=cfg["half_width"], n_eig=cfg["n_eig"],
                         n_electrons=cfg["n_electrons"], precision=abi.MIXED)
    s = abi.geometry(lib, d)
    atoms = cfg["atoms"] if cfg["atoms"] != "random8" else synthetic.random_atoms(1)
    v = synthetic.soft_coulomb(abi.quad_points(lib, d), atoms)
    nq = s.n_cells * s.quad_per_cell
    ctx = abi.Context(lib, d, v, np.zeros(nq), np.ones(nq), np.ones(s.n_nodes))
    ctx.set_veff_quad(v)
    B = cfg["n_eig"]
    a = ctx.mv(B, np.random.default_rng(0).standard_normal((s.n_nodes, B)))
    b = ctx.mv(B)
    for _ in range(3):
        ctx.adj_precondition_jacobi(b, a)
    log(f"copy calibration: 3 x (read {s.n_nodes * B * 8 + s.n_nodes * 8} B, "
        f"write {s.n_nodes * B * 8} B)")
    out = {}
    for name, prec in (("fp32", abi.MIXED), ("fp64", abi.FP64)):
        ctx.set_apply_shape(prec, *shape)
        out[name] = ctx.profile_apply(B, prec, reps=reps)
        log(f"{name} shape {shape}: operator {out[name][0]:.4f} ms, cell product "
            f"{out[name][1]:.4f} ms")
    ctx.close()
    print(json.dumps({"kernels_only": out, "shape": shape, "n_nodes": int(s.n_nodes)}),
          flush=True)


def adjoint_only(lib, cfg, reps, graph=True):
    """The multivector adjoint solve alone (the reference's
    TestMultiVectorAdjointProblem path): FP64 eigensolve of the wells plus
    the seeded v_xc, then Jacobi-preconditioned MINRES on
    (H~ - eps_i) p_i = b_i for every column, to a residual of 1e-10 relative
    to |b|_D, timed over `reps` solves, FP64 and mixed operator (graph=False:
    the MINRES steps launched one by one instead of replayed as HIP graphs)."""
    from invdft_amd import abi, synthetic
    prob = synthetic.make_problem(lib, seed=1, target_tol=1e-10, **cfg)
    out = {}
    for name, prec in (("fp64", abi.FP64), ("mixed", abi.MIXED)):
        ctx = prob.context(lib, precision=prec, minres_graph=1 if graph else 0)
        ctx.set_potential(prob.vxc0)
        ev, _, _ = ctx.eigensolve(1e-10, 200)
        occ, fermi = ctx.occupancies()
        psi = ctx.eigenvectors()
        u = prob.rho_target_q - 0.5 * ctx.density()
        B = psi.shape[1]
        pairs = [v for i in range(B) for j in range(B) if abs(ev[i] - ev[j]) < 0.002
                 for v in (i, j)]
        mpsi = ctx.mv(B, psi)
        ctx.adj_update_input_psi(mpsi, occ, u, pairs, fermi, ev.copy())
        x, rhs, drhs = ctx.mv(B), ctx.mv(B), ctx.mv(B)
        ctx.adj_compute_rhs(None, x, rhs)
        ctx.adj_precondition_jacobi(drhs, rhs)
        bnorm = float(np.sqrt(np.max(np.sum(rhs.get() * drhs.get(), axis=0))))
        tol = 1e-10 * bnorm
        ctx.minres_solve(x, None, tol, 5000, distribute=True)  # warm-up
        t0 = time.perf_counter()
        for _ in range(reps):
            its = ctx.minres_solve(x, None, tol, 5000, distribute=True)
        dt = (time.perf_counter() - t0) / reps
        out[name] = {"s_per_solve": round(dt, 5), "iterations_max": int(np.max(its)),
                     "columns": B, "occupied": int(np.sum(occ > 1e-8)),
                     "ms_per_iteration": round(1e3 * dt / max(int(np.max(its)), 1), 4)}
        log(f"  {name}: {out[name]}")
        ctx.close()
    print(json.dumps({"metric": "s per multivector adjoint MINRES solve (rel. residual 1e-10)",
                      "value": out["fp64"]["s_per_solve"], "unit": "s/solve", "n_gpus": 1,
                      "higher_is_better": False, "dtype": "f64", "data": "synthetic",
                      "config": {"workload": "adjoint_" + str(cfg["n_cells"]) + "c_p"
                                 + str(cfg["degree"]), "n_cells": cfg["n_cells"],
                                 "degree": cfg["degree"]},
                      "detail": out}), flush=True)


def uneven_batch(lib, count, steps, workers):
    """Uneven batch of independent small inverse problems: problems/s and
    per-problem p50/p99 seconds for `steps` L-BFGS iterations each, mixed
    precision on `workers` concurrent contexts against sequential FP64
    solves on the same GPU."""
    from invdft_amd import abi, batch
    params = batch.draw_problems(count)
    t0 = time.perf_counter()
    probs = []
    for k in range(0, count, 8):
        probs += batch.build_problems(lib, params[k:k + 8])
        log(f"  set-up {len(probs)}/{count} problems ({time.perf_counter() - t0:.1f} s)")
    tol_kw = dict(cheb_tol=1e-8, initial_tol_cheb=1e-8)
    done = [0]

    def progress(k, r):
        done[0] += 1
        p = params[k]
        log(f"    problem {k} ({p['n_cells']}^3 cells, p={p['degree']}, {p['n_eig']} states): "
            f"{r[0]:.2f} s, loss {r[1]:.3e} -> {r[2]:.3e} [{done[0]}/{count}]")

    res_m, wall_m = batch.run_concurrent(lib, probs, abi.MIXED, steps, workers, tol_kw, progress)
    log(f"  mixed, {workers} concurrent contexts: {wall_m:.1f} s")
    done[0] = 0
    res_f, wall_f = batch.run_sequential(lib, probs, abi.FP64, steps, tol_kw, progress)
    log(f"  FP64 sequential: {wall_f:.1f} s")
    sm, sf = batch.summary(res_m, wall_m), batch.summary(res_f, wall_f)
    out = {"metric": f"problems/s, uneven batch of {count} inverse problems x {steps} BFGS steps",
           "value": sm["problems_per_s"], "unit": "problems/s", "n_gpus": 1,
           "higher_is_better": True, "dtype": "f32+f64", "data": "synthetic",
           "config": {"workload": "uneven_batch", "problems": count, "bfgs_steps": steps,
                      "cells": "U{8..20}^3", "degree": "U{3,4,5}", "orbitals": "U{1..16}",
                      "workers": workers},
           "mixed_concurrent": sm, "fp64_sequential": sf,
           "speedup": round(sf["wall_s"] / sm["wall_s"], 3)}
    print(json.dumps(out), flush=True)


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=2)
    ap.add_argument("--warmup", type=int, default=1)
    ap.add_argument("--config", default="inverse_24c_p5")
    ap.add_argument("--cheb-tol", type=float, default=1e-8)
    ap.add_argument("--no-fp64", action="store_true")
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--c3", type=int, default=1,
                    help="1: time one iteration of the batched 40^3 workload per precision "
                         "after the headline (detail.c3); 0: skip")
    ap.add_argument("--kernels-only", action="store_true",
                    help="only the operator kernels at --shape (for counter runs)")
    ap.add_argument("--adjoint-only", action="store_true",
                    help="only the multivector adjoint MINRES solve of --config")
    ap.add_argument("--no-graph", action="store_true",
                    help="launch MINRES steps one by one instead of replaying a HIP graph "
                         "(for rocprofv3 --kernel-trace, whose graph interception crashes)")
    ap.add_argument("--shape", type=int, nargs=4, default=[1, 16, 0, 0],
                    metavar=("CELLS_PER_WG", "VECTORS_PER_TILE", "GATHER_ROWS", "TILE_PASS"))
    ap.add_argument("--reps", type=int, default=5)
    ap.add_argument("--relax-ratio", type=float, default=None,
                    help="MIXED MINRES: residual / tolerance ratio below which the FP32 cell "
                         "operator takes over (library default if omitted)")
    ap.add_argument("--batch-count", type=int, default=96,
                    help="problems of --config uneven_batch")
    ap.add_argument("--batch-steps", type=int, default=10)
    ap.add_argument("--workers", type=int, default=4)
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py measures one GPU only (--gpus {args.gpus} requested); the multi-GPU "
              "decomposition is a design note, not a measured path", file=sys.stderr)
        sys.exit(2)

    import invdft_amd
    from invdft_amd import abi, synthetic

    lib = invdft_amd.load()
    if args.config == "gradcheck_32c_p5":
        c4_large(lib, args.steps)
        return
    if args.config == "uneven_batch":
        uneven_batch(lib, args.batch_count, args.batch_steps, args.workers)
        return
    cfg = dict(synthetic.CONFIGS[args.config])
    if args.kernels_only:
        kernels_only(lib, cfg, args.shape, args.reps)
        return
    if args.adjoint_only:
        adjoint_only(lib, cfg, args.reps, graph=not args.no_graph)
        return
    log(f"config {args.config}: {cfg}")
    t0 = time.perf_counter()
    prob = synthetic.make_problem(lib, seed=2, target_tol=1e-10, **cfg)
    log(f"setup (target density by FP64 eigensolve on the GPU): {time.perf_counter() - t0:.1f} s")
    tol_kw = dict(cheb_tol=args.cheb_tol, initial_tol_cheb=args.cheb_tol)
    if args.no_graph:
        tol_kw["minres_graph"] = 0
    if args.relax_ratio is not None:
        tol_kw["relax_ratio"] = args.relax_ratio

    log("mixed precision run")
    cm, mixed = run_bfgs(lib, prob, abi.MIXED, args.warmup, args.steps, tol_kw)
    fp64 = None
    cf = None
    if not args.no_fp64:
        log("FP64 run")
        cf, fp64 = run_bfgs(lib, prob, abi.FP64, args.warmup, args.steps, tol_kw)

    # force error of the mixed path against FP64 at the same potential, both
    # solved tightly (eigen residual 1e-10, adjoint 1e-13) so that the
    # difference measures precision, not solver truncation
    # The workload also states the eigenvalue and density errors; the same
    # comparison at the timed run's own tolerances is reported beside it.
    force_err = None
    errors = None
    if cf is not None:
        x = cm.get_solution()
        tight = dict(cheb_tol=1e-10, initial_tol_cheb=1e-10)
        errors = {"tight": mixed_vs_fp64_errors(lib, prob, x, tight),
                  "timed_tolerances": mixed_vs_fp64_errors(lib, prob, x, tol_kw)}
        force_err = errors["tight"]["force"]
        log(f"mixed vs FP64 at the final potential: {errors}")

    # roofline of the dominant kernel: the cell product (phase 1 of the
    # operator) of the mixed run at each precision.  For the kernel the
    # autotuner chose:
    #  - stored-H kernels (k_cell_gemm, k_cell_symm) are HBM-bound; their
    #    algorithmic bytes per launch are the symmetric H_e (ne(ne+1)/2 entries
    #    per cell) read once, the block X and node scale S read once and the
    #    per-cell products written once (the gather kernel reads them back);
    #  - the sum-factorised kernel (k_cell_plane) is bound by the vector ALUs; its
    #    algorithmic work per launch is the 1D contractions, sf_flops(p) per
    #    cell and column, and it moves w_e + X + S + the per-cell products.
    # The timed launches are plain applications (no node scale on the input).
    s = cm.sizes
    B = prob.desc.n_eig
    p = prob.desc.degree
    ne = s.nodes_per_cell
    nh = ne * (ne + 1) // 2
    nq = s.quad_per_cell

    def gemm_bytes(sz):
        return s.n_cells * nh * sz + s.n_nodes * (B + 1) * sz + s.n_cells * ne * B * sz

    def sf_bytes(sz):
        return s.n_cells * nq * sz + s.n_nodes * (B + 1) * sz + s.n_cells * ne * B * sz

    def roofline(shape, fp32, ms_cell, ms_op):
        sz, tn = (4, "float") if fp32 else (8, "double")
        kern = shape["kernel"]
        if kern == abi.KERNEL_SUM_FACTOR:
            kname = f"k_cell_plane<{tn},{tn},{p},false,true>"
            fl = s.n_cells * B * sf_flops_per_cell_column(p)
            peak = FP32_PEAK_TFLOPS if fp32 else FP64_PEAK_TFLOPS
            tf = fl / (ms_cell * 1e-3) / 1e12
            r = {"bound": "valu", "achieved": round(tf, 2), "peak": peak,
                 "unit": "TFLOP/s", "frac": round(tf / peak, 4),
                 "traffic": MEASURED_TRAFFIC.get((args.config, kname)), "kernel": kname,
                 "ms_per_launch": round(ms_cell, 4), "flops_per_launch": fl,
                 "bytes_per_launch": sf_bytes(sz),
                 "achieved_GBs": round(sf_bytes(sz) / (ms_cell * 1e-3) / 1e9, 1)}
        else:
            nct = min(5, max(1, min(shape["vectors_per_tile"], (B + 15) // 16 * 16) // 16))
            kname = f"k_cell_{('gemm', 'symm')[kern]}<{tn},{tn},{p},{nct}>"
            achieved = gemm_bytes(sz) / (ms_cell * 1e-3) / 1e9
            r = {"bound": "hbm", "achieved": round(achieved, 1), "peak": HBM_PEAK_GBS,
                 "unit": "GB/s", "frac": round(achieved / HBM_PEAK_GBS, 4),
                 "traffic": MEASURED_TRAFFIC.get((args.config, kname)), "kernel": kname,
                 "ms_per_launch": round(ms_cell, 4), "bytes_per_launch": gemm_bytes(sz)}
        r["operator_ms"] = round(ms_op, 4)
        return r

    # The dominant kernel of the mixed iteration is the FP32 cell product of
    # the Chebyshev filter (the largest share of kernel time in the iteration
    # trace in single precision); the FP64 one of Rayleigh-Ritz is reported
    # beside it.  The FP64 MINRES steps run another kernel (k_cell_line).
    ms_op32, ms_cell32 = cm.profile_apply(B, abi.MIXED, reps=20)
    roof = roofline(mixed["tuned"]["fp32"], True, ms_cell32, ms_op32)
    ms_op64, ms_cell64 = cm.profile_apply(B, abi.FP64, reps=20)
    extra = {"fp64_cell_product": roofline(mixed["tuned"]["fp64"], False, ms_cell64, ms_op64)}
    # attainable FMA rates of this GPU (16 independent chains per thread,
    # unpacked FP32): the rate a latency- or issue-limited kernel can
    # approach, beside the published peaks that `frac` uses
    fma = fma_probe(lib)
    extra["attainable_fma_tflops"] = fma
    for r, key in ((roof, "fp32"), (extra["fp64_cell_product"], "fp64")):
        if r.get("unit") == "TFLOP/s" and fma.get(key):
            r["attainable_fma"] = fma[key]
            r["frac_of_attainable"] = round(r["achieved"] / fma[key], 4)
    if cf is not None:
        m64, g64 = cf.profile_apply(B, abi.FP64, reps=20)
        extra["fp64_run_cell_product"] = {"ms_per_launch": round(g64, 4),
                                          "operator_ms": round(m64, 4),
                                          "shape": fp64["tuned"]["fp64"]}
    cpu = None
    if not args.no_cpu:
        log("CPU baseline sample (oracle)")
        cpu = cpu_baseline(lib, prob, mixed["per_eval"] if fp64 is None else fp64["per_eval"], 2,
                           tol_kw)
    c3 = None
    if args.c3:
        log("batched workload (C3), one iteration per precision")
        c3 = c3_leg(lib, args.cheb_tol)

    out = {
        "metric": METRIC,
        "value": round(mixed["s_per_iter"], 4),
        "unit": "s/iter",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(mixed["timed_ms"] / mixed["iters"], 2),
        "higher_is_better": False,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32+f64",
        "data": "synthetic",
        "config": {"workload": args.config, "n_cells": cfg["n_cells"], "degree": cfg["degree"],
                   "nodes": int(s.n_nodes), "orbitals": B, "cheb_degree": prob.desc.cheb_degree,
                   "cheb_tol": args.cheb_tol, "evals_per_iter": 2, "parallelism": "single-gpu"},
        "fp64_s_per_iter": round(fp64["s_per_iter"], 4) if fp64 else None,
        "speedup_mixed_vs_fp64": round(fp64["s_per_iter"] / mixed["s_per_iter"], 3) if fp64 else None,
        "force_rel_err_mixed_vs_fp64": force_err,
        "errors_mixed_vs_fp64": errors,
        "roofline": roof,
        "cpu_baseline": cpu,
        "detail": {"mixed_per_eval": mixed["per_eval"], "fp64_per_eval": fp64["per_eval"] if fp64 else None,
                   "tile_shapes": {"mixed": mixed["tuned"], "fp64": fp64["tuned"] if fp64 else None},
                   "mixed_loss": mixed["loss"], "c3": c3, **extra},
    }
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
