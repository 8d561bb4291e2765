"""Benchmark: DOF/s solved to a 1e-8 FP64 relative residual on one MI355X.

Workload (default): the 2000 x 500 Q1 plane-stress cantilever beam, nodes
jittered by +-20% of the cell size (seed 0), 2,005,002 DOFs, E = 211 GPa,
nu = 0.3, left edge clamped, traction -1e6 N/m on the top edge, 2x2 Gauss.

One step = the first solve, from u = 0, of a freshly assembled device-resident
system until ||b - K u||_2 / ||b||_2 <= 1e-8 (true residual recomputed in
FP64): every per-system cost of the solver is inside it (FP32 matrix copy,
multigrid topology and numeric set-up, solver buffers; a first solve launches
its kernels directly, later solves of the system replay captured chunks), as
in each bfm_sim_run. value = DOFs / mean step time of the headline solver,
flexible CG in FP64 preconditioned by one FP32 smoothed-aggregation V-cycle.
A re-solve on the same system (its matrix unchanged, so the hierarchy and its
numeric set-up are reused: a new load case) is reported beside it, and
plain FP64 Jacobi-PCG is timed on the system (the speedups are reported).

Also reported: the batched workload (4096 seeded holed panels of 1k-60k DOFs,
assembled and solved by block-Jacobi PCG, each by a cluster of workgroups that
holds its matrix in registers: DOF/s, and the same batch in the multigrid
mode); the roofline of the headline solver's largest kernel (the
flexible-CG FP64 SpMV), of its finest-level post-smoothing step (FP32 SpMV +
block-Jacobi Chebyshev step) and of the FP64 CG SpMV (algorithmic bytes /
mean launch time from HIP events on the solver's stream), the end-to-end time (upload + renumbering + assembly + conditions +
solve), and CPU baselines: the reference libbfm compiled from its own C
sources (oracle/_ref), single-threaded as libbfm is, on a bounded sample (its
dense path cannot hold the 2M-DOF matrix: 32 TB); the oracle's OpenMP CSR
Jacobi-PCG on the full system (a bounded number of iterations, scaled); and
libbfm's RCM + band LU with the matrix kept sparse, on the full system
(interior pivot steps timed and scaled).

Usage: python bench.py [--gpus 1] [--steps K] [--warmup W] [--workload q1_2m]
"""

import argparse
import json
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

HBM_PEAK_GBS = 8000.0
# HBM bytes per launch on the q1_2m beam measured by two rocprofv3 counter runs
# (FETCH_SIZE x 1.9998 + WRITE_SIZE, the factors read off a 256 MiB
# device-to-device copy in the same runs): profiles/hbm_traffic_q1_2m.md
TRAFFIC_Q1_2M = {"k_cg_spmv": 389.3e6, "k_fcg_spmv": 397.4e6, "k_cheb": 254.9e6}
CPU_SAMPLE = (180, 45)   # Q1 beam cells for the reference CPU path (16,652 DOFs)


def log(msg):
    print(msg, file=sys.stderr, flush=True)


def cpu_baseline_reference():
    """libbfm (reference C) on a bounded beam sample, through its own C API."""
    sys.path.insert(0, os.path.join(ROOT, "oracle"))
    from bfm_amd import meshgen
    from bfm_amd import pybfm as pb
    ref = os.path.join(ROOT, "oracle", "_ref", "libbfm_ref.so")
    nx, ny = CPU_SAMPLE
    mesh = meshgen.beam(nx, ny, kind=4, jitter=0.2, seed=0)
    mat = meshgen.BEAM_MATERIAL
    if os.path.exists(ref):
        L = pb.Library(ref)
        cm = pb.Mesh_arrays.from_generated(mesh, lib=L)
        m = pb.Material("steel", mat["rho"], mat["E"], mat["nu"], lib=L)
        rule = pb.Rule_gauss_legendre(2, 4, lib=L)
        obj = pb.Obj(cm, m, rule, lib=L)
        inst = pb.Instance(obj, lib=L)
        conds = []
        kinds, values, flags = meshgen.beam_conditions(mesh)
        for k, v, f in zip(kinds, values, flags):
            c = pb.Condition(cm, int(k), float(v), lib=L)
            c.set_nodes(f)
            inst.add_condition(c)
            conds.append(c)
        sim = pb.Sim(pb.Sim.PLANAR_STRESS, lib=L)
        sim.add_instance(inst)
        t0 = time.perf_counter()
        sim.run()
        dt = time.perf_counter() - t0
        kind = "reference"
        what = "libbfm compiled from the reference C sources"
    else:
        import oracle as O
        kinds, values, flags = meshgen.beam_conditions(mesh)
        t0 = time.perf_counter()
        O.solve_dense(mesh, True, mat["E"], mat["nu"], mat["rho"], kinds, values, flags)
        dt = time.perf_counter() - t0
        kind = "port"
        what = "the oracle's C restatement of libbfm's path"
    return {
        "value": mesh.n_dof / dt,
        "unit": "DOF/s",
        "cores": 1,
        "kind": kind,
        "sample": (f"{what}, single-threaded: dense assembly, ordered conditions, RCM, band LU on the "
                   f"{nx}x{ny} jittered Q1 beam ({mesh.n_dof} DOFs) in {dt:.2f} s; the 2,005,002-DOF "
                   f"workload is infeasible for libbfm's dense path (32 TB matrix, int index overflow)"),
    }


def cpu_pcg_sample(mesh, stress, iterations_needed, iters=300):
    """The sparse FP64 Jacobi-PCG of the oracle (CSR, OpenMP) on the full
    workload's own system, timed for a bounded number of iterations on all
    host threads (at most 16) and on one, then scaled to the iterations the
    same algorithm needs to reach the tolerance on the GPU."""
    sys.path.insert(0, os.path.join(ROOT, "oracle"))
    import oracle as O
    from bfm_amd import meshgen
    mat = meshgen.BEAM_MATERIAL
    kinds, values, flags = meshgen.beam_conditions(mesh)
    A, b = O.assemble_csr(mesh, stress, mat["E"], mat["nu"], mat["rho"], kinds=kinds, values=values, flags=flags)
    out = {}
    for threads, n_it in ((min(16, os.cpu_count() or 1), iters), (1, max(20, iters // 6))):
        t0 = time.perf_counter()
        _, it, _ = O.pcg_csr(A, b, rtol=1e-300, max_iter=n_it, threads=threads)
        dt = time.perf_counter() - t0
        per = dt / max(1, it)
        out[threads] = {"value": mesh.n_dof / (per * iterations_needed), "s_per_iteration": per, "timed_iterations": it}
    all_t = max(out)
    return {
        "value": out[all_t]["value"], "unit": "DOF/s", "cores": all_t, "kind": "port",
        "sample": (f"the oracle's sparse FP64 CSR Jacobi-PCG (OpenMP) on the full {mesh.n_dof}-DOF system: "
                   f"{out[all_t]['timed_iterations']} iterations timed on {all_t} threads "
                   f"({out[all_t]['s_per_iteration'] * 1e3:.1f} ms each) and {out[1]['timed_iterations']} on one "
                   f"({out[1]['s_per_iteration'] * 1e3:.1f} ms each), scaled to the {iterations_needed} iterations "
                   f"Jacobi PCG needs for rtol 1e-8"),
        "single_core_value": out[1]["value"],
    }


def cpu_band_lu_sample(mesh, stress, target_s=8.0):
    """libbfm's direct path (sim.c:103-135: RCM of perm.c:117-331, band LU
    and substitution of matrix.c:253-404, restated in the oracle) on the full
    workload's own system, single-threaded as libbfm runs, with the matrix
    kept sparse until it is laid out as a band (the dense m x m matrix, 32 TB
    at 2M DOFs, cannot be held). The assembly with the conditions, RCM and
    half-bandwidth run in full; the band LU is timed over a window of its
    interior pivot steps (each costs the same, (k + 1) k multiply-adds,
    whatever the values) and the band fill and substitutions over that
    window's rows, each scaled to the m rows. The window is a principal
    submatrix of the permuted SPD matrix, so its LU has no breakdown."""
    sys.path.insert(0, os.path.join(ROOT, "oracle"))
    import oracle as O
    import numpy as np
    from bfm_amd import meshgen
    mat = meshgen.BEAM_MATERIAL
    kinds, values, flags = meshgen.beam_conditions(mesh)
    t0 = time.perf_counter()
    A, b = O.assemble_csr(mesh, stress, mat["E"], mat["nu"], mat["rho"], kinds=kinds, values=values, flags=flags)
    t_asm = time.perf_counter() - t0
    t0 = time.perf_counter()
    perm, inv = O.rcm_csr(A)
    k = O.bandwidth_csr(A, perm)
    t_rcm = time.perf_counter() - t0
    m = A.m

    def window(steps):
        nrows = min(m, steps + k + 1)
        r0 = (m - nrows) // 2
        t0 = time.perf_counter()
        band = O.band_window(A, perm, inv, k, r0, nrows)
        t_fill = time.perf_counter() - t0
        t0 = time.perf_counter()
        assert O.band_lu_steps(band, nrows, k, steps) == 0
        t_lu = time.perf_counter() - t0
        y = np.ones(nrows)
        t0 = time.perf_counter()
        assert O.band_lu_solve(band, nrows, k, y) == 0
        t_solve = time.perf_counter() - t0
        return t_fill / nrows, t_lu / steps, t_solve / nrows

    per_step = window(32)[1]
    steps = int(max(64, min(8000, target_s / per_step)))
    per_fill, per_step, per_solve = window(steps)
    total = t_asm + t_rcm + m * (per_fill + per_step + per_solve)
    return {
        "value": mesh.n_dof / total, "unit": "DOF/s", "cores": 1, "kind": "port",
        "sample": (f"libbfm's RCM + band LU + substitution (the oracle's restatement) with sparse assembly on the "
                   f"full {m}-DOF system, half-bandwidth {k}: assembly {t_asm:.1f} s and RCM {t_rcm:.1f} s in full, "
                   f"{steps} interior band-LU pivot steps timed ({per_step * 1e3:.2f} ms each) and the band fill "
                   f"and substitutions over their {min(m, steps + k + 1)} rows, scaled to {m} rows: "
                   f"{total:.0f} s in all"),
        "estimated_s": total,
    }


def copy_calibration(nbytes):
    """One hipMemcpy of nbytes between two device buffers (the runtime's copy
    kernel reads and writes nbytes): the reference that scales the
    FETCH_SIZE / WRITE_SIZE counters to bytes."""
    import ctypes as C
    hip = C.CDLL("libamdhip64.so")
    a, b = C.c_void_p(), C.c_void_p()
    assert hip.hipMalloc(C.byref(a), C.c_size_t(nbytes)) == 0 and hip.hipMalloc(C.byref(b), C.c_size_t(nbytes)) == 0
    assert hip.hipMemset(a, 1, C.c_size_t(nbytes)) == 0
    assert hip.hipMemcpy(b, a, C.c_size_t(nbytes), 3) == 0          # hipMemcpyDeviceToDevice
    assert hip.hipDeviceSynchronize() == 0
    hip.hipFree(a)
    hip.hipFree(b)
    log(f"copy calibration: {nbytes} bytes device to device")


def batched_leg(D, meshgen, count, rtol):
    """The batched workload: `count` seeded holed panels (1k-60k DOFs, plane
    strain, traction U(1e5, 1e7) N/m on top, bottom corners pinned), built
    into one batch from their meshes; one timed call assembles every panel
    (above 1,024 panels one workgroup each, else a launch per colour over all
    of them) and solves it by block-Jacobi PCG to rtol (a cluster of workgroups each; the autotuner's configurations are
    for panels that do not fit one)."""
    t = time.perf_counter()
    inst, sizes, dofs = [], [], 0
    for k in range(count):
        m, tr = meshgen.panel(k)
        inst.append(D.panel_instance(m, tr))
        sizes.append(m.n_nodes)
        dofs += m.n_dof
    t_mesh = time.perf_counter() - t
    t = time.perf_counter()
    b = D.Batch.from_instances(inst)
    del inst
    t_create = time.perf_counter() - t
    log(f"batched: {count} panels, {dofs} DOFs; meshes {t_mesh:.1f} s, batch set-up {t_create:.1f} s")
    pre = D.PRECOND_BLOCK_JACOBI
    t = time.perf_counter()
    picks, times = b.autotune(precond=pre)
    t_tune = time.perf_counter() - t
    log(f"batched: autotune {t_tune:.1f} s, picks {picks.tolist()}")
    b.solve(precond=pre, rtol=rtol, picks=picks)         # clusters planned, first launch
    t = time.perf_counter()
    st, ms = b.solve(precond=pre, rtol=rtol, picks=picks)
    wall = time.perf_counter() - t
    assert all(x["status"] == 0 and x["rel_residual"] <= rtol for x in st)
    its = np.array([x["iterations"] for x in st])
    nnzb = np.array([b.system(k).info()["nnzb"] for k in range(count)])
    # the clusters read each panel's matrix and load once and keep them; what
    # a streaming solve of the same iterations would move is given beside it
    byt = sum(D.batch_bytes(int(nnzb[k]), sizes[k], 1, 0, pre) for k in range(count))
    streamed = sum(D.batch_bytes(int(nnzb[k]), sizes[k], int(st[k]["iterations"]), int(st[k]["restarts"]), pre)
                   for k in range(count))
    gbs = byt / (ms / 1e3) / 1e9
    log(f"batched: {ms:.1f} ms device ({wall * 1e3:.1f} ms wall), {dofs / (ms / 1e3):.3e} DOF/s, "
        f"iterations mean {its.mean():.0f} max {its.max()}, {streamed / (ms / 1e3) / 1e9:.0f} GB/s if it were streamed")
    # multigrid mode: the same batch solved as one block-diagonal system by
    # flexible CG + the multigrid V-cycle (each load scaled to unit norm, the
    # tolerance checks testing every panel's own residual); the first launch
    # builds the union (its graph concatenated on host threads, its values
    # and coordinates gathered on the device) and its
    # hierarchy (finest and level-1 aggregates by host sweeps over whole
    # panels, the patterns on the GPU)
    t = time.perf_counter()
    b.solve(precond=D.PRECOND_AMG, rtol=rtol)
    t_mg_setup = time.perf_counter() - t
    t = time.perf_counter()
    st_mg, ms_mg = b.solve(precond=D.PRECOND_AMG, rtol=rtol)
    wall_mg = time.perf_counter() - t
    assert all(x["status"] == 0 and x["rel_residual"] <= rtol for x in st_mg)
    worst = max(x["rel_residual"] for x in st_mg)
    log(f"batched multigrid: {ms_mg:.1f} ms device ({wall_mg * 1e3:.1f} ms wall), {dofs / (ms_mg / 1e3):.3e} DOF/s, "
        f"{st_mg[0]['iterations']} iterations, worst instance residual {worst:.2e}, {ms / ms_mg:.2f}x the "
        f"block-Jacobi solve; first launch (union and hierarchy build) {t_mg_setup:.1f} s")
    return {
        "workload": f"{count} holed panels (seeds 0-{count - 1}), 1k-60k DOFs, plane strain, block-Jacobi PCG "
                    f"to rtol {rtol:g}, assembled and solved from one call",
        "n_dof": int(dofs), "ms_per_step": ms, "wall_ms": wall * 1e3, "value": dofs / (ms / 1e3),
        "unit": "DOF/s", "iterations_mean": float(its.mean()), "iterations_max": int(its.max()),
        "picks": picks.tolist(), "autotune_ms": times.tolist(), "setup_s": {"meshes": t_mesh,
                                                                              "batch_create": t_create,
                                                                              "autotune": t_tune},
        "roofline": {"bound": "latency of the clusters' exchanges and issue (the matrix stays in registers)",
                     "achieved": gbs, "peak": HBM_PEAK_GBS, "unit": "GB/s", "frac": gbs / HBM_PEAK_GBS,
                     "traffic": None, "kernel": "k_resident_batch (block Jacobi) + "
                                               f"{'k_batch_colors' if count > 1024 else 'k_batch_elements'} (whole call)",
                     "algorithmic_bytes": byt, "streamed_bytes_of_its_iterations": streamed},
        "multigrid": {
            "solver": "the batch as one block-diagonal system: flexible CG (FP64) + FP32 smoothed-aggregation "
                      "V-cycle, one dense coarsest inverse per panel, loads scaled to unit norm, every panel's "
                      f"own true residual checked against rtol {rtol:g}",
            "ms_per_step": ms_mg, "wall_ms": wall_mg * 1e3, "value": dofs / (ms_mg / 1e3), "unit": "DOF/s",
            "iterations": int(st_mg[0]["iterations"]), "worst_rel_residual": worst,
            "speedup_vs_persistent_launch": ms / ms_mg, "first_launch_s": t_mg_setup},
    }


def timed_solves(D, s, name, precond, rtol, warmup, steps, accept_floor=False):
    """warmup untimed then steps timed solves of s: (mean ms, last stats,
    reached rtol). accept_floor: a stop at the rounding floor (the solver's
    stagnation status) is timed and reported instead of raised."""
    times, st = [], None
    for k in range(warmup + steps):
        t = time.perf_counter()
        try:
            _, st = s.solve(precond=precond, rtol=rtol, want_u=False)
        except D.BfmxError as e:
            if not (accept_floor and e.code == -8):
                raise
            st = {"iterations": -1, "rel_residual": float(str(e).split("residual ")[1].split()[0]),
                  "fallback": 0, "status": e.code}
        dt = (time.perf_counter() - t) * 1e3
        if k >= warmup:
            times.append(dt)
        log(f"{name} {'warmup' if k < warmup else 'step'}: {dt:.1f} ms, {st['iterations']} iterations, "
            f"rel residual {st['rel_residual']:.3e}")
    return float(np.mean(times)), st, st["status"] == 0


def heterogeneous_leg(D, meshgen, args):
    """The mixed-precision workload: the 2M-DOF beam with E per element
    log-uniform over [1e9, 1e11] (seed 0), solved to 1e-8 by flexible CG in
    FP64 with the FP32 multigrid V-cycle (every SpMV of the V-cycle FP32;
    the true residual FP64, evaluated compensated): the first solve of a
    fresh system, a re-solve, the error against the same solver run down to
    its rounding floor, and Jacobi PCG beside it."""
    mesh, stress = meshgen.workload("q1_2m_het")
    t = time.perf_counter()
    s = D.beam_system(mesh, stress=stress)
    t_setup = time.perf_counter() - t
    first_ms, st_first, _ = timed_solves(D, s, "het fcg_amg first solve", D.PRECOND_AMG, args.rtol, 0, 1)
    ms, st, _ = timed_solves(D, s, "het fcg_amg", D.PRECOND_AMG, args.rtol, 1, max(1, args.steps))
    u, _ = s.solve(precond=D.PRECOND_AMG, rtol=args.rtol)
    try:
        u_t, st_t = s.solve(precond=D.PRECOND_AMG, rtol=1e-12)
        floor = st_t["rel_residual"]
    except D.BfmxError as e:
        u_t = s.get_u()
        floor = float(str(e).split("residual ")[1].split()[0])
    err = float(np.linalg.norm(u - u_t) / np.linalg.norm(u_t))
    out = {
        "workload": "q1_2m_het: 2000x500 Q1 beam, 20% jitter, E log-uniform [1e9, 1e11] per element (seed 0), "
                    f"{mesh.n_dof} DOFs, rtol {args.rtol:g}",
        "solver": "flexible CG (FP64, compensated true residual) + FP32 smoothed-aggregation V-cycle (FP32 SpMVs)",
        "setup_s": t_setup, "first_solve_ms": first_ms, "value": mesh.n_dof / (first_ms / 1e3),
        "resolve_ms": ms, "iterations": int(st["iterations"]), "rel_residual": st["rel_residual"],
        "floor_rel_residual": floor, "error_vs_floor_solution": err,
    }
    if not args.no_pcg:
        p_ms, p_st, reached = timed_solves(D, s, "het pcg_jacobi", D.PRECOND_JACOBI, args.rtol, 0, 1,
                                           accept_floor=True)
        out["pcg_jacobi_fp64"] = {"ms": p_ms, "rel_residual": p_st["rel_residual"], "reached_rtol": reached,
                                  "iterations": int(p_st["iterations"])}
        out["speedup_vs_pcg"] = p_ms / first_ms
    log(f"heterogeneous beam: first solve {first_ms:.1f} ms, re-solve {ms:.1f} ms, {st['iterations']} iterations, "
        f"residual {st['rel_residual']:.2e}, floor {floor:.2e}, error {err:.2e}")
    return out, s


def learned_leg(D, meshgen, args, seed=7):
    """The learned preconditioner on its evaluation workload: a held-out
    seed of the 2M-DOF heterogeneous beam (training used beams of seeds 100
    and up and panels of seeds 100000 and up): flexible CG preconditioned by
    the FP32 multigrid V-cycle plus the trained network's correction, after a
    warm-up, beside the method without the network (the multigrid FCG),
    block-Jacobi and Jacobi PCG."""
    from bfm_amd.learned import WEIGHTS_MULTIGRID
    mesh, stress = meshgen.workload("q1_2m_het", seed=seed)
    s = D.beam_system(mesh, stress=stress)
    s.set_model(D.Model.load(WEIGHTS_MULTIGRID))
    w = max(1, args.warmup)
    l_ms, l_st, _ = timed_solves(D, s, "learned_fcg", D.PRECOND_AMG_LEARNED, args.rtol, w, 1)
    a_ms, a_st, _ = timed_solves(D, s, "learned leg: fcg_amg", D.PRECOND_AMG, args.rtol, w, 1)
    out = {
        "workload": f"q1_2m_het seed {seed} (held out), {mesh.n_dof} DOFs, rtol {args.rtol:g}",
        "solver": "flexible CG (FP64) + FP32 multigrid V-cycle + the trained network's correction (BF16 weights, "
                  "FP32 activations), block-Jacobi PCG fallback",
        "ms_per_step": l_ms, "value": mesh.n_dof / (l_ms / 1e3), "iterations": int(l_st["iterations"]),
        "rel_residual": l_st["rel_residual"], "fallback": int(l_st["fallback"]),
        "multigrid_fcg_without_network": {"ms": a_ms, "iterations": int(a_st["iterations"])},
    }
    if not args.no_pcg:
        b_ms, b_st, b_ok = timed_solves(D, s, "learned leg: pcg_block_jacobi", D.PRECOND_BLOCK_JACOBI, args.rtol, 0,
                                        1, accept_floor=True)
        p_ms, p_st, p_ok = timed_solves(D, s, "learned leg: pcg_jacobi", D.PRECOND_JACOBI, args.rtol, 0, 1,
                                        accept_floor=True)
        out["block_jacobi_pcg"] = {"ms": b_ms, "rel_residual": b_st["rel_residual"], "reached_rtol": b_ok}
        out["jacobi_pcg"] = {"ms": p_ms, "rel_residual": p_st["rel_residual"], "reached_rtol": p_ok}
        # the PCG runs stop at their floor above rtol: their time to that stop
        out["speedup_vs_pcg"] = p_ms / l_ms
    log(f"learned FCG: {l_ms:.1f} ms, {l_st['iterations']} iterations, fallback {l_st['fallback']}; multigrid "
        f"FCG alone {a_ms:.1f} ms, {a_st['iterations']} iterations")
    return out


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=3)
    ap.add_argument("--warmup", type=int, default=1)
    ap.add_argument("--workload", default="q1_2m")
    ap.add_argument("--rtol", type=float, default=1e-8)
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline leg")
    ap.add_argument("--no-pcg", action="store_true", help="skip the plain Jacobi-PCG leg")
    ap.add_argument("--no-learned", action="store_true", help="skip the learned-preconditioner leg")
    ap.add_argument("--no-het", action="store_true", help="skip the heterogeneous-E (mixed-precision) leg")
    ap.add_argument("--no-batch", action="store_true", help="skip the batched holed-panel leg")
    ap.add_argument("--batch-count", type=int, default=4096, help="panels in the batched leg")
    ap.add_argument("--batch-only", action="store_true",
                    help="run only the batched leg and print its record (for profiling; not the bench line)")
    ap.add_argument("--copy-calibration", type=int, default=0, metavar="BYTES",
                    help="first run one device-to-device copy of BYTES (the HBM counters' reference)")
    ap.add_argument("--mixed-cg", action="store_true",
                    help="also run CG on the FP32 matrix with FP64 reliable updates")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py runs on one GPU only (asked for --gpus {args.gpus}): the solver has no "
              "multi-GPU sharding; value is one GPU's throughput", file=sys.stderr)
        sys.exit(2)

    from bfm_amd import device as D
    from bfm_amd import meshgen

    if args.copy_calibration:
        copy_calibration(args.copy_calibration)
    if args.batch_only:
        print(json.dumps(batched_leg(D, meshgen, args.batch_count, args.rtol)), flush=True)
        return
    mesh, stress = meshgen.workload(args.workload)
    log(f"workload {args.workload}: {mesh.n_nodes} nodes, {mesh.n_dof} DOFs, {mesh.n_elems} elements")

    def fresh():
        t = time.perf_counter()
        sys_ = D.beam_system(mesh, stress=stress)
        return sys_, time.perf_counter() - t

    # headline: the first solve of a freshly assembled system, so every
    # per-system cost of the solver is inside the step (the FP32 matrix copy,
    # the multigrid hierarchy's topology and numeric set-up, the solver's
    # buffers), as each bfm_sim_run pays it; the
    # system itself (upload, renumbering, pattern, assembly, conditions) is
    # built before the step's clock starts
    first_ms, first_st, setups = [], None, []
    s = None
    for k in range(args.warmup + args.steps):
        if s is not None:
            s.close()
        s, t_setup = fresh()
        setups.append(t_setup)
        t = time.perf_counter()
        _, st0 = s.solve(precond=D.PRECOND_AMG, rtol=args.rtol, want_u=False)
        dt = time.perf_counter() - t
        assert st0["status"] == 0 and st0["rel_residual"] <= args.rtol, st0
        tag = "warmup" if k < args.warmup else f"step {k - args.warmup}"
        log(f"fcg_amg first solve of a fresh system, {tag}: {dt * 1e3:.1f} ms, {st0['iterations']} iterations, "
            f"rel residual {st0['rel_residual']:.3e} (system set-up {t_setup:.2f} s)")
        if k >= args.warmup:
            first_ms.append(dt * 1e3)
            first_st = st0
    info = s.info()
    t_setup = float(np.mean(setups))
    log(f"setup {t_setup:.2f} s: {info}")

    def leg(name, precond, precision=D.FP64, steps=args.steps):
        for _ in range(args.warmup):
            t = time.perf_counter()
            _, st = s.solve(precond=precond, precision=precision, rtol=args.rtol, want_u=False)
            log(f"{name} warmup {(time.perf_counter() - t) * 1e3:.1f} ms, {st['iterations']} iterations")
        times, stats = [], []
        for k in range(steps):
            t = time.perf_counter()
            _, st = s.solve(precond=precond, precision=precision, rtol=args.rtol, want_u=False)
            dt = time.perf_counter() - t
            assert st["status"] == 0 and st["rel_residual"] <= args.rtol, st
            times.append(dt)
            stats.append(st)
            log(f"{name} step {k}: {dt * 1e3:.1f} ms, {st['iterations']} iterations, "
                f"rel residual {st['rel_residual']:.3e}")
        ms = 1e3 * float(np.mean(times))
        return ms, stats[-1]

    ms_first = float(np.mean(first_ms))
    value = mesh.n_dof / (ms_first / 1e3)
    # the same solver re-solving on a system whose hierarchy exists (the
    # matrix unchanged: the hierarchy's numeric set-up is reused as well)
    ms, st = leg("fcg_amg (cached hierarchy)", D.PRECOND_AMG)

    def roof(kernel, label):
        k_ms, k_bytes = s.time_kernel(kernel, reps=100)
        gbs = k_bytes / (k_ms / 1e3) / 1e9
        log(f"{label}: {k_ms * 1e3:.1f} us, {k_bytes / 1e6:.1f} MB, {gbs:.0f} GB/s")
        traffic = TRAFFIC_Q1_2M.get(label.split("<")[0].split(" ")[0]) if args.workload == "q1_2m" else None
        return {"bound": "hbm", "achieved": gbs, "peak": HBM_PEAK_GBS, "unit": "GB/s",
                "frac": gbs / HBM_PEAK_GBS, "traffic": traffic, "kernel": label,
                "kernel_us": k_ms * 1e3, "algorithmic_bytes": k_bytes}

    roof_fcg = roof(D.KERNEL_FCG_SPMV, "k_fcg_spmv (flexible-CG FP64 SpMV, the solve's largest kernel)")
    roof_smooth = roof(D.KERNEL_AMG_SMOOTH, "k_cheb<2,double,false,true> (finest-level post-smoothing step)")
    roof_spmv = roof(D.KERNEL_CG_SPMV64, "k_cg_spmv<double> (FP64 CG SpMV)")

    extra = {}
    if not args.no_pcg:
        p_ms, p_st = leg("pcg_jacobi", D.PRECOND_JACOBI, steps=max(1, min(args.steps, 2)))
        extra["pcg_jacobi_fp64"] = {
            "ms_per_step": p_ms, "value": mesh.n_dof / (p_ms / 1e3), "iterations": int(p_st["iterations"]),
            "rel_residual": p_st["rel_residual"],
        }
        extra["speedup_vs_pcg"] = p_ms / ms_first
        extra["speedup_vs_pcg_cached_hierarchy"] = p_ms / ms
        log(f"speedup of multigrid FCG over Jacobi-PCG: {p_ms / ms_first:.2f}x first solve, "
            f"{p_ms / ms:.2f}x re-solve")
    if not args.no_het:
        extra["mixed_het"], het_sys = heterogeneous_leg(D, meshgen, args)
    else:
        het_sys = None
    if not args.no_learned:
        extra["learned_fcg"] = learned_leg(D, meshgen, args)
    del het_sys
    if args.mixed_cg:
        try:
            m_ms, m_st = leg("cg_fp32_matrix", D.PRECOND_JACOBI, D.MIXED, steps=1)
            extra["cg_fp32_matrix"] = {"ms_per_step": m_ms, "iterations": int(m_st["iterations"])}
        except (D.BfmxError, AssertionError) as e:
            extra["cg_fp32_matrix"] = {"status": str(e)}
            log(f"cg_fp32_matrix: {e}")

    if not args.no_batch:
        extra["batched_panels"] = batched_leg(D, meshgen, args.batch_count, args.rtol)

    cpu = None
    if not args.no_cpu:
        log("cpu baseline ...")
        cpu = cpu_baseline_reference()
        log(f"cpu baseline {cpu['value']:.0f} DOF/s")
        if "pcg_jacobi_fp64" in extra:
            extra["cpu_baseline_sparse_pcg"] = cpu_pcg_sample(mesh, stress, extra["pcg_jacobi_fp64"]["iterations"])
            log(f"cpu sparse PCG sample: {extra['cpu_baseline_sparse_pcg']['value']:.3e} DOF/s "
                f"({extra['cpu_baseline_sparse_pcg']['cores']} threads)")
            extra["cpu_baseline_sparse_band_lu"] = cpu_band_lu_sample(mesh, stress)
            log(f"cpu sparse band LU sample: {extra['cpu_baseline_sparse_band_lu']['value']:.3e} DOF/s "
                f"({extra['cpu_baseline_sparse_band_lu']['estimated_s']:.0f} s estimated)")

    out = {
        "metric": "DOF/s solved to 1e-8 FP64 rel. residual; learned-FCG vs plain PCG speedup",
        "value": value,
        "unit": "DOF/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": ms_first,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64+f32",
        "data": "synthetic",
        "config": {
            "workload": f"{args.workload}: 2000x500 Q1 plane-stress cantilever beam, 20% jitter (seed 0), "
                        f"{mesh.n_dof} DOFs, solved to rtol {args.rtol:g} from u = 0",
            "solver": "flexible CG (FP64) + FP32 smoothed-aggregation multigrid V-cycle",
            "n_dof": mesh.n_dof,
            "n_elems": mesh.n_elems,
            "iterations": int(first_st["iterations"]),
            "rel_residual": first_st["rel_residual"],
            "step": "first solve of a freshly assembled system: FP32 matrix copy, multigrid topology and "
                    "numeric set-up, solver buffers, and the iterations to the tolerance",
            "setup_s": t_setup,
            "end_to_end_s": t_setup + ms_first / 1e3,
            "resolve_cached_hierarchy": {"ms_per_step": ms, "value": mesh.n_dof / (ms / 1e3),
                                         "iterations": int(st["iterations"]), "rel_residual": st["rel_residual"]},
        },
        "roofline": roof_fcg,
        "roofline_smoother": roof_smooth,
        "roofline_spmv_fp64": roof_spmv,
        "cpu_baseline": cpu,
    }
    out.update(extra)
    print(json.dumps(out))


if __name__ == "__main__":
    main()
