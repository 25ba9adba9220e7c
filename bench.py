"""Benchmark: FP64 sparse-grid kronmult apply on one MI355X.

Headline workload (one step = one apply y = A x over the whole grid, inputs
resident in HBM): d = 6, n = 2 (degree 1), |l|_1 <= 7 sparse grid (16,172
cells, 1,035,008 unknowns), 226,043,944 connected cell pairs, the 6 terms of
a 3x+3v Vlasov advection operator (DG div/mass 1D operators, 256 x 256 per
dimension), x ~ U[-1, 1], seed 0: 2,083 GFLOP pair by pair, 0.2 GFLOP one
dimension at a time.

Reported: GFLOP/s of the products the chosen kernel forms, in the x2 convention
of kronmult_matrix::compute_flops (pair by pair 2*d*n^(d+1)*T per connected
pair and term; one dimension at a time as the reference counts its global
operator), the roofline of that kernel (FP64 peak 78.6 TFLOP/s, vector and
matrix cores alike; the sum-factorised matrix-core kernel executes fewer flops
than the convention counts, and its executed matrix-core rate is reported
beside it from the committed counter profile; the dimension-by-dimension form
counts bytes), the FP64 parity of the GPU result against the CPU oracle on the
sampled rows, and the oracle's OpenMP kronmult (a restatement of the
reference's cpu_sparse) timed on this host's cores over a bounded row sample of
the same apply.  The d = 3, n = 3 |l|_1 <= 6 apply, FP32 applies, the global
operator and the implicit-step solves are reported as extras.

Usage: python bench.py [--gpus 1] [--steps K] [--warmup W]
"""
import argparse
import json
import os
import sys
import time

# thread placement of the CPU baseline's OpenMP runtime; set before any
# OpenMP library loads
os.environ.setdefault("OMP_PROC_BIND", "close")
os.environ.setdefault("OMP_PLACES", "cores")
# the CPUs this job may run on, read before an OpenMP runtime binds the
# initial thread to its first place (after which the mask holds one CPU)
JOB_CPUS = len(os.sched_getaffinity(0))

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

FP64_PEAK_TFLOPS = 78.6
#: kernel codes of akm_autotune / --shape
KERNEL_NAMES = {0: "row kernel, factors from global memory", 1: "row kernel, LDS factor tables",
                2: "sum-factorised matrix-core kernel",
                3: "one dimension at a time (identity factors left out)"}
FP32_PEAK_TFLOPS = 157.3
HBM_PEAK_GBS = 8000.0


def make_workload(d, n, L, T, seed=0):
    from asgard_amd import grid

    rng = np.random.default_rng(seed)
    table, _ = grid.element_table([L] * d)
    size1d = n * (1 << L)
    ops = [np.asfortranarray(rng.uniform(-1, 1, (size1d, size1d))) for _ in range(T * d)]
    vA = grid.build_vA(d, n, T, L, ops)
    x = rng.standard_normal(table.shape[0] * n ** d)
    return table, vA, x


def algorithmic_bytes(d, n, T, cells, nnz, nconn, kernel=0):
    """Unique bytes an apply must touch: x, y, CSR, cell 1D indices, vA (kernel
    3, one dimension at a time, has no CSR: x, y and vA)."""
    dof = cells * n ** d
    if kernel == 3:
        return 8 * dof + 8 * dof + 8 * n * n * d * T * nconn
    return 8 * dof + 8 * dof + 4 * (cells + 1 + nnz) + 4 * cells * d + 8 * n * n * d * T * nconn


def cpu_threads():
    """Threads of the CPU baseline: the OpenMP thread count the environment
    grants this job (OMP_NUM_THREADS), else every core in the affinity mask."""
    env = os.environ.get("OMP_NUM_THREADS", "")
    if env.isdigit() and int(env) > 0:
        return int(env)
    return JOB_CPUS


def cpu_host_info(threads):
    return {"cores": threads, "host_logical_cpus": os.cpu_count(),
            "affinity_cpus": JOB_CPUS,
            "omp_proc_bind": os.environ.get("OMP_PROC_BIND"),
            "omp_places": os.environ.get("OMP_PLACES")}


def cpu_baseline(d, n, table, vA, x, T, L, ref_y_gpu, reps=10):
    """The oracle's OpenMP kronmult (restatement of the reference's
    cpu_sparse) over the whole apply: 1 warm-up, median of `reps`."""
    import oracle

    threads = cpu_threads()
    oracle.set_num_threads(threads)
    pntr, indx, iA = oracle.sparse_pattern(table, n=n, T=T, max_level=L)
    y = np.zeros_like(x)
    oracle.kronmult_sparse(d, n, pntr, indx, T, iA, vA, 1.0, x, 0.0, y)  # warm-up
    times = []
    for _ in range(reps):
        t0 = time.perf_counter()
        oracle.kronmult_sparse(d, n, pntr, indx, T, iA, vA, 1.0, x, 0.0, y)
        times.append(time.perf_counter() - t0)
    flops = 2 * d * n ** (d + 1) * T * int(pntr[-1])
    med = float(np.median(times))
    err = float(np.abs(ref_y_gpu - y).max() / np.abs(y).max())
    rec = {"value": round(flops / med * 1e-9, 2), "unit": "GFLOP/s", "kind": "port", "count": "pair by pair",
           "sample": f"full apply of the same workload, median of {reps} after 1 warm-up "
                     "(OpenMP restatement of the reference's cpu_sparse)"}
    rec.update(cpu_host_info(threads))
    return rec, err


def cpu_baseline_rows(d, n, table, vA, x, T, L, y_gpu, stride=64, reps=10):
    """The oracle's OpenMP kronmult over a bounded sample of the apply: every
    `stride`-th row cell of the element table (rows of every length, in table
    order), all of each row's connected columns and terms; 1 warm-up, median
    of `reps`.  Also the FP64 parity of the GPU rows against it."""
    import oracle

    threads = cpu_threads()
    oracle.set_num_threads(threads)
    cells = table.shape[0]
    N = n ** d
    rows = np.arange(0, cells, stride, dtype=np.int32)
    pntr, indx, iA = oracle.sparse_pattern_rows(table, rows, n=n, T=T, max_level=L)
    y = np.zeros(len(rows) * N)
    oracle.kronmult_sparse(d, n, pntr, indx, T, iA, vA, 1.0, x, 0.0, y)  # warm-up
    times = []
    for _ in range(reps):
        t0 = time.perf_counter()
        oracle.kronmult_sparse(d, n, pntr, indx, T, iA, vA, 1.0, x, 0.0, y)
        times.append(time.perf_counter() - t0)
    pairs = int(pntr[-1])
    flops = 2 * d * n ** (d + 1) * T * pairs
    med = float(np.median(times))
    gpu_rows = y_gpu.reshape(cells, N)[rows].reshape(-1)
    err = float(np.abs(gpu_rows - y).max() / np.abs(y).max())
    rec = {"value": round(flops / med * 1e-9, 2), "unit": "GFLOP/s", "kind": "port", "count": "pair by pair",
           "sample": f"every {stride}th row cell of the element table: {len(rows)} of {cells} "
                     f"rows, {pairs:,} of the apply's connected pairs, all {T} terms, "
                     f"{flops / 1e9:.1f} GFLOP; 1 warm-up, median of {reps} applies "
                     f"({med:.2f} s each) of the OpenMP restatement of the reference's "
                     "cpu_sparse",
           "seconds_per_sample_apply": round(med, 4)}
    rec.update(cpu_host_info(threads))
    return rec, err


def profiled_traffic(profile, waves, lds_tables):
    """HBM bytes per apply of the chosen kernel shape, from a committed
    rocprofv3 FETCH_SIZE/WRITE_SIZE summary (each counter scaled by what it
    reads for a plain device copy of known size); None when the shape was not
    profiled."""
    key = "traffic_bytes W=%d lds=%d:" % (waves, int(lds_tables))
    try:
        with open(os.path.join(ROOT, "profiles", profile)) as f:
            for line in f:
                if line.startswith(key):
                    return int(line.split(":")[1])
    except OSError:
        pass
    return None


HEADLINE = dict(d=6, n=2, L=7, profile="kron_f64_d6n2_L7_T6_hbm_traffic.txt",
                workload="kronmult apply, d=6 n=2 |l|_1<=7 sparse grid, 6 terms "
                         "(3x+3v Vlasov advection operators)")
SMALL = dict(d=3, n=3, L=6, T=3, profile="kron_f64_d3n3_L6_T3_hbm_traffic.txt",
             workload="kronmult apply, d=3 n=3 |l|_1<=6 sparse grid, 3 terms, U[-1,1] "
                      "factors")


def headline_workload(seed=0):
    """The d=6 n=2 |l|_1<=7 grid with the Vlasov operator's 6 terms and
    x ~ U[-1, 1]."""
    from asgard_amd import dg, grid

    d, n, L = HEADLINE["d"], HEADLINE["n"], HEADLINE["L"]
    table, _ = grid.element_table([L] * d)
    ops = dg.operators_vlasov(n, L)
    T = len(ops) // d
    vA = grid.build_vA(d, n, T, L, ops)
    x = np.random.default_rng(seed).uniform(-1.0, 1.0, table.shape[0] * n ** d)
    return d, n, L, T, table, vA, x


def counted_flops(mat, table, vA, kernel):
    """Flops of one apply, for its rate.  Pair by pair: the reference's count,
    2*d*n^(d+1) per connected pair and term.  Kernel 3 never forms those
    products: its count is the reference's for the same operator taken one
    dimension at a time (the global operator's: two per entry of every
    non-identity 1D factor's pattern)."""
    import asgard_amd

    if kernel != 3:
        return mat.flops()
    d, n, T = mat.num_dimensions, mat.kron_size, mat.num_terms
    L = int(table[:, :d].max())
    _, _, diag = asgard_amd.connect_1d(L)
    unit = np.zeros((vA.size // (T * d * n * n), 1, 1, n * n))
    unit[diag] = np.eye(n).ravel()
    active = (vA.reshape(-1, T, d, n * n) != unit).any(axis=(0, 3)).astype(np.int32)
    glob = asgard_amd.KronmultMatrix.global_grid(d, n, table, L, T, vA, active=active)
    return glob.flops()


def choose_shape(mat, xd, yd, shape):
    """The kernel shape of an apply: the autotuner's choice, or `shape` =
    (waves per row, kernel) with kernel 0 = factors from global memory, 1 =
    LDS factor tables, 2 = matrix cores (for reproducible profiles)."""
    if shape is None:
        return mat.autotune(xd, yd)
    waves, kernel = shape
    mat.set_kernel_family(1 if kernel == 2 else 0)
    mat.set_tuning(waves_per_row=waves, lds_cap_bytes=-1 if kernel == 1 else 0)
    return waves, kernel


def time_steps(mat, xd, yd, steps, warmup, stream):
    """W untimed then K timed applies between HIP events recorded on the
    stream the kernel is launched on; returns (ms per apply, wall seconds)."""
    import torch

    for _ in range(warmup):
        mat.apply(1.0, xd, 0.0, yd)
    torch.cuda.synchronize()
    start = torch.cuda.Event(enable_timing=True)
    stop = torch.cuda.Event(enable_timing=True)
    t0 = time.perf_counter()
    start.record(stream)
    for _ in range(steps):
        mat.apply(1.0, xd, 0.0, yd)
    stop.record(stream)
    torch.cuda.synchronize()
    wall = time.perf_counter() - t0
    return start.elapsed_time(stop) / steps, wall


def roofline(flops, ms, peak, profile, waves, lds, alg_bytes):
    """Roofline record of a kronmult apply.  `flops` as counted_flops; kernel
    `lds` == 2 is the sum-factorised matrix-core kernel, which executes fewer
    flops than that count (its matrix-core utilisation comes from the committed
    SQ counter profile, `profiled_mfma`)."""
    achieved = flops / (ms * 1e-3) * 1e-12
    if lds == 3:
        # one dimension at a time: few flops per byte, so the bound is the
        # memory rate over the bytes it cannot avoid
        rate = alg_bytes / (ms * 1e-3) * 1e-9
        return {"bound": "hbm", "achieved": round(rate, 1), "peak": HBM_PEAK_GBS,
                "unit": "GB/s", "frac": round(rate / HBM_PEAK_GBS, 4), "traffic": None,
                "algorithmic_bytes": int(alg_bytes), "tflops": round(achieved, 3)}
    if lds == 2:
        bound = "mfma_fp64"
    else:
        bound = "valu_fp64" if peak == FP64_PEAK_TFLOPS else "valu_fp32"
    rec = {"bound": bound, "achieved": round(achieved, 3), "peak": peak, "unit": "TFLOP/s",
           "frac": round(achieved / peak, 4),
           "traffic": profiled_traffic(profile, waves, lds) if profile else None,
           "algorithmic_bytes": int(alg_bytes)}
    if lds == 2 and profile:
        busy = profiled_mfma(profile, waves)
        if busy is not None:
            # executed matrix-core flops per apply and their rate at this time
            rec["executed_mfma_tflop"] = busy
            rec["executed_mfma_tflops"] = round(busy / (ms * 1e-3), 3)
            rec["executed_mfma_frac"] = round(busy / (ms * 1e-3) / peak, 4)
    return rec


def profiled_mfma(profile, waves):
    """Executed matrix-core TFLOP per apply of the matrix-core kernel shape,
    from the SQ_INSTS_MFMA split recorded in a committed profile summary."""
    key = "executed_mfma_tflop W=%d:" % waves
    try:
        with open(os.path.join(ROOT, "profiles", profile)) as f:
            for line in f:
                if line.startswith(key):
                    return float(line.split(":")[1])
    except OSError:
        pass
    return None


SOLVE_WORKLOADS = {
    "d4n2": dict(workload="implicit step (I - dt A) u = b, d=4 n=2 |l|_1<=7, 4 terms "
                          "(advection in 2 dims, diffusion nu=0.1 in 2), dt=1e-3, GMRES(50), "
                          "b = (I - dt A) u0, u0 ~ U[-1,1]",
                 d=4, n=2, L=7, dt=1e-3, restart=50, rhs="operator", cpu=True),
    "d6n2": dict(workload="implicit step (I - dt A) u = u0, d=6 n=2 |l|_1<=7, 3x+3v Vlasov "
                          "advection (6 terms, central fluxes), dt=5e-4, GMRES(50), "
                          "u0 ~ U[-1,1]",
                 d=6, n=2, L=7, dt=5e-4, restart=50, rhs="state", cpu=False),
}


def solve_operators(key):
    from asgard_amd import dg

    w = SOLVE_WORKLOADS[key]
    if key == "d4n2":
        return dg.operators_advection_diffusion(w["d"], w["n"], w["L"], n_adv=2, nu=0.1)
    return dg.operators_vlasov(w["n"], w["L"])


def timed(fn):
    import torch

    torch.cuda.synchronize()
    t0 = time.perf_counter()
    out = fn()
    torch.cuda.synchronize()
    return out, time.perf_counter() - t0


def solve_comparison(key, samples=200_000, epochs=8, with_cpu=True):
    """Time to a 1e-10 relative FP64 residual of one implicit step: plain FP64
    GPU GMRES (the reference algorithm, absolute tolerance 1e-10*|b|) against
    FP64 refinement around FP32-kronmult GMRES cycles, with and without the
    learned preconditioner.  Each solve is run once untimed (workspace
    allocation) and then timed from the same initial guess x0 = b."""
    import torch

    import asgard_amd
    from asgard_amd import grid, learned

    w = SOLVE_WORKLOADS[key]
    d, n, L, dt, restart = w["d"], w["n"], w["L"], w["dt"], w["restart"]
    table, _ = grid.element_table([L] * d)
    ops = solve_operators(key)
    T = len(ops) // d
    vA = grid.build_vA(d, n, T, L, ops)
    m64 = asgard_amd.KronmultMatrix.sparse_grid(d, n, table, L, T, vA)
    m32 = asgard_amd.KronmultMatrix.sparse_grid(d, n, table, L, T, vA.astype(np.float32),
                                                dtype=np.float32)
    stream = torch.cuda.current_stream().cuda_stream
    m64.set_stream(stream)
    m32.set_stream(stream)
    size = m64.output_size()
    rng = np.random.default_rng(0)
    u0 = torch.from_numpy(rng.uniform(-1.0, 1.0, size)).cuda()
    scratch = torch.zeros_like(u0)
    m64.autotune(u0, scratch)
    m32.autotune(u0.float(), scratch.float())
    if w["rhs"] == "operator":
        b = m64.apply_euler(dt, 1.0, u0, 0.0, torch.zeros_like(u0))
    else:
        b = u0.clone()
    torch.cuda.synchronize()
    bnorm = float(torch.linalg.norm(b).item())

    def true_rel(x):
        r = m64.apply_euler(dt, 1.0, x, 0.0, torch.zeros_like(x))
        return float(torch.linalg.norm(b - r).item()) / bnorm

    out = {"workload": w["workload"], "unknowns": int(size), "pairs": int(m64.num_pairs()),
           "flops_per_apply": int(m64.flops())}
    # plain FP64 GPU GMRES
    plain = {}
    for rep in range(2):
        x = b.clone()
        info, t = timed(lambda: asgard_amd.simple_gmres_euler(dt, m64, x, b, restart, -1,
                                                              1e-10 * bnorm))
    plain.update(seconds=round(t, 5), applies_f64=info.iterations, rel_residual=true_rel(x))
    x_plain = x
    out["plain_fp64"] = plain

    def mixed(mat32, pre, label):
        for rep in range(2):
            xm = b.clone()
            st, t = timed(lambda: asgard_amd.gmres_euler_mixed(dt, m64, xm, b, mat32=mat32,
                                                               precond=pre, restart=restart,
                                                               tol=1e-10))
        rec = st.as_dict()
        rec.update(seconds=round(t, 5), speedup_vs_plain=round(plain["seconds"] / t, 3),
                   rel_residual_check=true_rel(xm),
                   rel_diff_vs_plain=float(torch.linalg.norm(xm - x_plain).item() /
                                           torch.linalg.norm(x_plain).item()))
        out[label] = rec
        return xm

    mixed(m32, None, "fp32_refinement")

    # the reference's default operator (global Kronecker, identity factors
    # skipped): its own solve is left-Jacobi-preconditioned, judged here by
    # the same true FP64 residual
    act = grid.identity_mask(ops, T, d)
    g64 = asgard_amd.KronmultMatrix.global_grid(d, n, table, L, T, vA, active=act)
    g32 = asgard_amd.KronmultMatrix.global_grid(d, n, table, L, T, vA.astype(np.float32),
                                                dtype=np.float32, active=act)
    g64.set_stream(stream)
    g32.set_stream(stream)
    g64.autotune(u0, scratch)
    g32.autotune(u0.float(), scratch.float())
    out["global_operator"] = {
        "chains_stages": list(g64.global_info()[1:]),
        "apply_us": {"pair_fp64": round(m64.time_apply(1.0, u0, 0.0, scratch, 5) * 1e3, 1),
                     "global_fp64": round(g64.time_apply(1.0, u0, 0.0, scratch, 20) * 1e3, 1),
                     "global_fp32": round(g32.time_apply(1.0, u0.float(), 0.0, scratch.float(),
                                                         20) * 1e3, 1)}}
    for rep in range(2):
        xg = b.clone()
        ginfo, tg = timed(lambda: asgard_amd.simple_gmres_euler(dt, g64, xg, b, restart, -1,
                                                                0.5e-10 * bnorm))
    out["global_plain_fp64_jacobi"] = dict(
        seconds=round(tg, 5), iterations=ginfo.iterations, rel_residual=true_rel(xg),
        speedup_vs_plain=round(plain["seconds"] / tg, 3))
    for rep in range(2):
        xg = b.clone()
        gst, tg = timed(lambda: asgard_amd.gmres_euler_mixed(dt, g64, xg, b, mat32=g32,
                                                             restart=restart, tol=1e-10))
    rec = gst.as_dict()
    rec.update(seconds=round(tg, 5), speedup_vs_plain=round(plain["seconds"] / tg, 3),
               speedup_vs_global_plain=round(out["global_plain_fp64_jacobi"]["seconds"] / tg,
                                             3),
               rel_residual_check=true_rel(xg))
    out["global_fp32_refinement"] = rec
    (pre, tinfo), t_train = timed(lambda: learned.train_preconditioner(
        m64, table, L, dt, samples=samples, epochs=epochs, batch=1024, lr=1e-3, hidden=256,
        seed=0))
    tinfo["seconds"] = round(t_train, 3)
    out["training"] = tinfo
    mixed(m32, pre, "fp32_refinement_learned")
    # the same network on the global operator (one operator: on a standard
    # grid the global and pair operators agree for any factors)
    for rep in range(2):
        xg = b.clone()
        gst, tg = timed(lambda: asgard_amd.gmres_euler_mixed(dt, g64, xg, b, mat32=g32,
                                                             precond=pre, restart=restart,
                                                             tol=1e-10))
    rec = gst.as_dict()
    rec.update(seconds=round(tg, 5), speedup_vs_plain=round(plain["seconds"] / tg, 3),
               speedup_vs_global_plain=round(out["global_plain_fp64_jacobi"]["seconds"] / tg,
                                             3),
               rel_residual_check=true_rel(xg))
    out["global_fp32_refinement_learned"] = rec
    mixed(None, None, "fp64_flexible")
    mixed(None, pre, "fp64_flexible_learned")
    if w["rhs"] == "operator":
        out["max_abs_error_vs_u0"] = {
            k: float((xx - u0).abs().max().item()) for k, xx in [("plain_fp64", x_plain)]}
    if with_cpu and w["cpu"]:
        out["cpu_baseline"] = solve_cpu_baseline(d, n, L, T, table, vA, dt, b.cpu().numpy(),
                                                 restart, x_plain.cpu().numpy())
    return out


def workload_variants(d, n, L, T, table, x, y64, stream, no_cpu):
    """GFLOP/s of the bench grid with the repo's DG advection/mass operators
    (parity vs the oracle unless no_cpu) and of the FP32 kronmult on the
    random factors (its error vs the FP64 GPU result)."""
    import torch

    import asgard_amd
    from asgard_amd import dg, grid

    out = {}
    xd = torch.from_numpy(x).cuda()
    ops = dg.operators_advection(d, n, L)
    vA_dg = grid.build_vA(d, n, T, L, ops)
    mdg = asgard_amd.KronmultMatrix.sparse_grid(d, n, table, L, T, vA_dg)
    mdg.set_stream(stream.cuda_stream)
    y = torch.zeros_like(xd)
    kernel = mdg.autotune(xd, y)[1]
    ms = mdg.time_apply(1.0, xd, 0.0, y, 50)
    mdg.apply(1.0, xd, 0.0, y)
    rec = {"gflops": round(counted_flops(mdg, table, vA_dg, kernel) / (ms * 1e-3) * 1e-9, 1),
           "ms_per_apply": round(ms, 5),
           "operators": "DG advection (upwind flux) in dimension t for term t, mass elsewhere"}
    if not no_cpu:
        import oracle

        pntr, indx, iA = oracle.sparse_pattern(table, n=n, T=T, max_level=L)
        ref = np.zeros_like(x)
        oracle.kronmult_sparse(d, n, pntr, indx, T, iA, vA_dg, 1.0, x, 0.0, ref)
        rec["parity_max_rel_err_vs_oracle"] = float(np.abs(y.cpu().numpy() - ref).max() /
                                                    np.abs(ref).max())
    out["dg_advection_mass"] = rec
    _, vA, _ = make_workload(d, n, L, T)
    m32 = asgard_amd.KronmultMatrix.sparse_grid(d, n, table, L, T, vA.astype(np.float32),
                                                dtype=np.float32)
    m32.set_stream(stream.cuda_stream)
    x32 = xd.float()
    y32 = torch.zeros_like(x32)
    kernel32 = m32.autotune(x32, y32)[1]
    ms32 = m32.time_apply(1.0, x32, 0.0, y32, 50)
    m32.apply(1.0, x32, 0.0, y32)
    err = float(((y32.double() - y64).abs().max() / y64.abs().max()).item())
    rate32 = counted_flops(m32, table, vA, kernel32) / (ms32 * 1e-3) * 1e-9
    out["fp32_random"] = {"gflops": round(rate32, 1), "ms_per_apply": round(ms32, 5),
                          "max_rel_err_vs_fp64": err,
                          "roofline_frac_fp32": round(rate32 * 1e-3 / FP32_PEAK_TFLOPS, 4)}
    return out


def global_operator_applies(reps=20):
    """Applies of the global Kronecker operator (the reference's default
    mode) on the two solve workloads' operators and on the bench workload's
    random factors; per apply the time, the layout the autotuner chose and
    the algorithmic bytes (chain layouts: every stage reads and writes one
    padded vector per chain, the chain sum reads one vector per chain and
    writes y; slab layout: every term group reads x and writes one vector,
    the sum reads the group vectors and writes y)."""
    import torch

    import asgard_amd
    from asgard_amd import grid

    out = {}
    cases = [("d4n2_adv_diff", "d4n2"), ("d6n2_vlasov", "d6n2"), ("d3n3_random", None)]
    for label, key in cases:
        if key is None:
            d, n, L, T = 3, 3, 6, 3
            table, vA, _ = make_workload(d, n, L, T)
            act = None
        else:
            w = SOLVE_WORKLOADS[key]
            d, n, L = w["d"], w["n"], w["L"]
            table, _ = grid.element_table([L] * d)
            ops = solve_operators(key)
            T = len(ops) // d
            vA = grid.build_vA(d, n, T, L, ops)
            act = grid.identity_mask(ops, T, d)
        rec = {}
        for prec, dtype in (("fp64", np.float64), ("fp32", np.float32)):
            m = asgard_amd.KronmultMatrix.global_grid(d, n, table, L, T, vA.astype(dtype),
                                                      dtype=dtype, active=act)
            x = torch.from_numpy(np.random.default_rng(0).standard_normal(
                m.output_size()).astype(dtype)).cuda()
            y = torch.zeros_like(x)
            layout = m.autotune(x, y)[0]
            ms = m.time_apply(1.0, x, 0.0, y, reps)
            pad, chains, stages = m.global_info()
            dofs = m.output_size()
            padded = dofs + pad * n ** d
            esize = np.dtype(dtype).itemsize
            if layout == 6:
                # slab layout: every group reads x and writes its sum once, the
                # remaining chains run stage by stage, the final sum reads its
                # sources and writes y
                groups, rest, sources = m.slab_info()
                moved = (2 * groups * dofs + rest * stages * 2 * padded +
                         (sources + 1) * dofs) * esize
            else:
                moved = (chains * stages * 2 * padded + (chains + 1) * dofs) * esize
            rec[prec] = {"us_per_apply": round(ms * 1e3, 2), "layout": layout,
                         "chains": chains, "stages": stages,
                         "algorithmic_bytes": int(moved),
                         "achieved_GBps": round(moved / (ms * 1e-3) * 1e-9, 1)}
        out[label] = rec
    return out


def batch_systems(count=64, seed=0, inputs=None):
    """The batched-solve workload: `count` implicit steps, d ~ U{2..5}, n in
    {2, 3}, each on the |l|_1 <= 5 sparse grid with 10-30% of its leaf cells
    refined one level (seeded), d terms (advection in the first d/2
    dimensions, diffusion nu = 0.1 in the others), dt = 1e-3, b ~ U[-1, 1].
    When `inputs` is a list, (d, n, table, max level, vA) of every system is
    appended to it."""
    import asgard_amd
    from asgard_amd import dg, grid

    rng = np.random.default_rng(seed)
    mats, dts, bs = [], [], []
    for q in range(count):
        d = int(rng.integers(2, 6))
        n = int(rng.choice([2, 3]))
        frac = float(rng.uniform(0.1, 0.3))
        table, _ = grid.element_table([5] * d)
        table = grid.refine(table, frac, seed=seed * 1000 + q)
        L = int(table[:, :d].max())
        ops = dg.operators_advection_diffusion(d, n, L, n_adv=max(1, d // 2), nu=0.1)
        vA = grid.build_vA(d, n, d, L, ops)
        mats.append(asgard_amd.KronmultMatrix.sparse_grid(d, n, table, L, d, vA))
        if inputs is not None:
            inputs.append((d, n, table, L, vA))
        dts.append(1e-3)
        bs.append(rng.uniform(-1.0, 1.0, table.shape[0] * n ** d))
    return mats, dts, bs


def batch_comparison(count=64, restart=50):
    """Aggregate solves per second of `count` implicit steps: one at a time
    with the device GMRES (the reference algorithm, absolute tolerance
    1e-10*|b|) against all at once with the batched solver (true FP64
    residual <= 1e-10*|b|).  Both start from x0 = b; the batch is built and
    solved once untimed (graph instantiation, first launches) first."""
    import torch

    import asgard_amd

    mats, dts, bs_host = batch_systems(count)
    bs = [torch.from_numpy(b).cuda() for b in bs_host]
    for m in mats:
        m.set_stream(torch.cuda.current_stream().cuda_stream)
    sizes = [m.output_size() for m in mats]
    out = {"workload": f"{count} implicit steps (I - dt A_s) x_s = b_s, d ~ U{{2..5}}, n in {{2,3}}, "
                       "|l|_1<=5 sparse grids with 10-30% of leaf cells refined one level, d terms "
                       "(advection + diffusion nu=0.1), dt=1e-3, b ~ U[-1,1], GMRES(50), "
                       "tol 1e-10 relative",
           "systems": count, "unknowns_total": int(sum(sizes)), "unknowns_max": int(max(sizes)),
           "pairs_total": int(sum(m.num_pairs() for m in mats))}

    def sequential():
        xs = [b.clone() for b in bs]
        its = 0
        for m, dt, x, b in zip(mats, dts, xs, bs):
            info = asgard_amd.simple_gmres_euler(dt, m, x, b, restart, -1,
                                                 1e-10 * float(torch.linalg.norm(b).item()))
            its += info.iterations
        return xs, its

    sequential()  # workspaces
    (xs_seq, its_seq), t_seq = timed(sequential)
    batch = asgard_amd.BatchSolver(mats, dts, restart=restart)
    warm = [b.clone() for b in bs]
    batch.solve(warm, bs)
    xs = [b.clone() for b in bs]
    (res, its, conv), t_batch = timed(lambda: batch.solve(xs, bs))
    diff = max(float(torch.linalg.norm(a - c).item() / torch.linalg.norm(c).item())
               for a, c in zip(xs, xs_seq))
    out.update({
        "sequential_fp64": {"seconds": round(t_seq, 4), "solves_per_s": round(count / t_seq, 2),
                            "applies": int(its_seq)},
        "batched_fp64": {"seconds": round(t_batch, 4), "solves_per_s": round(count / t_batch, 2),
                         "applies": int(its.sum()), "converged": int(conv.sum()),
                         "max_rel_residual": float(res.max()), **batch.info()},
        "speedup": round(t_seq / t_batch, 3),
        "max_rel_diff_batched_vs_sequential": diff,
    })
    return out


def solve_cpu_baseline(d, n, L, T, table, vA, dt, b, restart, x_gpu):
    """The oracle's restatement of simple_gmres_euler with its OpenMP kronmult
    on the host cores, same system, same tolerance; and the GPU solution's
    difference from it."""
    import oracle

    threads = min(16, os.cpu_count() or 1)
    oracle.set_num_threads(threads)
    pntr, indx, iA = oracle.sparse_pattern(table, n=n, T=T, max_level=L)
    x = b.copy()
    bn = float(np.linalg.norm(b))
    t0 = time.perf_counter()
    x, err, its = oracle.gmres_euler_sparse(d, n, pntr, indx, T, iA, vA, dt, x, b, restart,
                                            1000, 1e-10 * bn)
    t = time.perf_counter() - t0
    return {"seconds": round(t, 3), "cores": threads, "kind": "port", "count": "pair by pair", "applies": its,
            "sample": "the whole solve (oracle restatement of simple_gmres_euler)",
            "rel_diff_gpu_plain_vs_oracle": float(np.linalg.norm(x_gpu - x) / np.linalg.norm(x))}


def calibrate_copy(mib=512, reps=5):
    """A plain device copy of known size, profiled with the same HBM counters
    (FETCH_SIZE, WRITE_SIZE) as the kronmult to scale them to bytes."""
    import torch

    n = mib * 1024 * 1024 // 8
    src = torch.ones(n, dtype=torch.float64, device="cuda")
    dst = torch.empty_like(src)
    for _ in range(reps):
        dst.copy_(src)
    torch.cuda.synchronize()
    print(json.dumps({"copy_bytes_read": n * 8, "copy_bytes_written": n * 8, "reps": reps}))


def small_apply(stream, no_cpu, steps=100, warmup=10, shape=None):
    """The d=3 n=3 |l|_1<=6 apply with 3 random terms: its GFLOP/s, roofline
    and parity against the oracle's full apply, and its DG / FP32 variants."""
    import torch

    import asgard_amd

    d, n, L, T = SMALL["d"], SMALL["n"], SMALL["L"], SMALL["T"]
    table, vA, x = make_workload(d, n, L, T)
    mat = asgard_amd.KronmultMatrix.sparse_grid(d, n, table, L, T, vA)
    mat.set_stream(stream.cuda_stream)
    xd = torch.from_numpy(x).cuda()
    yd = torch.zeros_like(xd)
    waves, lds = choose_shape(mat, xd, yd, shape)
    ms, _ = time_steps(mat, xd, yd, steps, warmup, stream)
    nconn = len(asgard_amd.connect_1d(L)[1])
    flops = counted_flops(mat, table, vA, lds)
    rec = {"workload": SMALL["workload"], "cells": int(table.shape[0]),
           "connected_pairs": int(mat.num_pairs()), "flops_per_apply": int(flops),
           "ms_per_apply": round(ms, 5), "gflops": round(flops / (ms * 1e-3) * 1e-9, 1),
           "waves_per_row": waves, "lds_factor_tables": lds,
           "roofline": roofline(flops, ms, FP64_PEAK_TFLOPS, SMALL["profile"], waves, lds,
                                algorithmic_bytes(d, n, T, table.shape[0], mat.num_pairs(),
                                                  nconn, lds))}
    if not no_cpu:
        cpu, parity = cpu_baseline(d, n, table, vA, x, T, L, yd.cpu().numpy())
        rec["cpu_baseline"] = cpu
        rec["parity_max_rel_err_vs_oracle"] = parity
    rec["variants"] = workload_variants(d, n, L, T, table, x, yd, stream, no_cpu)
    gmat = asgard_amd.KronmultMatrix.global_grid(d, n, table, L, T, vA)
    gmat.set_stream(stream.cuda_stream)
    glanes = gmat.autotune(xd, torch.zeros_like(xd))[0]
    gy = torch.zeros_like(xd)
    gmat.apply(1.0, xd, 0.0, gy)
    mat.set_tuning(waves_per_row=4)  # pair by pair
    mat.apply(1.0, xd, 0.0, yd)
    torch.cuda.synchronize()
    rec["global_operator"] = {
        "us_per_apply": round(gmat.time_apply(1.0, xd, 0.0, gy, 50) * 1e3, 2),
        "chains_stages": list(gmat.global_info()[1:]), "layout": glanes,
        "max_rel_diff_vs_pair": float((gy - yd).abs().max().item() / yd.abs().max().item())}
    return rec


def headline_fp32(d, n, L, T, table, vA, xd, y64, stream):
    """The FP32 kronmult of the headline workload: GFLOP/s, FP32 roofline and
    its error against the FP64 GPU result."""
    import torch

    import asgard_amd

    m32 = asgard_amd.KronmultMatrix.sparse_grid(d, n, table, L, T, vA.astype(np.float32),
                                                dtype=np.float32)
    m32.set_stream(stream.cuda_stream)
    x32 = xd.float()
    y32 = torch.zeros_like(x32)
    waves, lds = m32.autotune(x32, y32)
    ms = m32.time_apply(1.0, x32, 0.0, y32, 5)
    m32.apply(1.0, x32, 0.0, y32)
    err = float(((y32.double() - y64).abs().max() / y64.abs().max()).item())
    ach = counted_flops(m32, table, vA, lds) / (ms * 1e-3) * 1e-12
    return {"ms_per_apply": round(ms, 4), "gflops": round(ach * 1e3, 1),
            "waves_per_row": waves, "lds_factor_tables": lds,
            "roofline_frac_fp32": round(ach / FP32_PEAK_TFLOPS, 4),
            "max_rel_err_vs_fp64": err}


def solve_targets(solve):
    """Time-to-1e-10 ratios of the implicit step, FP32 kronmult + learned
    preconditioner against plain FP64 GMRES on the same operator (the pair
    operator, and the global operator), per solve workload."""
    out = {}
    for k, rec in solve.items():
        if "plain_fp64" not in rec:
            continue
        r = {}
        if "fp32_refinement_learned" in rec:
            r["pair_fp64_plain_s"] = rec["plain_fp64"]["seconds"]
            r["pair_fp32_learned_s"] = rec["fp32_refinement_learned"]["seconds"]
            r["pair_ratio"] = round(r["pair_fp64_plain_s"] / r["pair_fp32_learned_s"], 3)
            r["pair_fp32_no_network_s"] = rec["fp32_refinement"]["seconds"]
        if "global_fp32_refinement_learned" in rec:
            r["global_fp64_plain_s"] = rec["global_plain_fp64_jacobi"]["seconds"]
            r["global_fp32_learned_s"] = rec["global_fp32_refinement_learned"]["seconds"]
            r["global_ratio"] = round(r["global_fp64_plain_s"] / r["global_fp32_learned_s"], 3)
        r["target"] = 4.0
        r["met"] = bool(max(r.get("pair_ratio", 0), r.get("global_ratio", 0)) >= 4.0)
        out[k] = r
    return out


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline legs")
    ap.add_argument("--no-extras", action="store_true",
                    help="headline apply only (no d=3 apply, FP32, global operator)")
    ap.add_argument("--small-only", action="store_true",
                    help="print only the d=3 n=3 apply record (one JSON line)")
    ap.add_argument("--calibrate-copy", action="store_true",
                    help="run only a 512 MiB device copy (HBM counter calibration)")
    ap.add_argument("--solve", default="d4n2,d6n2,batch64",
                    help="implicit-step solve comparisons to run (comma list of "
                         + ", ".join(list(SOLVE_WORKLOADS) + ["batch64"]) + "; 'none' to skip)")
    ap.add_argument("--solve-only", action="store_true",
                    help="print only the solve comparisons (one JSON line each)")
    ap.add_argument("--global-only", action="store_true",
                    help="print only the global-operator applies (one JSON line)")
    ap.add_argument("--samples", type=int, default=200_000,
                    help="per-cell training samples of the learned preconditioner")
    ap.add_argument("--shape", default=None,
                    help="W:K pins the kronmult kernel shape instead of autotuning: W "
                         "wavefronts per row, K = 0 factors from global memory, 1 LDS "
                         "factor tables, 2 matrix cores (for profiling)")
    args = ap.parse_args()
    shape = tuple(int(v) for v in args.shape.split(":")) if args.shape else None
    if args.gpus != 1:
        print(f"bench.py: this build runs on one GPU only; --gpus {args.gpus} is not "
              "supported (the row-sharded multi-GPU design is described in DESIGN.md)",
              file=sys.stderr)
        sys.exit(2)
    if args.calibrate_copy:
        calibrate_copy()
        return
    if args.global_only:
        print(json.dumps({"global_operator_applies": global_operator_applies()}), flush=True)
        return
    solves = [] if args.solve == "none" else [k for k in args.solve.split(",") if k]

    def run_solve(k):
        if k == "batch64":
            return batch_comparison(64)
        return solve_comparison(k, samples=args.samples, with_cpu=not args.no_cpu)

    if args.solve_only:
        for k in solves:
            print(json.dumps({"solve": k, **run_solve(k)}), flush=True)
        return

    import torch

    import asgard_amd

    stream = torch.cuda.current_stream()
    if args.small_only:
        print(json.dumps(small_apply(stream, args.no_cpu, shape=shape)), flush=True)
        return

    d, n, L, T, table, vA, x = headline_workload()
    cells = table.shape[0]
    mat = asgard_amd.KronmultMatrix.sparse_grid(d, n, table, L, T, vA)
    mat.set_stream(stream.cuda_stream)
    xd = torch.from_numpy(x).cuda()
    yd = torch.zeros_like(xd)
    nnz = mat.num_pairs()
    nconn = len(asgard_amd.connect_1d(L)[1])
    # setup, untimed: the autotuner picks the workgroup shape and LDS layout
    waves, lds_tables = choose_shape(mat, xd, yd, shape)
    flops = counted_flops(mat, table, vA, lds_tables)
    ms_per_step, wall = time_steps(mat, xd, yd, args.steps, args.warmup, stream)
    gflops = flops / (ms_per_step * 1e-3) * 1e-9

    cpu = None
    parity = None
    if not args.no_cpu:
        cpu, parity = cpu_baseline_rows(d, n, table, vA, x, T, L, yd.cpu().numpy())

    line = {
        "metric": "kronmult GFLOP/s (FP64 apply)",
        "value": round(gflops, 2),
        "unit": "GFLOP/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(ms_per_step, 5),
        "wall_s": round(wall, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64",
        "data": "synthetic",
        "config": {"workload": HEADLINE["workload"], "d": d, "n": n, "max_level": L,
                   "terms": T, "cells": int(cells), "unknowns": int(mat.output_size()),
                   "connected_pairs": int(nnz), "flops_per_apply": int(flops),
                   "pair_count_flops": int(mat.flops()),
                   "parallelism": "single GPU", "waves_per_row": waves,
                   "kernel": KERNEL_NAMES.get(lds_tables, str(lds_tables))},
        "roofline": roofline(flops, ms_per_step, FP64_PEAK_TFLOPS, HEADLINE["profile"], waves,
                             lds_tables,
                             algorithmic_bytes(d, n, T, cells, nnz, nconn, lds_tables)),
        "cpu_baseline": cpu,
        "parity_max_rel_err_vs_oracle": parity,
    }
    print(json.dumps({"progress": "headline done", "value": line["value"]}), file=sys.stderr,
          flush=True)
    if not args.no_extras:
        line["fp32_apply"] = headline_fp32(d, n, L, T, table, vA, xd, yd, stream)
        line["variants"] = {"d3n3_L6_T3": small_apply(stream, args.no_cpu)}
    del mat
    torch.cuda.empty_cache()
    if solves:
        line["solve"] = {}
        for k in solves:
            print(json.dumps({"progress": f"solve {k}"}), file=sys.stderr, flush=True)
            try:
                line["solve"][k] = run_solve(k)
            except Exception as e:  # report, keep the kronmult line
                line["solve"][k] = {"error": f"{type(e).__name__}: {e}"}
        line["solve_target_4x"] = solve_targets(line["solve"])
    print(json.dumps(line))


if __name__ == "__main__":
    main()
